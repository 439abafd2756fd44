// Precision conversion of column-major blocks (src/convert.cu:324-360).
// HBM-bound streaming kernels: each thread takes 8 consecutive rows of 4
// columns with vector accesses, so a wavefront reads 512 consecutive elements
// of a column; the y grid dimension walks the columns.
#include "common.hpp"

namespace remifa {
namespace {

struct bf16s {
  uint16_t v;
};
struct e4m3s {
  uint8_t v;
};

__device__ __forceinline__ double ld_wide(const float* p) { return (double)*p; }
__device__ __forceinline__ double ld_wide(const double* p) { return *p; }
__device__ __forceinline__ double ld_wide(const half_t* p) { return (double)(float)*p; }
__device__ __forceinline__ double ld_wide(const bf16s* p) { return (double)bf16_bits_to_f32(p->v); }
__device__ __forceinline__ double ld_wide(const e4m3s* p) { return (double)e4m3_bits_to_f32(p->v); }

// Narrowing from float sources goes through float (exact), from double
// sources straight from the double value: one rounding either way.
template <typename S>
struct is_double_src {
  static constexpr bool value = false;
};
template <>
struct is_double_src<double> {
  static constexpr bool value = true;
};

template <typename S>
__device__ __forceinline__ void st_narrow(float* p, const S* s) {
  if constexpr (is_double_src<S>::value)
    *p = (float)*s;
  else
    *p = (float)ld_wide(s);
}
template <typename S>
__device__ __forceinline__ void st_narrow(double* p, const S* s) {
  *p = ld_wide(s);
}
template <typename S>
__device__ __forceinline__ void st_narrow(half_t* p, const S* s) {
  if constexpr (is_double_src<S>::value)
    *p = (half_t)*s;  // fptrunc f64 -> f16: single rounding
  else
    *p = (half_t)(float)ld_wide(s);
}
template <typename S>
__device__ __forceinline__ void st_narrow(bf16s* p, const S* s) {
  p->v = f32_to_bf16_bits((float)ld_wide(s));
}
template <typename S>
__device__ __forceinline__ void st_narrow(e4m3s* p, const S* s) {
  p->v = f32_to_e4m3_bits((float)ld_wide(s));
}

// CV rows x CJ columns per thread: every load of the thread goes out before
// the first store. Column starts have the alignment of an element only (any
// leading dimension), so the vectors are declared with that alignment and the
// hardware splits a 16-byte access that crosses a line. m below 2048: the
// workgroup is BX threads along the rows, 256 / BX along the columns.
// Measured (MI355X, fp32 -> fp16): 16384 x 16384 421 -> 309 us (5.2 TB/s), against
// four rows with element accesses.
constexpr int CV = 8, CJ = 4;

template <typename T, int N>
struct vec_of {
  T e[N];
};
// N elements from / to p, element-aligned
template <typename T, int N>
__device__ __forceinline__ vec_of<T, N> ld_vec(const T* p) {
  vec_of<T, N> v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}
template <typename T, int N>
__device__ __forceinline__ void st_vec(T* p, const vec_of<T, N>& v) {
  __builtin_memcpy(p, &v, sizeof(v));
}

// threads along the rows for vectors of v rows: a power of two, at most 256
int rows_of_block(int64_t m, int v) {
  int bx = 256;
  while (bx > 8 && (int64_t)(bx / 2) * v >= m) bx /= 2;
  return bx;
}

template <typename S, typename D>
__global__ void __launch_bounds__(256) convert_kernel(int64_t m, int64_t n, const S* __restrict__ a,
                                                      int64_t lda, D* __restrict__ b, int64_t ldb) {
  const int64_t i0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * CV;
  if (i0 >= m) return;
  const int64_t jstep = (int64_t)gridDim.y * blockDim.y * CJ;
  for (int64_t j0 = ((int64_t)blockIdx.y * blockDim.y + threadIdx.y) * CJ; j0 < n; j0 += jstep) {
    if (i0 + CV <= m && j0 + CJ <= n) {
      vec_of<S, CV> x[CJ];
#pragma unroll
      for (int c = 0; c < CJ; ++c) x[c] = ld_vec<S, CV>(a + i0 + (j0 + c) * lda);
#pragma unroll
      for (int c = 0; c < CJ; ++c) {
        vec_of<D, CV> y;
#pragma unroll
        for (int r = 0; r < CV; ++r) st_narrow(&y.e[r], &x[c].e[r]);
        st_vec<D, CV>(b + i0 + (j0 + c) * ldb, y);
      }
    } else {
      for (int c = 0; c < CJ && j0 + c < n; ++c) {
        S x[CV];
#pragma unroll
        for (int r = 0; r < CV; ++r) x[r] = a[(i0 + r < m ? i0 + r : i0) + (j0 + c) * lda];
#pragma unroll
        for (int r = 0; r < CV; ++r)
          if (i0 + r < m) st_narrow(b + i0 + r + (j0 + c) * ldb, &x[r]);
      }
    }
  }
}

template <typename S, typename D>
int launch_typed(hipStream_t s, int64_t m, int64_t n, const void* a, int64_t lda, void* b,
                 int64_t ldb) {
  const int bx = rows_of_block(m, CV), by = 256 / bx;
  const int64_t gy = ceil_div(n, (int64_t)by * CJ);
  dim3 grid((unsigned)ceil_div(m, (int64_t)bx * CV), (unsigned)(gy < 65535 ? gy : 65535));
  convert_kernel<S, D>
      <<<grid, dim3(bx, by), 0, s>>>(m, n, (const S*)a, lda, (D*)b, ldb);
  RF_HIP(hipGetLastError());
  return 0;
}

template <typename S>
int launch_src(hipStream_t s, int dst_t, int64_t m, int64_t n, const void* a, int64_t lda,
               void* b, int64_t ldb) {
  switch (dst_t) {
    case REMIFA_R_32F: return launch_typed<S, float>(s, m, n, a, lda, b, ldb);
    case REMIFA_R_16F: return launch_typed<S, half_t>(s, m, n, a, lda, b, ldb);
    case REMIFA_R_64F: return launch_typed<S, double>(s, m, n, a, lda, b, ldb);
    case REMIFA_R_16BF: return launch_typed<S, bf16s>(s, m, n, a, lda, b, ldb);
    case REMIFA_R_8F_E4M3: return launch_typed<S, e4m3s>(s, m, n, a, lda, b, ldb);
  }
  return -3;
}

}  // namespace

int convert_launch(remifa_handle_t h, int src_t, int dst_t, int64_t m, int64_t n, const void* a,
                   int64_t lda, void* b, int64_t ldb) {
  if (m == 0 || n == 0) return 0;
  hipStream_t s = h->stream;
  double bytes = (double)m * n * (dtype_size(src_t) + dtype_size(dst_t));
  timer_begin(h, KC_CONVERT, bytes);
  int st;
  switch (src_t) {
    case REMIFA_R_32F: st = launch_src<float>(s, dst_t, m, n, a, lda, b, ldb); break;
    case REMIFA_R_16F: st = launch_src<half_t>(s, dst_t, m, n, a, lda, b, ldb); break;
    case REMIFA_R_64F: st = launch_src<double>(s, dst_t, m, n, a, lda, b, ldb); break;
    case REMIFA_R_16BF: st = launch_src<bf16s>(s, dst_t, m, n, a, lda, b, ldb); break;
    case REMIFA_R_8F_E4M3: st = launch_src<e4m3s>(s, dst_t, m, n, a, lda, b, ldb); break;
    default: st = -2;
  }
  timer_end(h);
  return st;
}

}  // namespace remifa
