// Equilibration on the GPU: the power-of-two row and column scalings of
// LAPACK's sgeequb and their application as slaqge does, which the
// reference harness runs on the host before factoring (--scale,
// tests/testing_lu_gpu.hxx:288-311, through src/wrappers.cxx:209-250).
//
// geequb: r_i = 1 / 2^trunc(log2 max_j |a_ij|), c_j = 1 / 2^trunc(log2
// max_i |a_ij| r_i) (each clamped to [SMLNUM, BIGNUM] before inverting),
// ROWCND / COLCND = min / max of the unclamped powers, AMAX = the largest row
// power; a zero row i (column j) stops with INFO = i (m + j), 1-based.
// laqge: with THRESH = 0.1 and SMALL = 2^-103 (SLAMCH('S') / SLAMCH('P')):
// no scaling, columns only, rows only or both (a_ij = (c_j r_i) a_ij);
// powers of two multiply exactly, so the scaled matrix is exact barring
// overflow or underflow.
//
// HBM-bound: the row maxima are one read of A (lanes on consecutive rows,
// column chunks in the grid, maxima combined by integer atomicMax on the
// bit patterns of non-negative floats, which orders like the values), the
// column maxima one more read (a workgroup per column), the scaling one read
// and one write. trunc(log2 x) is taken exactly from the exponent.
#include <algorithm>
#include <cfloat>

#include "common.hpp"

namespace remifa {
namespace {

constexpr int EQ_COLS = 128;  // columns per workgroup of the row-maxima pass
constexpr int EQ_SWEEP = 8;   // columns per thread of the scaling

// four consecutive rows (element-aligned: any leading dimension)
struct f4 {
  float e[4];
};
__device__ __forceinline__ f4 ld4(const float* p) {
  f4 v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}

// threads of a 256-thread workgroup along the rows (four rows each); the rest
// of them lie along the columns
int eq_rows_of_block(int64_t m) {
  int bx = 256;
  while (bx > 8 && (int64_t)bx * 2 >= m) bx /= 2;
  return bx;
}

__device__ __forceinline__ float pow2_trunc_log2(float x) {
  int e;
  const float f = frexpf(x, &e);  // x = f 2^e, f in [0.5, 1)
  const int k = (x >= 1.0f || f == 0.5f) ? e - 1 : e;
  return ldexpf(1.0f, k);
}

__global__ void fill_u32_kernel(unsigned* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// rmax[i] = max_j |a_ij| (as float bits): four rows per thread, eight
// columns' loads in flight; the threads along the columns meet in LDS, so that
// few rows are not one atomic per thread on a few words. A grid has at most
// 65535 workgroups along the columns: each takes chunks of EQ_COLS that far
// apart. Measured (MI355X) at 16384 x 16384: 244 us, 4.4 TB/s (one row per
// thread: 298 us).
__global__ void __launch_bounds__(256) row_absmax_kernel(int64_t m, int64_t n,
                                                         const float* __restrict__ a, int64_t lda,
                                                         unsigned* __restrict__ rmax) {
  __shared__ float4 part[256];
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  const int dj = blockDim.y;
  float mx[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t j0 = (int64_t)blockIdx.y * EQ_COLS; j0 < n; j0 += (int64_t)gridDim.y * EQ_COLS) {
    const int64_t j1 = std::min<int64_t>(n, j0 + EQ_COLS);
    int64_t j = j0 + threadIdx.y;
    if (i + 4 <= m) {
      for (; j + 7 * dj < j1; j += 8 * dj) {
        f4 v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = ld4(a + i + (j + c * dj) * lda);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], fabsf(v[c].e[r]));
      }
      for (; j < j1; j += dj) {
        const f4 v = ld4(a + i + j * lda);
#pragma unroll
        for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], fabsf(v.e[r]));
      }
    } else if (i < m) {
      for (; j < j1; j += dj)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          mx[r] = fmaxf(mx[r], fabsf(a[(i + r < m ? i + r : i) + j * lda]));
    }
  }
  if (dj > 1) {  // (uniform)
    part[threadIdx.y * blockDim.x + threadIdx.x] = make_float4(mx[0], mx[1], mx[2], mx[3]);
    __syncthreads();
    if (threadIdx.y > 0) return;
    for (int y = 1; y < dj; ++y) {
      const float4 v = part[y * blockDim.x + threadIdx.x];
      mx[0] = fmaxf(mx[0], v.x), mx[1] = fmaxf(mx[1], v.y);
      mx[2] = fmaxf(mx[2], v.z), mx[3] = fmaxf(mx[3], v.w);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (i + r < m) atomicMax(rmax + i + r, __float_as_uint(mx[r]));
}

// min, max and (as an index) minimum over a 1024-thread workgroup, in every
// thread
struct Extrema {
  float mn, mx;
  int z;
};
__device__ __forceinline__ Extrema block_extrema(Extrema e) {
  __shared__ Extrema w[16];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    e.mn = fminf(e.mn, __shfl_xor(e.mn, d, 64));
    e.mx = fmaxf(e.mx, __shfl_xor(e.mx, d, 64));
    e.z = std::min(e.z, __shfl_xor(e.z, d, 64));
  }
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = e;
  __syncthreads();
  e = w[0];
#pragma unroll
  for (int q = 1; q < 16; ++q) {
    e.mn = fminf(e.mn, w[q].mn);
    e.mx = fmaxf(e.mx, w[q].mx);
    e.z = std::min(e.z, w[q].z);
  }
  return e;
}

// vectors of scales are read eight entries per thread at a time, so that one
// workgroup (they need a global minimum and maximum) is not bound by the
// latency of each read
constexpr int EQ_VB = 8;

// one workgroup: powers of the row maxima, their min / max, INFO, then r
// (out[0] = rowcnd, out[1] = amax, info[0] = first zero row + 1 or 0)
__global__ void __launch_bounds__(1024) row_scale_kernel(int64_t m,
                                                         const unsigned* __restrict__ rmax,
                                                         float* __restrict__ r,
                                                         float* __restrict__ out,
                                                         int* __restrict__ info) {
  const int t = threadIdx.x;
  Extrema e{FLT_MAX, 0.0f, INT32_MAX};
  for (int64_t i0 = t; i0 < m; i0 += 1024 * EQ_VB) {
    float v[EQ_VB];
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t i = i0 + 1024 * b;
      v[b] = __uint_as_float(rmax[i < m ? i : i0]);
    }
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t i = i0 + 1024 * b;
      if (i >= m) break;
      if (v[b] > 0.0f) v[b] = pow2_trunc_log2(v[b]);
      e.mn = fminf(e.mn, v[b]);
      e.mx = fmaxf(e.mx, v[b]);
      if (v[b] == 0.0f) e.z = std::min<int>(e.z, (int)i);
    }
  }
  e = block_extrema(e);
  const float smlnum = FLT_MIN, bignum = 1.0f / FLT_MIN;
  if (t == 0) {
    out[1] = e.mx;
    info[0] = e.z == INT32_MAX ? 0 : e.z + 1;
    out[0] = fmaxf(fminf(e.mn, bignum), smlnum) / fminf(e.mx, bignum);
  }
  const bool zero_row = e.z != INT32_MAX;  // then r holds the powers
  for (int64_t i0 = t; i0 < m; i0 += 1024 * EQ_VB) {
    float v[EQ_VB];
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t i = i0 + 1024 * b;
      v[b] = __uint_as_float(rmax[i < m ? i : i0]);
    }
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t i = i0 + 1024 * b;
      if (i >= m) break;
      if (v[b] > 0.0f) v[b] = pow2_trunc_log2(v[b]);
      r[i] = zero_row ? v[b] : 1.0f / fminf(fmaxf(v[b], smlnum), bignum);
    }
  }
}

// c[j] = 2^trunc(log2 max_i |a_ij| r_i): a workgroup per column, four rows
// per thread and four sweeps of loads in flight. Measured (MI355X) at
// 16384 x 16384: 171 us, 6.3 TB/s (one row per thread: 293 us).
__global__ void __launch_bounds__(256) col_absmax_kernel(int64_t m, int64_t n,
                                                         const float* __restrict__ a,
                                                         int64_t lda, const float* __restrict__ r,
                                                         const int* __restrict__ info,
                                                         float* __restrict__ c) {
  __shared__ float red[4];
  if (info[0] != 0) return;  // a zero row: LAPACK returns before the columns
  // columns from the last to the first: the row pass left the last ones in
  // the last-level cache
  const int64_t j = n - 1 - blockIdx.x;
  const float* const p = a + j * lda;
  float mx = 0.0f;
  int64_t i = (int64_t)threadIdx.x * 4;
  for (; i + 3 * 1024 + 4 <= m; i += 4 * 1024) {
    f4 v[4], w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = ld4(p + i + 1024 * q);
      w[q] = ld4(r + i + 1024 * q);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fabsf(v[q].e[e]) * w[q].e[e]);
  }
  for (; i < m; i += 1024)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t ie = i + e < m ? i + e : i;
      mx = fmaxf(mx, fabsf(p[ie]) * r[ie]);
    }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    c[j] = mx > 0.0f ? pow2_trunc_log2(mx) : 0.0f;
  }
}

// one workgroup: min / max of the column powers, INFO, then c
// (out[2] = colcnd; info[0] = m + first zero column + 1 if no zero row)
__global__ void __launch_bounds__(1024) col_scale_kernel(int64_t m, int64_t n,
                                                         float* __restrict__ c,
                                                         float* __restrict__ out,
                                                         int* __restrict__ info) {
  if (info[0] != 0) return;
  const int t = threadIdx.x;
  Extrema e{FLT_MAX, 0.0f, INT32_MAX};
  for (int64_t j0 = t; j0 < n; j0 += 1024 * EQ_VB) {
    float v[EQ_VB];
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t j = j0 + 1024 * b;
      v[b] = c[j < n ? j : j0];
    }
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t j = j0 + 1024 * b;
      if (j >= n) break;
      e.mn = fminf(e.mn, v[b]);
      e.mx = fmaxf(e.mx, v[b]);
      if (v[b] == 0.0f) e.z = std::min<int>(e.z, (int)j);
    }
  }
  e = block_extrema(e);
  const float smlnum = FLT_MIN, bignum = 1.0f / FLT_MIN;
  if (e.z != INT32_MAX) {
    if (t == 0) info[0] = (int)(m + e.z + 1);
    return;
  }
  if (t == 0) out[2] = fmaxf(fminf(e.mn, bignum), smlnum) / fminf(e.mx, bignum);
  for (int64_t j0 = t; j0 < n; j0 += 1024 * EQ_VB) {
    float v[EQ_VB];
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t j = j0 + 1024 * b;
      v[b] = c[j < n ? j : j0];
    }
#pragma unroll
    for (int b = 0; b < EQ_VB; ++b) {
      const int64_t j = j0 + 1024 * b;
      if (j < n) c[j] = 1.0f / fminf(fmaxf(v[b], smlnum), bignum);
    }
  }
}

// a_ij <- s a_ij for EQUED 'R' (r_i), 'C' (c_j), 'B' ((c_j r_i) a_ij): four
// rows and EQ_SWEEP columns per thread, the loads of all of them before the
// stores (r once for the eight columns). One-dimensional grid: row blocks
// first (rb of them). Measured (MI355X) at 16384 x 16384: 339 us,
// 6.3 TB/s (one element per thread: 676 us).
template <int MODE>
__global__ void __launch_bounds__(256) scale_kernel(int64_t m, int64_t n, int64_t rb,
                                                    float* __restrict__ a, int64_t lda,
                                                    const float* __restrict__ r,
                                                    const float* __restrict__ c) {
  const int64_t i = ((blockIdx.x % rb) * blockDim.x + threadIdx.x) * 4;
  const int64_t j0 = ((blockIdx.x / rb) * blockDim.y + threadIdx.y) * EQ_SWEEP;
  if (i >= m || j0 >= n) return;
  auto scaled = [](float x, float ri, float cj) {
    if constexpr (MODE == 0) return ri * x;
    if constexpr (MODE == 1) return cj * x;
    return (cj * ri) * x;
  };
  if (i + 4 <= m && j0 + EQ_SWEEP <= n) {
    f4 ri = {{1.0f, 1.0f, 1.0f, 1.0f}}, v[EQ_SWEEP];
    if constexpr (MODE != 1) ri = ld4(r + i);
#pragma unroll
    for (int q = 0; q < EQ_SWEEP; ++q) v[q] = ld4(a + i + (j0 + q) * lda);
#pragma unroll
    for (int q = 0; q < EQ_SWEEP; ++q) {
      const float cj = MODE != 0 ? c[j0 + q] : 1.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[q].e[e] = scaled(v[q].e[e], ri.e[e], cj);
      __builtin_memcpy(a + i + (j0 + q) * lda, &v[q], sizeof(f4));
    }
  } else {
    for (int64_t j = j0; j < n && j < j0 + EQ_SWEEP; ++j) {
      const float cj = MODE != 0 ? c[j] : 1.0f;
      for (int e = 0; e < 4 && i + e < m; ++e) {
        float* const p = a + i + e + j * lda;
        *p = scaled(*p, MODE != 1 ? r[i + e] : 1.0f, cj);
      }
    }
  }
}

}  // namespace
}  // namespace remifa

using namespace remifa;

extern "C" {

int remifa_geequb(remifa_handle_t h, int64_t m, int64_t n, const float* d_a, int64_t lda,
                  float* d_r, float* d_c, float* rowcnd, float* colcnd, float* amax, int* info) {
  if (!h) return -1;
  if (m < 0 || m > INT32_MAX) return -2;
  if (n < 0 || n > INT32_MAX) return -3;
  if (!d_a && m > 0 && n > 0) return -4;
  if (lda < std::max<int64_t>(m, 1)) return -5;
  if (!d_r && m > 0) return -6;
  if (!d_c && n > 0) return -7;
  if (!rowcnd) return -8;
  if (!colcnd) return -9;
  if (!amax) return -10;
  if (!info) return -11;
  *info = 0;
  if (m == 0 || n == 0) {
    *rowcnd = 1.0f;
    *colcnd = 1.0f;
    *amax = 0.0f;
    return 0;
  }
  // workspace: row maxima (m), results (rowcnd, amax, colcnd), info
  RF_CHECK(ensure_workspace(h, sizeof(unsigned) * (size_t)m + 256));
  unsigned* rmax = (unsigned*)h->ws;
  char* tail = (char*)h->ws + ((sizeof(unsigned) * (size_t)m + 127) & ~(size_t)127);
  float* out = (float*)tail;
  int* dinfo = (int*)(tail + 3 * sizeof(float));
  hipStream_t s = h->stream;
  fill_u32_kernel<<<(unsigned)ceil_div(m, 256), 256, 0, s>>>(rmax, m);
  const int bx = eq_rows_of_block(m);
  const unsigned gy = (unsigned)std::min<int64_t>(ceil_div(n, EQ_COLS), 65535);
  row_absmax_kernel<<<dim3((unsigned)ceil_div(m, 4 * bx), gy), dim3(bx, 256 / bx), 0, s>>>(
      m, n, d_a, lda, rmax);
  row_scale_kernel<<<1, 1024, 0, s>>>(m, rmax, d_r, out, dinfo);
  col_absmax_kernel<<<(unsigned)n, 256, 0, s>>>(m, n, d_a, lda, d_r, dinfo, d_c);
  col_scale_kernel<<<1, 1024, 0, s>>>(m, n, d_c, out, dinfo);
  RF_HIP(hipGetLastError());
  struct {
    float o[3];
    int info;
  } back;  // out and info are neighbours: one copy
  RF_HIP(hipMemcpyAsync(&back, out, sizeof(back), hipMemcpyDeviceToHost, s));
  RF_HIP(hipStreamSynchronize(s));
  const float* const ho = back.o;
  const int hi = back.info;
  *info = hi;
  *amax = ho[1];
  if (hi > 0 && hi <= m) return 0;  // zero row: LAPACK leaves rowcnd / colcnd unset
  *rowcnd = ho[0];
  if (hi > m) return 0;  // zero column: colcnd unset
  *colcnd = ho[2];
  return 0;
}

int remifa_laqge(remifa_handle_t h, int64_t m, int64_t n, float* d_a, int64_t lda,
                 const float* d_r, const float* d_c, float rowcnd, float colcnd, float amax,
                 char* equed) {
  if (!h) return -1;
  if (m < 0 || n < 0) return m < 0 ? -2 : -3;
  if (n > INT32_MAX) return -3;
  if (!d_a && m > 0 && n > 0) return -4;
  if (lda < std::max<int64_t>(m, 1)) return -5;
  if (!equed) return -11;
  if (m == 0 || n == 0) {
    *equed = 'N';
    return 0;
  }
  const float thresh = 0.1f;
  const float small = ldexpf(1.0f, -103), large = 1.0f / small;  // SLAMCH('S') / SLAMCH('P')
  int mode;
  if (rowcnd >= thresh && amax >= small && amax <= large) {
    if (colcnd >= thresh) {
      *equed = 'N';
      return 0;
    }
    mode = 1;
    *equed = 'C';
  } else if (colcnd >= thresh) {
    mode = 0;
    *equed = 'R';
  } else {
    mode = 2;
    *equed = 'B';
  }
  if ((mode != 1 && !d_r)) return -6;
  if ((mode != 0 && !d_c)) return -7;
  const int64_t rb = ceil_div(m, 256);
  if (rb * n > INT32_MAX) return -2;
  const int bx = eq_rows_of_block(m);
  const int64_t sb = ceil_div(m, 4 * bx);
  const unsigned g = (unsigned)(sb * ceil_div(n, (int64_t)(256 / bx) * EQ_SWEEP));
  const dim3 blk(bx, 256 / bx);
  hipStream_t s = h->stream;
  timer_begin(h, KC_CONVERT, 8.0 * (double)m * (double)n, 3);
  if (mode == 0) scale_kernel<0><<<g, blk, 0, s>>>(m, n, sb, d_a, lda, d_r, d_c);
  if (mode == 1) scale_kernel<1><<<g, blk, 0, s>>>(m, n, sb, d_a, lda, d_r, d_c);
  if (mode == 2) scale_kernel<2><<<g, blk, 0, s>>>(m, n, sb, d_a, lda, d_r, d_c);
  timer_end(h);
  RF_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
