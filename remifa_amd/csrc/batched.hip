// Batched no-pivot LU and solve of many independent small matrices (orders
// up to 512), fp32 storage with matrix-core updates (TC32: fp16 operands,
// fp32 accumulation; BF16_TC32: bf16 operands).
//
// One persistent launch: a grid of as many workgroups as the chip holds (or
// as there are matrices) takes matrices from an atomic queue (callers order
// the batch largest first, so the queue is a longest-processing-time
// schedule). A workgroup factors its matrix right-looking with 32-wide
// panels, which is the reference's RL driver with nb = ib = 32
// (src/lu_nopiv.hxx:53-208): per panel
//  1. the 32 pivots of the panel: lane i keeps row i of the panel in
//     registers; wavefront 0 factors the top 32 x 32 block (pivot rows by
//     readlane), then every lane takes its row below against U11 from LDS,
//     pivots in order: reciprocal, multiply, fused update in fp32
//     (src/lu_nopiv.cu:123-170), two barriers per panel;
//  2. the block row U12 = L11^-1 A12, one lane per column;
//  3. the Schur update A22 -= L21 U12 on the matrix cores from fp16 (bf16)
//     copies of L21 and U12 staged in LDS, products summed from zero and
//     subtracted once (the update GEMMs of gemm.hip do the same); two or four
//     32 x 32 tiles of C per wavefront in flight together.
// The matrix stays in HBM; every element of the trailing matrix is read and
// written once per panel, which is what bounds large batches of orders above
// 256 (about 7 TB/s over the chip); the pivots and the two triangular steps (25
// us per panel of order 500, against 24 us of update) run under another
// workgroup's update.
//
// Two instantiations. MANY: 128 registers per lane, so that four wavefronts
// share a SIMD and hide each other's latencies, two tiles of C in flight. The
// other: one wavefront per SIMD with all its registers (none spilled) and four
// tiles in flight, for batches whose time is that of a matrix or two per
// workgroup, and for the smallest orders, whose panels are all latency. Measured
// (MI355X, us, orders 33 to 64 / 65 to 128 / 129 to 256 / 257 to 512), MANY against
// the other: 32 matrices 49 / 106 / 257 / 675 and 39 / 82 / 188 / 628; 600 matrices
// 54 / 122 / 311 / 1240 and 43 / 103 / 351 / 1141; 1500 matrices 79 / 152 / 491 /
// 2527 and 76 / 188 / 772 / 2619; 4000 matrices 148 / 324 / 1167 / 6681 and 139 /
// 468 / 2037 / 6931.
//
// The batched solve runs one workgroup per matrix: x in LDS, 32-row blocks,
// the 32x32 diagonal block substitution inside one wavefront, the rest of
// each block column as a matrix-vector update by all lanes.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace remifa {
namespace {

constexpr int PW = 32;     // panel width
constexpr int BMAX = 512;  // largest order

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// LDS of a workgroup for orders up to BM: 69 KB for 512, so that two
// workgroups share a CU and one's serial pivots run under the other's updates
template <int BM>
struct BatchLds {
  uint16_t Lh[BM - PW][PW];  // L21 (rows below the panel's top block), fp16/bf16 bits
  uint16_t Ut[BM - PW][PW];  // U12 transposed: [column][k]
  __attribute__((aligned(16))) float L11[PW][PW];   // the panel's top block (unit L and U)
  __attribute__((aligned(16))) float L11t[PW][PW];  // its transpose
  float Rk[PW];           // reciprocals of the panel's pivots
  int item;
  int info;
};

// 16-byte unit c (k-values 8 c .. 8 c + 7) of row r of a staged operand: rows
// are 64 bytes without padding, units permuted so that the rows of a read
// phase hit different banks
__device__ __forceinline__ int unit_at(int r, int c) { return 8 * (c ^ ((r >> 2) & 3)); }

template <bool BF>
__device__ __forceinline__ uint16_t op_bits(float v) {
  if constexpr (BF)
    return f32_to_bf16_bits(v);
  else
    return __builtin_bit_cast(uint16_t, (half_t)v);
}

// BM: largest order taken (a size bucket), BT: threads (BT >= BM: one lane
// per row of a panel and per column of a block row)
template <bool BF, int BM, int BT, bool MANY>
__global__ void __launch_bounds__(BT, MANY ? 4 : 1)
    batched_lu_kernel(int count, const int* __restrict__ d_n, const int* __restrict__ d_ld,
                      float* const* __restrict__ d_ptrs, int* __restrict__ d_info,
                      int* __restrict__ queue) {
  static_assert(BT >= BM && BT >= 64 && BT % 64 == 0, "one lane per row");
  __shared__ BatchLds<BM> S;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int l32 = lane & 31, lh = lane >> 5;
  for (;;) {
    if (t == 0) {
      S.item = __hip_atomic_fetch_add(queue, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      S.info = 0;
    }
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(S.item);  // (uniform addresses below)
    if (item >= count) break;  // every workgroup reaches this: the grid drains
    const int n = d_n[item];
    const int64_t ld = d_ld[item];
    float* __restrict__ a = d_ptrs[item];
    if (n <= 0 || n > BM) {
      if (t == 0 && d_info) d_info[item] = n > BM ? -1 : 0;
      __syncthreads();
      continue;
    }
    for (int k0 = 0; k0 < n; k0 += PW) {
      const int pw = n - k0 < PW ? n - k0 : PW;
      const int mp = n - k0;  // rows of the panel
      // ---- 1. the panel's pivots, row t in registers
      float x[PW];
      {
        const int r = t < mp ? t : mp - 1;
#pragma unroll
        for (int j = 0; j < PW; ++j) {
          const int jc = j < pw ? j : pw - 1;
          const float v = (a + k0 + (int64_t)(k0 + jc) * ld)[(unsigned)r];
          x[j] = (t < mp && j < pw) ? v : (t == j ? 1.0f : 0.0f);
        }
      }
      // (a) the top pw x pw block inside wavefront 0: lane i < pw holds row
      // i; pivot kk's row comes to every lane by readlane
      if (wave == 0) {
#pragma unroll
        for (int kk = 0; kk < PW; ++kk) {
          if (kk < pw) {
            float u[PW];
#pragma unroll
            for (int j = kk; j < PW; ++j)
              u[j] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(
                                                   __builtin_bit_cast(int, x[j]), kk));
            const float p = u[kk];
            const float rk = 1.0f / p;
            if (t == 0) {
              S.Rk[kk] = rk;
              if ((p == 0.0f || !__builtin_isfinite(p)) && S.info == 0) S.info = k0 + kk + 1;
            }
            if (t > kk && t < PW && t < mp) {
              const float lk = x[kk] * rk;
              x[kk] = lk;
#pragma unroll
              for (int j = kk + 1; j < PW; ++j) x[j] = __builtin_fmaf(-lk, u[j], x[j]);
            }
          }
        }
        if (t < PW) {
#pragma unroll
          for (int j = 0; j < PW; ++j) S.L11[t][j] = x[j];
#pragma unroll
          for (int j = 0; j < PW; ++j) S.L11t[j][t] = x[j];
        }
      }
      __syncthreads();
      // (b) every row below it against U11, pivots in order (the same
      // operations as the pivot-by-pivot elimination)
      if (t >= PW && t < mp) {
#pragma unroll
        for (int kk = 0; kk < PW; ++kk) {
          if (kk < pw) {
            // row kk of U11 as 16-byte broadcast reads
            float ur[PW];
#pragma unroll
            for (int j = (kk + 1) / 4 * 4; j < PW; j += 4) {
              const float4 v = *(const float4*)&S.L11[kk][j];
              ur[j] = v.x, ur[j + 1] = v.y, ur[j + 2] = v.z, ur[j + 3] = v.w;
            }
            const float lk = x[kk] * S.Rk[kk];
            x[kk] = lk;
#pragma unroll
            for (int j = kk + 1; j < PW; ++j) x[j] = __builtin_fmaf(-lk, ur[j], x[j]);
          }
        }
      }
      // store the panel; keep L11/U11 (fp32) and L21 (operand precision)
      if (t < mp) {
#pragma unroll
        for (int j = 0; j < PW; ++j)
          if (j < pw) (a + k0 + (int64_t)(k0 + j) * ld)[(unsigned)t] = x[j];
      }
      const int mr = n - k0 - pw;  // rows (and columns) of the trailing matrix
      const int mr32 = (mr + 31) & ~31;
      if (t >= PW && t - PW < mr32) {
        const int r = t - PW;
        u16x8 v[PW / 8];
#pragma unroll
        for (int j = 0; j < PW; ++j) v[j / 8][j % 8] = r < mr ? op_bits<BF>(x[j]) : (uint16_t)0;
#pragma unroll
        for (int q = 0; q < PW / 8; ++q) *(u16x8*)&S.Lh[r][unit_at(r, q)] = v[q];
      }
      __syncthreads();
      if (mr <= 0) continue;
      // ---- 2. U12 = L11^-1 A12, one lane per column
      if (t < mr32) {
        const int c = t < mr ? t : mr - 1;
        float* col = a + k0 + (int64_t)(k0 + pw + c) * ld;
        float u[PW];  // (the column's 128 bytes as 16-byte accesses, element-aligned)
        __builtin_memcpy(u, col, sizeof(u));
#pragma unroll
        for (int kk = 0; kk < PW; ++kk) {
          {
            // column kk of L11 (row kk of its transpose), 16-byte reads
            float lc[PW];
#pragma unroll
            for (int i = (kk + 1) / 4 * 4; i < PW; i += 4) {
              const float4 v = *(const float4*)&S.L11t[kk][i];
              lc[i] = v.x, lc[i + 1] = v.y, lc[i + 2] = v.z, lc[i + 3] = v.w;
            }
#pragma unroll
            for (int i = kk + 1; i < PW; ++i) u[i] = __builtin_fmaf(-lc[i], u[kk], u[i]);
          }
        }
        if (t < mr) __builtin_memcpy(col, u, sizeof(u));
        u16x8 v[PW / 8];
#pragma unroll
        for (int i = 0; i < PW; ++i) v[i / 8][i % 8] = t < mr ? op_bits<BF>(u[i]) : (uint16_t)0;
#pragma unroll
        for (int q = 0; q < PW / 8; ++q) *(u16x8*)&S.Ut[t][unit_at(t, q)] = v[q];
      }
      __syncthreads();
      // ---- 3. A22 -= L21 U12 on the matrix cores, 32 x 32 tiles, two per
      // wavefront at a time (their C entries read in one round trip)
      const int nt = mr32 / 32;
      constexpr int TQ = MANY ? 2 : 4;
      for (int tile0 = wave; tile0 < nt * nt; tile0 += TQ * (BT / 64)) {
        f16v acc[TQ];
        float cv[TQ][16];
#pragma unroll
        for (int z = 0; z < TQ; ++z) {
          const int tile = tile0 + z * (BT / 64);
          const int tc = tile < nt * nt ? tile : 0;
          const int tm = tc % nt, tn = tc / nt;
          const int m = tm * 32 + l32;
          const float* cm = a + (k0 + pw + (m < mr ? m : 0)) + (int64_t)(k0 + pw) * ld;
#pragma unroll
          for (int q = 0; q < 16; ++q) {
            const int nn = tn * 32 + 4 * lh + 8 * (q >> 2) + (q & 3);
            cv[z][q] = cm[(int64_t)(nn < mr ? nn : 0) * ld];
          }
#pragma unroll
          for (int q = 0; q < 16; ++q) acc[z][q] = 0.0f;
#pragma unroll
          for (int ks = 0; ks < PW; ks += 16) {
            const int rb = tn * 32 + l32, ra = tm * 32 + l32, c = ks / 8 + lh;
            const u16x8 xb = *(const u16x8*)&S.Ut[rb][unit_at(rb, c)];
            const u16x8 ya = *(const u16x8*)&S.Lh[ra][unit_at(ra, c)];
            if constexpr (BF)
              acc[z] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  __builtin_bit_cast(bf8, xb), __builtin_bit_cast(bf8, ya), acc[z], 0, 0, 0);
            else
              acc[z] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                  __builtin_bit_cast(h8, xb), __builtin_bit_cast(h8, ya), acc[z], 0, 0, 0);
          }
        }
        // lane holds C[m = tm*32 + l32][n = tn*32 + 4 lh + 8 (q / 4) + q % 4]
#pragma unroll
        for (int z = 0; z < TQ; ++z) {
          const int tile = tile0 + z * (BT / 64);
          const int tm = tile % nt, tn = tile / nt;
          const int m = tm * 32 + l32;
          if (tile < nt * nt && m < mr) {
            float* cm = a + (k0 + pw + m) + (int64_t)(k0 + pw) * ld;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
              const int nn = tn * 32 + 4 * lh + 8 * (q >> 2) + (q & 3);
              if (nn < mr) cm[(int64_t)nn * ld] = cv[z][q] - acc[z][q];
            }
          }
        }
      }
      __syncthreads();  // the trailing matrix is complete before the next panel
    }
    if (t == 0 && d_info) d_info[item] = S.info;
    __syncthreads();
  }
}

// lane k's value in every lane
__device__ __forceinline__ float lane_value(float v, int k) {
  return __builtin_bit_cast(float,
                            __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}

// One matrix per workgroup: b <- (L U)^-1 b with the factors in place. Bound by
// the latency of a 32-column step (a read of the factors, the substitution, two
// barriers): the step's entries of the factors, which do not depend on the
// solution, are all requested before the substitution, NV rows of the update
// per thread. BT threads and NV for the caller's largest order (64 threads up
// to 64, 256 and one row up to 288, else two rows); an order above it still
// takes the remaining rows one by one. Measured (MI355X), 2000 matrices of
// order 257 to 512: 739 -> 375 us; 129 to 256: 285 -> 121 us; 16 to
// 64: 25 -> 19 us.
template <int BT, int NV>
__global__ void __launch_bounds__(BT) batched_getrs_kernel(int count, const int* __restrict__ d_n,
                                                            const int* __restrict__ d_ld,
                                                            float* const* __restrict__ d_ptrs,
                                                            float* const* __restrict__ d_b) {
  __shared__ float xs[BMAX];
  const int item = blockIdx.x;
  const int n = d_n[item];
  if (n <= 0 || n > BMAX) return;  // uniform: the whole workgroup leaves
  const int64_t ld = d_ld[item];
  const float* __restrict__ a = d_ptrs[item];
  float* __restrict__ b = d_b[item];
  const int t = threadIdx.x;
  for (int i = t; i < n; i += BT) xs[i] = b[i];
  __syncthreads();
  // row i (in bounds) of the columns k0 .. k0 + kw - 1, the last repeated
  auto read_row = [&](int i, int k0, int kw, float (&w)[32]) {
#pragma unroll
    for (int k = 0; k < 32; ++k)
      w[k] = (a + (int64_t)(k0 + (k < kw ? k : kw - 1)) * ld)[(unsigned)i];
  };
  // x_i -= the row's products with x_k0 .. in order
  auto update = [&](int i, int k0, int kw, const float (&w)[32]) {
    float s = xs[i];
#pragma unroll
    for (int k = 0; k < 32; ++k)
      if (k < kw) s = __builtin_fmaf(-w[k], xs[k0 + k], s);
    xs[i] = s;
  };
  float rowv[32], w0[32], w1[32];  // (w1: two rows per thread)
  // forward: unit lower L
  for (int k0 = 0; k0 < n; k0 += 32) {
    const int kw = n - k0 < 32 ? n - k0 : 32;
    const int i0 = k0 + kw + t, below = n - k0 - kw;
    if (t < 64) read_row(k0 + (t < kw ? t : 0), k0, kw, rowv);
    if (t < below) read_row(i0, k0, kw, w0);
    if (NV == 2 && t + BT < below) read_row(i0 + BT, k0, kw, w1);
    if (t < 64) {
      // the diagonal block inside one wavefront (lanes 0..kw-1 own its rows)
      float xi = t < kw ? xs[k0 + t] : 0.0f;
#pragma unroll
      for (int k = 0; k < 32; ++k) {
        if (k < kw) {
          const float xk = lane_value(xi, k);
          if (t > k && t < kw) xi = __builtin_fmaf(-rowv[k], xk, xi);
        }
      }
      if (t < kw) xs[k0 + t] = xi;
    }
    __syncthreads();
    if (t < below) update(i0, k0, kw, w0);
    if (NV == 2 && t + BT < below) update(i0 + BT, k0, kw, w1);
    if constexpr (BT * NV < BMAX)
      for (int i = i0 + BT * NV; i < n; i += BT) {
        read_row(i, k0, kw, w0);
        update(i, k0, kw, w0);
      }
    __syncthreads();
  }
  // backward: upper U
  for (int k1 = n; k1 > 0; k1 -= 32) {
    const int k0 = k1 - 32 > 0 ? k1 - 32 : 0;
    const int kw = k1 - k0;
    if (t < 64) read_row(k0 + (t < kw ? t : 0), k0, kw, rowv);
    if (t < k0) read_row(t, k0, kw, w0);
    if (NV == 2 && t + BT < k0) read_row(t + BT, k0, kw, w1);
    if (t < 64) {
      float xi = t < kw ? xs[k0 + t] : 0.0f;
#pragma unroll
      for (int k = 31; k >= 0; --k) {
        if (k < kw) {
          if (t == k) xi = xi / rowv[k];
          const float xk = lane_value(xi, k);
          if (t < k) xi = __builtin_fmaf(-rowv[k], xk, xi);
        }
      }
      if (t < kw) xs[k0 + t] = xi;
    }
    __syncthreads();
    if (t < k0) update(t, k0, kw, w0);
    if (NV == 2 && t + BT < k0) update(t + BT, k0, kw, w1);
    if constexpr (BT * NV < BMAX)
      for (int i = t + BT * NV; i < k0; i += BT) {
        read_row(i, k0, kw, w0);
        update(i, k0, kw, w0);
      }
    __syncthreads();
  }
  for (int i = t; i < n; i += BT) b[i] = xs[i];
}

__global__ void zero_queue_kernel(int* q) {
  if (threadIdx.x == 0) q[0] = 0;
}

}  // namespace
}  // namespace remifa

using namespace remifa;

namespace remifa {
void batched_shape(remifa_handle_t h, int bm, int* bt, int* per_cu);
}

extern "C" int remifa_lu_nopiv_batched(remifa_handle_t h, int ctype, int64_t count, const int* d_n,
                                       const int* d_ld, float* const* d_ptrs, int* d_info,
                                       int max_n) {
  if (!h) return -1;
  if (ctype != REMIFA_TC32 && ctype != REMIFA_BF16_TC32) {
    set_last_error("remifa_lu_nopiv_batched: update types TC32 and BF16_TC32 are built");
    return REMIFA_ERR_UNSUPPORTED;
  }
  if (count < 0 || count > INT32_MAX) return -3;
  if (count > 0 && (!d_n || !d_ld || !d_ptrs)) return -4;
  if (max_n < 0 || max_n > BMAX) return -8;
  if (count == 0) return 0;
  // the queue counter lives in the handle's workspace; it is reset by a
  // kernel (not a memset), so the call can be captured in a graph
  RF_CHECK(ensure_workspace(h, 256));
  int* queue = (int*)h->ws;
  zero_queue_kernel<<<1, 64, 0, h->stream>>>(queue);
  // the size bucket of max_n picks the kernel (LDS for orders up to the
  // bucket's bound) and, from the handle's tuning table, its threads and
  // persistent workgroups per CU; count the instantiation (where the two take
  // the same time, see above) and at most as many workgroups as matrices
  int bm = 512;
  for (int b : {64, 128, 256})
    if (max_n <= b) {
      bm = b;
      break;
    }
  int bt = 0, per_cu = 0;
  batched_shape(h, bm, &bt, &per_cu);
  const bool many = bm > 64 && count > (bm == 128 ? 4 : (bm == 256 ? 2 : 3)) * (int64_t)h->num_cu;
  if (!many) per_cu = std::min(per_cu, std::max(1, 256 / bt));  // one wavefront per SIMD
  const int grid = (int)std::min<int64_t>((int64_t)per_cu * h->num_cu, count);
  timer_begin(h, KC_OTHER, 0.0, 1);
  int st = 0;
  auto launch = [&](auto bf, auto bmc, auto btc) {
    constexpr bool BF = decltype(bf)::value;
    constexpr int M = decltype(bmc)::value, T = decltype(btc)::value;
    if (M > 64 && many)
      batched_lu_kernel<BF, M, T, (M > 64)>
          <<<grid, T, 0, h->stream>>>((int)count, d_n, d_ld, d_ptrs, d_info, queue);
    else
      batched_lu_kernel<BF, M, T, false>
          <<<grid, T, 0, h->stream>>>((int)count, d_n, d_ld, d_ptrs, d_info, queue);
  };
#define RF_BATCHED(BM, BT)                              \
  if (bm == BM && bt == BT) {                           \
    using M = std::integral_constant<int, BM>;          \
    using T = std::integral_constant<int, BT>;          \
    if (ctype == REMIFA_TC32)                           \
      launch(std::false_type{}, M{}, T{});              \
    else                                                \
      launch(std::true_type{}, M{}, T{});               \
  } else
  RF_BATCHED(64, 64)
  RF_BATCHED(64, 128)
  RF_BATCHED(128, 128)
  RF_BATCHED(128, 256)
  RF_BATCHED(256, 256)
  RF_BATCHED(256, 512)
  RF_BATCHED(512, 512)
  st = REMIFA_ERR_UNSUPPORTED;
#undef RF_BATCHED
  timer_end(h);
  if (st) {
    set_last_error("remifa_lu_nopiv_batched: no kernel for this bucket / thread count");
    return st;
  }
  RF_HIP(hipGetLastError());
  return 0;
}

// Threads and workgroups per CU of the batched factorization for orders up
// to bm: the handle's table (remifa_set_batched_tuning) or the defaults.
void remifa::batched_shape(remifa_handle_t h, int bm, int* bt, int* per_cu) {
  *bt = bm;
  *per_cu = bm == 128 ? 8 : (bm <= 256 ? 4 : 2);
  for (const auto& r : h->batched_rules)
    if (r[0] == bm) {
      *bt = r[1];
      *per_cu = r[2];
    }
}

extern "C" int remifa_getrs_nopiv_batched(remifa_handle_t h, int64_t count, const int* d_n,
                                          const int* d_ld, float* const* d_ptrs,
                                          float* const* d_b, int max_n) {
  if (!h) return -1;
  if (count < 0 || count > INT32_MAX) return -2;
  if (count > 0 && (!d_n || !d_ld || !d_ptrs || !d_b)) return -3;
  if (max_n < 0 || max_n > BMAX) return -7;
  if (count == 0) return 0;
  timer_begin(h, KC_OTHER, 0.0, 2);
  const unsigned grid = (unsigned)count;
  if (max_n <= 64)
    batched_getrs_kernel<64, 1><<<grid, 64, 0, h->stream>>>((int)count, d_n, d_ld, d_ptrs, d_b);
  else if (max_n <= 288)
    batched_getrs_kernel<256, 1><<<grid, 256, 0, h->stream>>>((int)count, d_n, d_ld, d_ptrs, d_b);
  else
    batched_getrs_kernel<256, 2><<<grid, 256, 0, h->stream>>>((int)count, d_n, d_ld, d_ptrs, d_b);
  timer_end(h);
  RF_HIP(hipGetLastError());
  return 0;
}

// Batched tuning table: rules[3 i .. 3 i + 2] = (bucket bound, threads,
// workgroups per CU), bucket bound in {64, 128, 256, 512}, threads a
// multiple of 64 between the bound and twice it (at most 512), 1..16
// workgroups per CU. count = 0 restores the defaults.
extern "C" int remifa_set_batched_tuning(remifa_handle_t h, int count, const int* rules) {
  if (!h) return -1;
  if (count < 0 || count > 64) return -2;
  if (count > 0 && !rules) return -3;
  std::vector<std::array<int, 3>> r((size_t)count);
  for (int i = 0; i < count; ++i) {
    const int bm = rules[3 * i], bt = rules[3 * i + 1], pc = rules[3 * i + 2];
    const bool bm_ok = bm == 64 || bm == 128 || bm == 256 || bm == 512;
    const bool bt_ok = (bm == 64 && (bt == 64 || bt == 128)) ||
                       (bm == 128 && (bt == 128 || bt == 256)) ||
                       (bm == 256 && (bt == 256 || bt == 512)) || (bm == 512 && bt == 512);
    if (!bm_ok || !bt_ok || pc < 1 || pc > 16) return -3;
    r[i] = {bm, bt, pc};
  }
  h->batched_rules.swap(r);
  return 0;
}
