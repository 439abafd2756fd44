// Triangular solves with the stored no-pivot factors, the FP64 residual and
// iterative refinement.
//
// TRSM (forward L, backward U and the transposed pair for A^T): the 128 x 128
// diagonal blocks are inverted first, all in parallel (diag_inv_kernel), so
// the sequential chain of the substitution is one small matrix-vector product
// per block row instead of 128 dependent steps. Then one launch per triangle:
// workgroups take 128-row block rows in dependency order from an atomic
// ticket, so every block a workgroup waits for belongs to a workgroup that is
// already running (no deadlock whatever the residency). Block row i
// accumulates B_i - sum_j T_ij X_j, multiplies by its inverted diagonal block
// (from the seventh on, the last dependency is folded into it ahead of time:
// X_i = (T_ii)^-1 (B_i - sum of the others) - ((T_ii)^-1 T_i,i-1) X_i-1, so
// one product follows the last wait instead of two) and publishes X_i as
// tagged 64-bit words (value, 1) written with agent-scope atomic stores into
// a tag buffer cleared before the launches: a
// reader retries until every word it needs carries the tag, so a value and
// its "published" mark arrive together (one memory round trip per hop
// instead of store, wait, counter, poll, load). Every wait is bounded: on
// timeout the kernel records an error and exits, so the grid always drains.
// One right-hand side runs on vector fma, several on the fp32 matrix cores,
// groups of 16 side by side in one launch.
//
// Residual R = B - A X in FP64: A widened in registers, vector fma for one
// right-hand side, the FP64 matrix cores for several (up to 64 per read of A);
// partials over chunks of A summed in chunk order by a second kernel
// (deterministic), which in the refinement also rounds the next right-hand
// side and takes its norm.
#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"

namespace remifa {
namespace {

constexpr int NBS = 128;     // block size of the triangular solves
constexpr int TT = 4 * NBS;  // threads of a triangular-solve workgroup
constexpr int QC = NBS / 4;  // columns of a block per lane (column quarter)
constexpr int RC = 16;       // right-hand sides of a group
constexpr long long kSpinLimit = 1LL << 22;  // retries of a wait (each a memory round trip)

template <typename LT>
__device__ __forceinline__ float ldf(const LT* p) {
  return (float)*p;
}

// element T[r][c] of the effective triangle
template <typename LT, bool TRANS>
__device__ __forceinline__ float tel(const LT* lu, int64_t ld, int64_t r, int64_t c) {
  return TRANS ? ldf(lu + c + r * ld) : ldf(lu + r + c * ld);
}

typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));

// Inverses of the diagonal blocks: blockIdx.y = 0 for the unit lower L_bb,
// 1 for the upper U_bb. inv[b][r][c] (128 x 128 row-major per block); rows
// and columns past n are the identity. The eight 16 x 16 diagonal blocks are
// inverted by substitution (a lane per column); then three doublings: the
// off-diagonal half of a 2 s x 2 s inverse is -V22 D21 V11 (lower) or -V11
// D12 V22 (upper), s x s products in 16 x 16 tiles on the fp32 matrix cores.
// Latency-bound (two workgroups per block row, one pass). Measured (MI355X) at
// n = 1000: 19 us against 73 us with 64 x 64 substitutions (2016 dependent,
// fully unrolled steps, most of the time fetching their code).
template <typename LT>
__global__ void __launch_bounds__(256) diag_inv_kernel(int64_t n, const LT* __restrict__ lu,
                                                       int64_t ld, float* __restrict__ inv_l,
                                                       float* __restrict__ inv_u) {
  constexpr int P = NBS + 4;  // row pitch: the A fragments of a product hit every bank once
  __shared__ float D[NBS * P];
  __shared__ float V[NBS * P];  // the inverse
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int64_t r0 = (int64_t)blockIdx.x * NBS;
  const bool upper = blockIdx.y == 1;
  {
    const int r = t % NBS;
    const int64_t R = r0 + r, Rc = R < n ? R : n - 1;
#pragma unroll 32
    for (int z = 0; z < NBS / 2; ++z) {
      const int c = t / NBS + 2 * z;
      const int64_t C = r0 + c, Cc = C < n ? C : n - 1;
      const float v = ldf(lu + Rc + Cc * ld);
      D[r * P + c] = (R < n && C < n) ? v : (r == c ? 1.0f : 0.0f);
      V[r * P + c] = 0.0f;
    }
  }
  __syncthreads();
  if (t < NBS) {
    const int o = t & ~15, c = t & 15;
    const float* const d = &D[o * P + o];
    float x[16];
    if (!upper) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float s = (r == c) ? 1.0f : 0.0f;
#pragma unroll
        for (int k = 0; k < r; ++k) s = __builtin_fmaf(-d[r * P + k], x[k], s);
        x[r] = s;
      }
    } else {
#pragma unroll
      for (int r = 15; r >= 0; --r) {
        float s = (r == c) ? 1.0f : 0.0f;
#pragma unroll
        for (int k = r + 1; k < 16; ++k) s = __builtin_fmaf(-d[r * P + k], x[k], s);
        x[r] = s / d[r * P + r];
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) V[(o + r) * P + o + c] = x[r];
  }
  __syncthreads();
#pragma unroll 1
  for (int sz = 16; sz < NBS; sz *= 2) {
    const int tp = sz / 16, nt = NBS / (2 * sz) * tp * tp;
    // the corner of the off-diagonal block of pair p, and of the diagonal
    // blocks after / before it in the products
    const int ro = upper ? 0 : sz, co = upper ? sz : 0;
    auto product = [&](const float* A, int ai, int ak, const float* B, int bk, int bj) {
      f4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
      for (int k = 0; k < sz; k += 4)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[(ai + l16) * P + ak + k + lq],
                                                   B[(bk + k + lq) * P + bj + l16], acc, 0, 0, 0);
      return acc;
    };
    // P = D21 V11 (D12 V22), held in registers until every wave has read D
    f4v pr[4];
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const int tile = wave + 4 * z;
      if (tile < nt) {
        const int o = 2 * sz * (tile / (tp * tp)), ti = tile / tp % tp, tj = tile % tp;
        pr[z] = product(D, o + ro + 16 * ti, o + co, V, o + co, o + co + 16 * tj);
      }
    }
    __syncthreads();
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const int tile = wave + 4 * z;
      if (tile < nt) {
        const int o = 2 * sz * (tile / (tp * tp)), ti = tile / tp % tp, tj = tile % tp;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          D[(o + ro + 16 * ti + 4 * lq + j) * P + o + co + 16 * tj + l16] = pr[z][j];
      }
    }
    __syncthreads();
    // V21 = -V22 P (V12 = -V11 P)
    for (int tile = wave; tile < nt; tile += 4) {
      const int o = 2 * sz * (tile / (tp * tp)), ti = tile / tp % tp, tj = tile % tp;
      const f4v v = product(V, o + ro + 16 * ti, o + ro, D, o + ro, o + co + 16 * tj);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        V[(o + ro + 16 * ti + 4 * lq + j) * P + o + co + 16 * tj + l16] = -v[j];
    }
    __syncthreads();
  }
  float* const out = (upper ? inv_u : inv_l) + (int64_t)blockIdx.x * NBS * NBS;
#pragma unroll 8
  for (int z = 0; z < NBS / 2; ++z) {
    const int r = t / NBS + 2 * z;
    out[r * NBS + t % NBS] = V[r * P + t % NBS];
  }
}

// Block rows later than this in dependency order fold the last dependency
// into their inverted diagonal block: forming the product takes about as long
// as the chain needs to get that far.
constexpr int kFoldFrom = 6;

// One block row of T X = B per workgroup (see the file comment). Lane
// (row, cq) owns row `row` of the block and the column quarter cq (32
// columns) of every 128 x 128 block it multiplies; the four partial sums are
// added in LDS in a fixed order. One right-hand side. *ticket hands out the
// block rows, *err is the error flag; tags[r] = (value, 1) once entry r of the
// solution is published (both zeroed before the launch).
template <typename LT, bool LOWER, bool TRANS>
__global__ void __launch_bounds__(TT) trsm_kernel(int64_t n, const LT* __restrict__ lu,
                                                  int64_t ld, float* __restrict__ b,
                                                  const float* __restrict__ inv,
                                                  int* __restrict__ ticket, int* __restrict__ err,
                                                  unsigned long long* __restrict__ tags,
                                                  int nblk) {
  constexpr int CH = 2;  // solution blocks staged in LDS at a time
  // Xs and Red share their LDS with the near block of T, which is only read
  // before the first solution block is staged (a barrier between)
  static_assert(CH * NBS + 4 * NBS <= NBS * NBS, "shared with the near block");
  __shared__ __attribute__((aligned(16))) float ush[NBS * NBS];
  float* const Xs = ush;
  float(*const Red)[NBS] = reinterpret_cast<float(*)[NBS]>(ush + CH * NBS);
  float(*const Ts)[NBS] = reinterpret_cast<float(*)[NBS]>(ush);
  __shared__ int s_ticket;
  const int t = threadIdx.x;
  const int row = t % NBS, cq = t / NBS;
  if (t == 0)
    s_ticket = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int tk = s_ticket;
  const int bi = LOWER ? tk : nblk - 1 - tk;
  const int64_t gr = (int64_t)bi * NBS + row;

  // The last dependency (block tk-1 in dependency order, the "near" block)
  // is folded into the diagonal block's inverse ahead of time, M =
  // (T_ii)^-1 T_i,near, so that once X_near is published only X_i = C - M
  // X_near remains (one product and one reduction), with C = (T_ii)^-1 (B_i
  // - sum over the other blocks) formed while waiting.
  const bool fold = tk >= kFoldFrom;
  const int nsteps = fold ? tk - 1 : tk;  // blocks summed before the wait for the near one
  // rows of the stored factors start on 16 bytes (16-byte vector reads of
  // the transposed triangle's rows)
  const bool vec_rows =
      TRANS && ((uintptr_t)lu % 16 == 0) && (ld % (16 / (int64_t)sizeof(LT)) == 0);
  const int64_t grc = gr < n ? gr : n - 1;  // in-bounds row for the loads
  // (T_ii)^-1 in LDS (rows padded against bank conflicts; transposed for the
  // transposed triangles: (T_ii)^-1 = ((D_ii)^-1)^T), for M and the diagonal
  // product
  __shared__ float Ds[NBS][NBS + 1];
  {
    float dv[QC];
    const float* ib = inv + (int64_t)bi * NBS * NBS;
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const int col = cq * QC + c;
      dv[c] = TRANS ? ib[col * NBS + row] : ib[row * NBS + col];
    }
#pragma unroll
    for (int c = 0; c < QC; ++c) Ds[row][cq * QC + c] = dv[c];
  }
  // this lane's entry of b (lanes cq = 0), loaded now so that no memory round
  // trip follows the last dependency wait (only this workgroup writes these
  // rows of b)
  const float bv = b[grc];
  float mv[QC];
  if (fold) {
    // M: this lane's row and column quarter, from (T_ii)^-1 and T_i,near in
    // LDS
    const int bjn = LOWER ? tk - 1 : nblk - 1 - (tk - 1);
    const int64_t c0 = (int64_t)bjn * NBS + cq * QC;
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const int64_t C = c0 + c < n ? c0 + c : n - 1;
      const float v = tel<LT, TRANS>(lu, ld, grc, C);
      Ts[row][cq * QC + c] = (gr < n && c0 + c < n) ? v : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < QC; ++c) mv[c] = 0.0f;
#pragma unroll 2
    for (int k = 0; k < NBS; ++k) {
      const float d = Ds[row][k];
#pragma unroll
      for (int c = 0; c < QC; ++c) mv[c] = __builtin_fmaf(d, Ts[k][cq * QC + c], mv[c]);
    }
    __syncthreads();  // (Ts is Xs and Red from here on)
  }
  // the solution blocks s0 .. s0 + cnt - 1 (dependency order) into Xs:
  // agent-scope atomic loads of the tagged words, each wavefront retrying
  // its own until every one carries the published tag (a wavefront vote),
  // then one barrier; bounded, and a wavefront that gives up raises the
  // error flag that ends the others' waits
  auto stage_blocks = [&](int s0, int cnt) {
    for (long long tries = 0;; ++tries) {
      int bad = 0;
      for (int e = t; e < cnt * NBS; e += TT) {
        const int q = e / NBS, c = e % NBS;
        const int bj = LOWER ? s0 + q : nblk - 1 - (s0 + q);
        const int64_t C = (int64_t)bj * NBS + c;
        float v = 0.0f;
        if (C < n) {
          const unsigned long long w =
              __hip_atomic_load(&tags[C], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          bad |= (unsigned)(w >> 32) != 1u;
          v = __uint_as_float((unsigned)w);
        }
        Xs[e] = v;
      }
      if (__ballot(bad) == 0) break;
      if (tries > kSpinLimit ||
          ((tries & 63) == 63 &&
           __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        // give up (the host reports the error and discards the results)
        if ((t & 63) == 0)
          __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    __syncthreads();
  };
  float acc = 0.0f;
  for (int s0 = 0; s0 < nsteps; s0 += CH) {
    const int cnt = nsteps - s0 < CH ? nsteps - s0 : CH;
    // this lane's entries of the chunk's blocks of T: issued before the wait
    // (they do not depend on it), with clamped addresses and no branches so
    // the loads are all in flight together
    float tv[CH][QC];
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int qq = q < cnt ? q : cnt - 1;
      const int bj = LOWER ? s0 + qq : nblk - 1 - (s0 + qq);
      const int64_t c0 = (int64_t)bj * NBS + cq * QC;
      if (TRANS && vec_rows && gr < n && c0 + QC <= n) {
        // the transposed triangle: the lane's 32 entries are contiguous in
        // its row of the stored factors, read as 16-byte vectors
        const LT* pr = lu + c0 + grc * ld;
        if constexpr (sizeof(LT) == 2) {
          typedef _Float16 h8 __attribute__((ext_vector_type(8)));
#pragma unroll
          for (int u = 0; u < QC / 8; ++u) {
            const h8 v = *(const h8*)(pr + 8 * u);
#pragma unroll
            for (int j = 0; j < 8; ++j) tv[q][8 * u + j] = (float)v[j];
          }
        } else {
#pragma unroll
          for (int u = 0; u < QC / 4; ++u) {
            const float4 v = *(const float4*)(pr + 4 * u);
            tv[q][4 * u] = v.x, tv[q][4 * u + 1] = v.y, tv[q][4 * u + 2] = v.z,
                      tv[q][4 * u + 3] = v.w;
          }
        }
        continue;
      }
#pragma unroll
      for (int c = 0; c < QC; ++c) {
        const int64_t C = c0 + c < n ? c0 + c : n - 1;
        const float v = tel<LT, TRANS>(lu, ld, grc, C);
        tv[q][c] = (gr < n && c0 + c < n) ? v : 0.0f;
      }
    }
    stage_blocks(s0, cnt);
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      if (q < cnt) {
#pragma unroll
        for (int c = 0; c < QC; ++c)
          acc = __builtin_fmaf(tv[q][c], Xs[q * NBS + cq * QC + c], acc);
      }
    }
    __syncthreads();
  }

  // the sum of the four column quarters' parts, in a fixed order
  auto total = [&]() { return ((Red[0][row] + Red[1][row]) + Red[2][row]) + Red[3][row]; };
  // right-hand side of the diagonal block: B_i - sum_j T_ij X_j (over the
  // blocks summed so far)
  Red[cq][row] = acc;
  __syncthreads();
  if (cq == 0) Xs[row] = gr < n ? bv - total() : 0.0f;
  __syncthreads();
  // X_i = (T_ii)^-1 (B_i - ...)  (with the fold: C)
  float y = 0.0f;
#pragma unroll
  for (int c = 0; c < QC; ++c) y = __builtin_fmaf(Ds[row][cq * QC + c], Xs[cq * QC + c], y);
  Red[cq][row] = y;
  __syncthreads();
  float xv = cq == 0 ? total() : 0.0f;
  if (fold) {
    // then the near block: X_i = C - M X_near
    __syncthreads();  // (Red and Xs are rewritten below)
    stage_blocks(tk - 1, 1);
    float z = 0.0f;
#pragma unroll
    for (int c = 0; c < QC; ++c) z = __builtin_fmaf(mv[c], Xs[cq * QC + c], z);
    Red[cq][row] = z;
    __syncthreads();
    if (cq == 0) xv -= total();
  }
  if (cq == 0 && gr < n) {
    b[gr] = xv;  // the caller's copy
    __hip_atomic_store(&tags[gr], (1ull << 32) | (unsigned long long)__float_as_uint(xv),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The same for up to 16 right-hand sides at a time, the products on the fp32
// matrix cores (16x16x4): wavefront w owns rows 16 w .. 16 w + 15 of the
// block, so nothing is summed across wavefronts. A fragments: lane (i, q),
// i = lane % 16, q = lane / 16, holds T[16 w + i][32 q + s], s = 0..31 (one
// run per lane along the rows of the transposed triangles); B fragments: the
// staged solution block [s][q][rhs] in LDS. Groups of 16 right-hand sides run
// as independent chains of one launch (ticket = block row * ngrp + group).
// What bounds it is the hop from one block row to the next: publish, poll, one
// 128 x 128 x 16 product (2048 cycles at the fp32 matrix rate). Measured
// (MI355X) at n = 4096, 64 right-hand sides: 140 us per triangle against 4 x
// 225 us (one launch per 16, fma with LDS broadcasts, sums over quarters).
template <typename LT, bool LOWER, bool TRANS>
__global__ void __launch_bounds__(TT) trsm16_kernel(int64_t n, int nrhs, int ngrp,
                                                    const LT* __restrict__ lu, int64_t ld,
                                                    float* __restrict__ b, int64_t ldb,
                                                    const float* __restrict__ inv,
                                                    int* __restrict__ ticket,
                                                    int* __restrict__ err,
                                                    unsigned long long* __restrict__ tags,
                                                    int nblk) {
  constexpr int KS = 32;            // matrix-core steps of a 128-deep product
  constexpr int XP = 65;            // pitch of a step's 4 x 16 staged values
  constexpr int TQ = 144, TP = 577;  // near block [s][q][column]: conflict-free both ways
  constexpr int MP = NBS + 4;       // its product with the inverse [row][s][q]
  __shared__ float xs[2][KS * XP];
  __shared__ float big[KS * TP > NBS * MP ? KS * TP : NBS * MP];
  __shared__ int s_ticket;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  if (t == 0)
    s_ticket = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int tk = __builtin_amdgcn_readfirstlane(s_ticket / ngrp);
  const int grp = __builtin_amdgcn_readfirstlane(s_ticket % ngrp);
  const int nr = nrhs - RC * grp < RC ? nrhs - RC * grp : RC;
  b += (int64_t)RC * grp * ldb;
  tags += (int64_t)RC * grp * n;
  const int bi = LOWER ? tk : nblk - 1 - tk;
  const int64_t rb = (int64_t)bi * NBS;
  const int64_t gr = rb + 16 * w + l16;       // this lane's row of the A fragments
  const int64_t grc = gr < n ? gr : n - 1;    // (in-bounds for the loads)
  const int64_t go = rb + 16 * w + 4 * lq;    // rows go .. go + 3 of column l16 of results

  // A fragments of the inverted diagonal block (transposed for the transposed
  // triangles), its diagonal at this lane's results, and the right-hand side
  float dv[KS], dd[4];
  {
    const float* const ib = inv + (int64_t)bi * NBS * NBS;
#pragma unroll
    for (int j = 0; j < 4; ++j) dd[j] = ib[(16 * w + 4 * lq + j) * (NBS + 1)];
#pragma unroll
    for (int s = 0; s < KS; ++s)
      dv[s] = TRANS ? ib[(32 * lq + s) * NBS + 16 * w + l16]
                    : ib[(16 * w + l16) * NBS + 32 * lq + s];
  }
  float bv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float v = b[(go + j < n ? go + j : n - 1) + (l16 < nr ? l16 : 0) * ldb];
    bv[j] = (go + j < n && l16 < nr) ? v : 0.0f;
  }
  const bool vec_rows =
      TRANS && ((uintptr_t)lu % 16 == 0) && (ld % (16 / (int64_t)sizeof(LT)) == 0);
  // block bj of this block row of T as A fragments, 0 outside the matrix
  auto load_t = [&](int bj, float(&tv)[KS]) {
    const int64_t c0 = (int64_t)bj * NBS + 32 * lq;
    if (TRANS && vec_rows && (int64_t)(bi + 1) * NBS <= n && (int64_t)(bj + 1) * NBS <= n) {
      const LT* const p = lu + c0 + grc * ld;
      if constexpr (sizeof(LT) == 2) {
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
#pragma unroll
        for (int u = 0; u < KS / 8; ++u) {
          const h8 v = *(const h8*)(p + 8 * u);
#pragma unroll
          for (int e = 0; e < 8; ++e) tv[8 * u + e] = (float)v[e];
        }
      } else {
#pragma unroll
        for (int u = 0; u < KS / 4; ++u) {
          const float4 v = *(const float4*)(p + 4 * u);
          tv[4 * u] = v.x, tv[4 * u + 1] = v.y, tv[4 * u + 2] = v.z, tv[4 * u + 3] = v.w;
        }
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int64_t C = c0 + s < n ? c0 + s : n - 1;
      const float v = tel<LT, TRANS>(lu, ld, grc, C);
      tv[s] = (gr < n && c0 + s < n) ? v : 0.0f;
    }
  };
  auto product = [&](const float(&f)[KS], const float* x, f4v c) {
    f4v d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KS; s += 2) {
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(f[s], x[s * XP + lane], c, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x4f32(f[s + 1], x[(s + 1) * XP + lane], d, 0, 0, 0);
    }
    return c + d;
  };
  // solution block q (dependency order) into x: the tagged words, retried
  // until each carries the tag (a wavefront vote), then one barrier; bounded,
  // and a wavefront that gives up raises the flag that ends the others' waits
  auto stage = [&](int q, float* x) {
    const int64_t c0 = (int64_t)(LOWER ? q : nblk - 1 - q) * NBS;
    for (long long tries = 0;; ++tries) {
      int bad = 0;
      unsigned long long wd[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rr = t % NBS, k = t / NBS + 4 * i;
        wd[i] = 1ull << 32;
        if (c0 + rr < n && k < nr)
          wd[i] = __hip_atomic_load(&tags[c0 + rr + (int64_t)k * n], __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rr = t % NBS, k = t / NBS + 4 * i;
        bad |= (unsigned)(wd[i] >> 32) != 1u;
        x[(rr % KS) * XP + (rr / KS) * RC + k] = __uint_as_float((unsigned)wd[i]);
      }
      if (__ballot(bad) == 0) break;
      if (tries > kSpinLimit ||
          ((tries & 63) == 63 &&
           __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        // give up (the host reports the error and discards the results)
        if (lane == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    __syncthreads();
  };

  // with the fold: M = (T_ii)^-1 T_i,near, as A fragments
  const bool fold = tk >= kFoldFrom;
  const int nsteps = fold ? tk - 1 : tk;
  float mv[KS];
  if (fold) {
    const int64_t cn = (int64_t)(LOWER ? tk - 1 : nblk - 1 - (tk - 1)) * NBS;
#pragma unroll 8
    for (int e = t; e < NBS * NBS; e += TT) {
      // lanes along the stored columns
      const int k = TRANS ? e / NBS : e % NBS, c = TRANS ? e % NBS : e / NBS;
      const int64_t R = rb + k < n ? rb + k : n - 1, C = cn + c < n ? cn + c : n - 1;
      const float v = tel<LT, TRANS>(lu, ld, R, C);
      big[(k % KS) * TP + (k / KS) * TQ + c] = (rb + k < n && cn + c < n) ? v : 0.0f;
    }
    __syncthreads();
    f4v m[NBS / 16];
#pragma unroll
    for (int ct = 0; ct < NBS / 16; ++ct) {
      m[ct] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
        m[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(dv[s], big[s * TP + lq * TQ + 16 * ct + l16],
                                                     m[ct], 0, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < NBS / 16; ++ct) {
      const int c = 16 * ct + l16;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        big[(16 * w + 4 * lq + j) * MP + (c % KS) * 4 + c / KS] = m[ct][j];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; ++s) mv[s] = big[(16 * w + l16) * MP + 4 * s + lq];
  }

  // the inverted block's diagonal term last, on top of the sum of the others:
  // where it is the largest (factors of dominant matrices) the chain's
  // roundings are those of the small sum. Error against 64 bits, n = 100 to
  // 12000: 4.4e-8 to 6.0e-8, against 1.3e-7 to 1.7e-7 with the diagonal inside
  // the chain (the one-column kernel, which adds quarters: 1.2e-7).
#pragma unroll
  for (int s = 0; s < KS; ++s)
    if (32 * lq + s == 16 * w + l16) dv[s] = 0.0f;

  // B_i - sum over the solution blocks (the block's loads are in flight while
  // it waits for the solution); two staging buffers, one barrier per block
  f4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
  for (int q = 0; q < nsteps; ++q) {
    float tv[KS];
    load_t(LOWER ? q : nblk - 1 - q, tv);
    stage(q, xs[q & 1]);
    acc = product(tv, xs[q & 1], acc);
  }
  float* const xr = xs[nsteps & 1];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int rr = 16 * w + 4 * lq + j;
    xr[(rr % KS) * XP + (rr / KS) * RC + l16] = bv[j] - acc[j];
  }
  __syncthreads();
  f4v y = product(dv, xr, (f4v){0.0f, 0.0f, 0.0f, 0.0f}), z = {0.0f, 0.0f, 0.0f, 0.0f};
  if (fold) {
    float* const xn = xs[(nsteps + 1) & 1];
    stage(tk - 1, xn);
    z = product(mv, xn, z);
    y -= z;
  }
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    y[j] = __builtin_fmaf(dd[j], bv[j] - acc[j], y[j]);
    nan |= y[j] != y[j];
  }
  if (__ballot(nan) != 0) {
    // an infinite entry times the diagonal's place, zero above, is NaN: where
    // an entry is not finite its row takes the product with the diagonal in it
    const float* const ib = inv + (int64_t)bi * NBS * NBS;
    f4v yd = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 16
    for (int s = 0; s < KS; ++s)
      yd = __builtin_amdgcn_mfma_f32_16x16x4f32(TRANS ? ib[(32 * lq + s) * NBS + 16 * w + l16]
                                                      : ib[(16 * w + l16) * NBS + 32 * lq + s],
                                                xr[s * XP + lane], yd, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (!__builtin_isfinite(bv[j] - acc[j])) y[j] = yd[j] - z[j];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (go + j < n && l16 < nr) {
      __hip_atomic_store(&tags[go + j + (int64_t)l16 * n],
                         (1ull << 32) | (unsigned long long)__float_as_uint(y[j]),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (go + j < n && l16 < nr) b[go + j + l16 * ldb] = y[j];  // the caller's copy
}

// clears the sync words (the error flag only if asked: it is kept over the
// parts of a solve), the tagged words and a few FP64 maxima of the refinement
__global__ void clear_kernel(int* sync, int with_err, unsigned long long* tags, int64_t ntags,
                             double* nrm0, int n0, double* nrm1, int n1) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < ntags) tags[i] = 0;
  if (blockIdx.x == 0) {
    const int t = threadIdx.x;
    if (t == 0) sync[0] = 0;
    if (t == 1 && with_err) sync[1] = 0;
    if (t == 2) sync[2] = 0;
    for (int k = t; k < n0; k += 256) nrm0[k] = 0.0;
    for (int k = t; k < n1; k += 256) nrm1[k] = 0.0;
  }
}

// ---------------------------------------------------------------- residual
constexpr int RES_ROWS = 256;  // rows per workgroup (one per lane)
constexpr int RES_COLS = 512;  // columns per chunk
constexpr int RES_RHS = 16;    // right-hand sides of a matrix-core tile
constexpr int RES_T1 = 2048;   // rows per chunk of the transposed one-column pass

// One right-hand side. part[chunk][n] = sum over the chunk's columns j of
// a_ij x_j, in FP64: four interleaved accumulators (j mod 4) combined in a
// fixed order, so several loads are in flight per lane.
__global__ void __launch_bounds__(256) resid_partial_kernel(int64_t n, const float* __restrict__ a,
                                                            int64_t lda,
                                                            const double* __restrict__ x,
                                                            double* __restrict__ part) {
  __shared__ double xs[RES_COLS];
  const int64_t i = (int64_t)blockIdx.x * RES_ROWS + threadIdx.x;
  const int64_t j0 = (int64_t)blockIdx.y * RES_COLS;
  for (int c = threadIdx.x; c < RES_COLS; c += 256) xs[c] = j0 + c < n ? x[j0 + c] : 0.0;
  __syncthreads();
  if (i >= n) return;
  const int jn = (int)(n - j0 < RES_COLS ? n - j0 : RES_COLS);
  const float* ai = a + i + j0 * lda;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  int j = 0;
  for (; j + 8 <= jn; j += 8) {
    float av[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) av[q] = ai[(int64_t)(j + q) * lda];
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q & 3] = __builtin_fma((double)av[q], xs[j + q], s[q & 3]);
  }
  for (; j < jn; ++j) s[j & 3] = __builtin_fma((double)ai[(int64_t)j * lda], xs[j], s[j & 3]);
  part[(int64_t)blockIdx.y * n + i] = (s[0] + s[1]) + (s[2] + s[3]);
}

// The same for R = B - A^T X: entry i is column i of A dotted with x over the
// chunk's rows. 16 lanes per column (64-byte contiguous reads of the column),
// 16 columns per workgroup; the 16 lane sums of a column are added in lane
// order (deterministic).
__global__ void __launch_bounds__(256) resid_t_partial_kernel(int64_t n,
                                                              const float* __restrict__ a,
                                                              int64_t lda,
                                                              const double* __restrict__ x,
                                                              double* __restrict__ part) {
  __shared__ double xs[RES_T1];
  __shared__ double red[16][16];
  const int t = threadIdx.x;
  const int c = t / 16, q = t % 16;
  const int64_t i = (int64_t)blockIdx.x * 16 + c;  // column of A = entry of r
  const int64_t j0 = (int64_t)blockIdx.y * RES_T1;
  for (int jj = t; jj < RES_T1; jj += 256) xs[jj] = j0 + jj < n ? x[j0 + jj] : 0.0;
  __syncthreads();
  double s = 0.0;
  if (i < n) {
    const int jn = (int)(n - j0 < RES_T1 ? n - j0 : RES_T1);
    const float* ac = a + j0 + i * lda;
#pragma unroll 8
    for (int jj = q; jj < jn; jj += 16) s = __builtin_fma((double)ac[jj], xs[jj], s);
  }
  red[c][q] = s;
  __syncthreads();
  if (q == 0 && i < n) {
    double v = 0.0;
    for (int r = 0; r < 16; ++r) v += red[c][r];
    part[(int64_t)blockIdx.y * n + i] = v;
  }
}

// Two to 16 GR right-hand sides: A X (A^T X) on the FP64 matrix cores
// (16x16x4, A widened in registers), part[chunk][n][nrhs]. A wavefront owns
// 64 entries of the result (rows of A, or columns for A^T), a workgroup 256,
// over jc columns (rows) of A. Plain: a lane reads four consecutive rows of a
// column, 16 lanes 256 bytes of it, and component e of the read belongs to
// tile e (rows 4 m + e). Transposed: a lane reads four consecutive rows of its
// column, component e being one of the four k-values 4 q + e of step e.
// HBM-bound up to 16 columns (one read of A), bound by the FP64 matrix rate
// (72 TFLOP/s) at 64. Measured (MI355X) at n = 4096, 64 right-hand sides: 62
// us (plain) and 66 us (transposed) against 4 x 68 and 4 x 177 us (one pass
// per 16 columns, vector fma).
template <int GR, bool TRANS>
__global__ void __launch_bounds__(256) resid_mm_kernel(int64_t n, int nrhs,
                                                       const float* __restrict__ a, int64_t lda,
                                                       const double* __restrict__ x, int64_t ldx,
                                                       double* __restrict__ part, int64_t jc,
                                                       int vec) {
  constexpr int JS = 32;                // columns (rows) of A staged at a time
  constexpr int PX = 16 * GR + 16;      // row pitch of the staged X
  __shared__ double xs[JS * PX];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * 256 + 64 * w;
  const int64_t jb = (int64_t)blockIdx.y * jc, je = jb + jc < n ? jb + jc : n;
  d4v acc[4][GR];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < GR; ++g) acc[i][g] = (d4v){0.0, 0.0, 0.0, 0.0};
  const bool inside = vec && m0 + 64 <= n;  // (uniform over the wavefront)
  for (int64_t j0 = jb; j0 < je; j0 += JS) {
    __syncthreads();
#pragma unroll 8
    for (int e = t; e < JS * 16 * GR; e += 256) {
      const int j = e % JS, k = e / JS;
      xs[j * PX + k] = (j0 + j < je && k < nrhs) ? x[j0 + j + k * ldx] : 0.0;
    }
    // eight 16-byte pieces of A: plain, columns j0 + 4 z + q, rows m0 + 4
    // l16 ..; transposed, column m0 + 16 (z / 2) + l16, rows j0 + 16 (z % 2)
    // + 4 q ..
    float4 v[8];
    if (inside && j0 + JS <= je) {
#pragma unroll
      for (int z = 0; z < 8; ++z)
        v[z] = TRANS ? *(const float4*)(a + j0 + 16 * (z & 1) + 4 * lq +
                                        (m0 + 16 * (z >> 1) + l16) * lda)
                     : *(const float4*)(a + m0 + 4 * l16 + (j0 + 4 * z + lq) * lda);
    } else {
#pragma unroll
      for (int z = 0; z < 8; ++z) {
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t i = TRANS ? m0 + 16 * (z >> 1) + l16 : m0 + 4 * l16 + e;
          const int64_t j = TRANS ? j0 + 16 * (z & 1) + 4 * lq + e : j0 + 4 * z + lq;
          const int64_t ic = i < n ? i : n - 1, jj = j < je ? j : je - 1;
          const float y = TRANS ? a[jj + ic * lda] : a[ic + jj * lda];
          f[e] = (i < n && j < je) ? y : 0.0f;
        }
        v[z] = make_float4(f[0], f[1], f[2], f[3]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int z = 0; z < 8; ++z) {
      const double av[4] = {v[z].x, v[z].y, v[z].z, v[z].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // plain: tile e, k = 4 z + q; transposed: tile z / 2, k = 16 (z % 2) +
        // 4 q + e
        const double* const xr =
            &xs[(TRANS ? 16 * (z & 1) + 4 * lq + e : 4 * z + lq) * PX + l16];
#pragma unroll
        for (int g = 0; g < GR; ++g) {
          d4v& c = acc[TRANS ? z >> 1 : e][g];
          c = __builtin_amdgcn_mfma_f64_16x16x4f64(av[e], xr[16 * g], c, 0, 0, 0);
        }
      }
    }
  }
  // lane (l16, q) holds entries 4 j + q of right-hand side l16 of each tile
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = 4 * j + lq;
      const int64_t row = m0 + (TRANS ? 16 * i + m : 4 * m + i);
      if (row < n) {
#pragma unroll
        for (int g = 0; g < GR; ++g)
          if (16 * g + l16 < nrhs)
            part[((int64_t)blockIdx.y * n + row) * nrhs + 16 * g + l16] = acc[i][g][j];
      }
    }
}

// maximum of |v| over a workgroup's lanes into *out (bit patterns of
// non-negative doubles order like the values, NaN above all; *out starts at
// zero)
__device__ __forceinline__ void block_absmax(double v, double* out) {
  __shared__ unsigned long long red[4];
  unsigned long long m = (unsigned long long)__double_as_longlong(fabs(v));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long u = __shfl_xor(m, o, 64);
    m = u > m ? u : m;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < 4; ++q) m = red[q] > m ? red[q] : m;
    atomicMax((unsigned long long*)out, m);
  }
}

// r = b - the partials, chunk by chunk (chunk order: deterministic). ONE: one
// right-hand side, else nrhs per entry (a workgroup takes 16 entries of 16
// right-hand sides). With w: the fp32 copy the correction solve takes, and max
// |r| per column, instead of r.
template <bool ONE>
__global__ void __launch_bounds__(256) resid_reduce_kernel(int64_t n, int nrhs, int nchunk,
                                                           const double* __restrict__ part,
                                                           const double* __restrict__ b,
                                                           int64_t ldb, double* __restrict__ r,
                                                           int64_t ldr, float* __restrict__ w,
                                                           double* __restrict__ rmax) {
  const int t = threadIdx.x;
  if constexpr (ONE) {
    const int64_t i = (int64_t)blockIdx.x * 256 + t;
    double v = 0.0;
    if (i < n) {
      double s = 0.0;
#pragma unroll 8
      for (int c = 0; c < nchunk; ++c) s += part[(int64_t)c * n + i];
      v = b[i] - s;
      if (w)
        w[i] = (float)v;
      else
        r[i] = v;
    }
    if (rmax) block_absmax(v, rmax);
  } else {
    __shared__ unsigned long long red[16][16];
    const int k = 16 * blockIdx.y + t % 16, q = t / 16;
    const int64_t i = (int64_t)blockIdx.x * 16 + q;
    double v = 0.0;
    if (i < n && k < nrhs) {
      double s = 0.0;
#pragma unroll 8
      for (int c = 0; c < nchunk; ++c) s += part[((int64_t)c * n + i) * nrhs + k];
      v = b[i + k * ldb] - s;
      if (w)
        w[i + k * n] = (float)v;
      else
        r[i + k * ldr] = v;
    }
    if (rmax) {
      red[q][t % 16] = (unsigned long long)__double_as_longlong(fabs(v));
      __syncthreads();
      if (q == 0 && k < nrhs) {
        unsigned long long m = red[0][t];
        for (int e = 1; e < 16; ++e) m = red[e][t] > m ? red[e][t] : m;
        atomicMax((unsigned long long*)(rmax + k), m);
      }
    }
  }
}

// ---------------------------------------------------------------- IR helpers
__global__ void d2f_kernel(int64_t n, int nrhs, const double* __restrict__ src, int64_t lds,
                           float* __restrict__ dst, int64_t ldd) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i + blockIdx.y * ldd] = (float)src[i + blockIdx.y * lds];
}
// x = w (assign) or x += w, and max |x| per column
__global__ void __launch_bounds__(256) axpy_f2d_kernel(int64_t n, const float* __restrict__ w,
                                                       int64_t ldw, double* __restrict__ x,
                                                       int64_t ldx, int assign,
                                                       double* __restrict__ xmax) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  double v = 0.0;
  if (i < n) {
    v = (double)w[i + blockIdx.y * ldw];
    double* p = x + i + blockIdx.y * ldx;
    if (!assign) v += *p;
    *p = v;
  }
  block_absmax(v, xmax + blockIdx.y);
}

// max_j sum_i |a_ij| (one-norm) and per-column inf norms, FP64
__global__ void colsum_kernel(int64_t n, const float* __restrict__ a, int64_t lda,
                              double* __restrict__ cs) {
  __shared__ double red[256];
  const int64_t j = blockIdx.x;
  double s = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 256) s += fabs((double)a[i + j * lda]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) cs[j] = red[0];
}

// rs[i] = sum_j |a_ij| (one-norm of A^T): 64 rows per workgroup, 16 lanes per
// row (columns j mod 16), added in lane order. Measured (MI355X) at n = 4096:
// below 50 us against 996 us with one lane per row (16 workgroups).
__global__ void __launch_bounds__(1024) rowsum_kernel(int64_t n, const float* __restrict__ a,
                                                      int64_t lda, double* __restrict__ rs) {
  __shared__ double red[16][64];
  const int r = threadIdx.x % 64, g = threadIdx.x / 64;
  const int64_t i = (int64_t)blockIdx.x * 64 + r;
  double s = 0.0;
  if (i < n) {
#pragma unroll 8
    for (int64_t j = g; j < n; j += 16) s += fabs((double)a[i + j * lda]);
  }
  red[g][r] = s;
  __syncthreads();
  if (g == 0 && i < n) {
    double v = 0.0;
    for (int q = 0; q < 16; ++q) v += red[q][r];
    rs[i] = v;
  }
}

// out[k] = max_i |v_ik| (NaN propagates); one workgroup per column
__global__ void colmax_kernel(int64_t n, const double* __restrict__ v, int64_t ldv,
                              double* __restrict__ out) {
  __shared__ double red[256];
  const int k = blockIdx.x;
  double m = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 256) {
    double x = fabs(v[i + k * ldv]);
    m = (x > m || x != x) ? x : m;
  }
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      double o = red[threadIdx.x + w];
      double s = red[threadIdx.x];
      red[threadIdx.x] = (o > s || o != o) ? o : s;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[k] = red[0];
}

__global__ void __launch_bounds__(1024) maxreduce_kernel(int64_t n, const double* __restrict__ v,
                                                         double* __restrict__ out) {
  __shared__ double red[1024];
  double m = 0.0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < n; i += 1024) m = fmax(m, v[i]);
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

}  // namespace

// solve workspace: sync words (ticket of the first triangle, error flag,
// ticket of the second), the inverted diagonal blocks of L and of U, and the
// tagged solution words: nset sets (one per triangle, or one used twice) of
// ngrp groups of 16 right-hand sides
struct TrsmWs {
  int* sync;
  float* inv_l;
  float* inv_u;
  unsigned long long* tags;
  int ngrp, nset;
};

// groups of 16 right-hand sides that run as chains of one launch, at most
constexpr int kMaxGroups = 8;

static size_t trsm_ws_bytes(int64_t n, int ngrp = 1, int nset = 1) {
  return 256 + 2 * sizeof(float) * NBS * NBS * (size_t)ceil_div(n, NBS) +
         sizeof(unsigned long long) * (size_t)n * RC * ngrp * nset;
}

static TrsmWs trsm_ws(void* p, int64_t n, int ngrp = 1, int nset = 1) {
  char* c = (char*)p;
  const size_t inv = sizeof(float) * NBS * NBS * (size_t)ceil_div(n, NBS);
  return TrsmWs{(int*)c, (float*)(c + 256), (float*)(c + 256 + inv),
                (unsigned long long*)(c + 256 + 2 * inv), ngrp, nset};
}

namespace {

template <typename LT, bool LOWER, bool TRANS>
int launch_trsm(remifa_handle_t h, int64_t n, int nrhs, bool one, int set, const void* lu,
                int64_t ld, float* b, int64_t ldb, const float* inv, const TrsmWs& w) {
  const int nblk = (int)ceil_div(n, NBS);
  int* const ticket = w.sync + (set ? 2 : 0);
  unsigned long long* const tags = w.tags + (size_t)set * n * RC * w.ngrp;
  if (one) {
    trsm_kernel<LT, LOWER, TRANS><<<nblk, TT, 0, h->stream>>>(n, (const LT*)lu, ld, b, inv, ticket,
                                                              w.sync + 1, tags, nblk);
  } else {
    const int ngrp = (nrhs + RC - 1) / RC;
    trsm16_kernel<LT, LOWER, TRANS><<<nblk * ngrp, TT, 0, h->stream>>>(
        n, nrhs, ngrp, (const LT*)lu, ld, b, ldb, inv, ticket, w.sync + 1, tags, nblk);
  }
  RF_HIP(hipGetLastError());
  return 0;
}

// nrm0 / nrm1 (n0, n1 doubles): cleared with the first sync words
template <typename LT>
int getrs_typed(remifa_handle_t h, int trans, int64_t n, int64_t nrhs, const void* lu,
                int64_t ld, float* b, int64_t ldb, const TrsmWs& w, double* nrm0, int n0,
                double* nrm1, int n1) {
  const int64_t step = (int64_t)RC * w.ngrp;
  // the kernel is the call's choice, not a remainder's: a column's solution
  // does not depend on how the columns are grouped
  const bool one = nrhs == 1;
  auto clear = [&](int nr, int sets, bool first) {
    // the words in use: whole columns of the groups of each set
    const int64_t nt = (sets - 1) * n * RC * w.ngrp + n * (int64_t)nr;
    clear_kernel<<<(unsigned)ceil_div(nt, 256), 256, 0, h->stream>>>(
        w.sync, first, w.tags, nt, nrm0, first ? n0 : 0, nrm1, first ? n1 : 0);
  };
  for (int64_t k0 = 0; k0 < nrhs; k0 += step) {
    const int nr = (int)std::min<int64_t>(step, nrhs - k0);
    float* bk = b + k0 * ldb;
    clear(nr, w.nset, k0 == 0);
    const int s2 = w.nset - 1;  // tag set of the second triangle
    if (!trans)
      RF_CHECK((launch_trsm<LT, true, false>(h, n, nr, one, 0, lu, ld, bk, ldb, w.inv_l, w)));
    else  // A^T = U^T L^T: U^T (lower) then L^T (upper, unit)
      RF_CHECK((launch_trsm<LT, true, true>(h, n, nr, one, 0, lu, ld, bk, ldb, w.inv_u, w)));
    if (s2 == 0) clear(nr, 1, false);
    if (!trans)
      RF_CHECK((launch_trsm<LT, false, false>(h, n, nr, one, s2, lu, ld, bk, ldb, w.inv_u, w)));
    else
      RF_CHECK((launch_trsm<LT, false, true>(h, n, nr, one, s2, lu, ld, bk, ldb, w.inv_l, w)));
  }
  return 0;
}

}  // namespace

// groups of right-hand sides and tag sets for a solve of nrhs columns whose
// other workspace takes `rest` bytes: as many as run side by side; with a
// caller's workspace, what fits it (one group and one set always do where a
// call was accepted before)
static void trsm_shape(remifa_handle_t h, int64_t n, int64_t nrhs, size_t rest, int* ngrp,
                       int* nset) {
  *ngrp = (int)std::min<int64_t>(kMaxGroups, ceil_div(nrhs, RC));
  *nset = 2;
  if (h->ws_user && trsm_ws_bytes(n, *ngrp, *nset) + rest > h->ws_bytes) *ngrp = *nset = 1;
}

// invert the diagonal blocks of the stored factors (once per factorization)
static int trsm_invert_launch(remifa_handle_t h, int lu_t, int64_t n, const void* lu, int64_t ld,
                              const TrsmWs& w) {
  const int nblk = (int)ceil_div(n, NBS);
  timer_begin(h, KC_TRSM, (double)n * NBS * (lu_t == REMIFA_R_16F ? 2 : 4) * 2, 1);
  if (lu_t == REMIFA_R_16F)
    diag_inv_kernel<half_t><<<dim3(nblk, 2), 256, 0, h->stream>>>(n, (const half_t*)lu, ld,
                                                                  w.inv_l, w.inv_u);
  else
    diag_inv_kernel<float><<<dim3(nblk, 2), 256, 0, h->stream>>>(n, (const float*)lu, ld, w.inv_l,
                                                                 w.inv_u);
  RF_HIP(hipGetLastError());
  timer_end(h);
  return 0;
}

// (L U) X = B or (L U)^T X = B in place in b; the diagonal blocks must have
// been inverted into w
int getrs_launch(remifa_handle_t h, int lu_t, int trans, int64_t n, int64_t nrhs, const void* lu,
                 int64_t ld, float* b, int64_t ldb, const TrsmWs& w, double* nrm0 = nullptr,
                 int n0 = 0, double* nrm1 = nullptr, int n1 = 0) {
  if (n == 0 || nrhs == 0) return 0;
  // bytes: both triangles read once per 16 right-hand sides
  const double es = lu_t == REMIFA_R_16F ? 2.0 : 4.0;
  timer_begin(h, KC_TRSM, (double)n * (double)n * es * (double)ceil_div(nrhs, RC), 0);
  int st = lu_t == REMIFA_R_16F ? getrs_typed<half_t>(h, trans, n, nrhs, lu, ld, b, ldb, w, nrm0,
                                                      n0, nrm1, n1)
                                : getrs_typed<float>(h, trans, n, nrhs, lu, ld, b, ldb, w, nrm0,
                                                     n0, nrm1, n1);
  timer_end(h);
  return st;
}

// right-hand sides of one residual pass: one, or up to 16, 32 or 64 on the
// matrix cores; lean: up to 16 in chunks of 256, for a caller's workspace (the
// smallest accepted one holds their partials)
static int resid_group(int64_t nrhs, bool lean) {
  if (nrhs == 1) return 1;
  return (nrhs <= RES_RHS || lean ? 1 : (nrhs <= 2 * RES_RHS ? 2 : 4)) * RES_RHS;
}
// Chunks that the sum over A is cut into: enough workgroups to fill the chip,
// two (16 columns four) per CU, each chunk at least one staged piece of 32
// long. Measured (MI355X, us, 16 columns, two with chunks of 256 against four):
// n = 130 27 / 12, n = 1000 40 / 13, n = 12000 324 / 215, n = 20000 832 / 560 (eight
// per CU: n = 12000 182, n = 8000 76 against 66).
static int64_t resid_chunks(int64_t n, int trans, int kw, bool lean) {
  if (kw == 1) return trans ? ceil_div(n, RES_T1) : ceil_div(n, RES_COLS);
  const int64_t want = ceil_div(kw == RES_RHS ? 1024 : 512, ceil_div(n, 256));
  return std::min(ceil_div(n, lean ? 256 : 32), want);
}

static size_t resid_part_bytes(int64_t n, int64_t nrhs, bool lean) {
  const int kw = resid_group(nrhs, lean);
  // the largest of the two layouts
  const int64_t ch = std::max(resid_chunks(n, 0, kw, lean), resid_chunks(n, 1, kw, lean));
  return sizeof(double) * (size_t)ch * (size_t)std::min<int64_t>(kw, nrhs) * (size_t)n;
}

// R = B - A X (A^T X when trans): to r, or to w (fp32, leading dimension n)
// with the columns' max |r| in rmax
int residual_launch(remifa_handle_t h, int64_t n, int64_t nrhs, const float* a, int64_t lda,
                    const double* x, int64_t ldx, const double* b, int64_t ldb, double* r,
                    int64_t ldr, double* part, int trans, bool lean, float* w = nullptr,
                    double* rmax = nullptr) {
  if (n == 0 || nrhs == 0) return 0;
  const int kw = resid_group(nrhs, lean);
  // bytes: A once per pass
  timer_begin(h, KC_RESID, 4.0 * (double)n * (double)n * (double)ceil_div(nrhs, kw), trans);
  const int vec = (uintptr_t)a % 16 == 0 && lda % 4 == 0;
  for (int64_t k0 = 0; k0 < nrhs; k0 += kw) {
    const int nr = (int)std::min<int64_t>(kw, nrhs - k0);
    const int nchunk0 = (int)resid_chunks(n, trans, kw, lean);
    const int64_t jc = ceil_div(ceil_div(n, nchunk0), 32) * 32;
    const int nchunk = kw == 1 ? nchunk0 : (int)ceil_div(n, jc);
    const double *xk = x + k0 * ldx, *bk = b + k0 * ldb;
    double *rk = r ? r + k0 * ldr : nullptr, *mk = rmax ? rmax + k0 : nullptr;
    float* const wk = w ? w + k0 * n : nullptr;
    hipStream_t s = h->stream;
    if (kw == 1) {
      if (trans)
        resid_t_partial_kernel<<<dim3((unsigned)ceil_div(n, 16), nchunk), 256, 0, s>>>(n, a, lda,
                                                                                       xk, part);
      else
        resid_partial_kernel<<<dim3((unsigned)ceil_div(n, RES_ROWS), nchunk), 256, 0, s>>>(
            n, a, lda, xk, part);
      resid_reduce_kernel<true><<<(unsigned)ceil_div(n, 256), 256, 0, s>>>(n, 1, nchunk, part, bk,
                                                                        ldb, rk, ldr, wk, mk);
      continue;
    }
    const dim3 g1((unsigned)ceil_div(n, 256), nchunk);
    const dim3 g2((unsigned)ceil_div(n, 16), (unsigned)ceil_div(nr, 16));
#define RF_RESID(GR)                                                                            \
  if (trans)                                                                                    \
    resid_mm_kernel<GR, true><<<g1, 256, 0, s>>>(n, nr, a, lda, xk, ldx, part, jc, vec);        \
  else                                                                                          \
    resid_mm_kernel<GR, false><<<g1, 256, 0, s>>>(n, nr, a, lda, xk, ldx, part, jc, vec);       \
  resid_reduce_kernel<false><<<g2, 256, 0, s>>>(n, nr, nchunk, part, bk, ldb, rk, ldr, wk, mk)
    if (kw == RES_RHS) {
      RF_RESID(1);
    } else if (kw == 2 * RES_RHS) {
      RF_RESID(2);
    } else {
      RF_RESID(4);
    }
#undef RF_RESID
  }
  timer_end(h);
  RF_HIP(hipGetLastError());
  return 0;
}

}  // namespace remifa

using namespace remifa;

extern "C" {

int remifa_getrs_nopiv(remifa_handle_t h, int lu_t, int trans, int64_t n, int64_t nrhs,
                       const void* d_lu, int64_t ldlu, float* d_b, int64_t ldb) {
  if (!h) return -1;
  if (lu_t != REMIFA_R_32F && lu_t != REMIFA_R_16F) return -2;
  if (n < 0) return -4;
  if (nrhs < 0) return -5;
  if (!d_lu && n > 0) return -6;
  if (ldlu < std::max<int64_t>(n, 1)) return -7;
  if (!d_b && n > 0 && nrhs > 0) return -8;
  if (ldb < std::max<int64_t>(n, 1)) return -9;
  if (n == 0 || nrhs == 0) return 0;
  int ngrp, nset;
  trsm_shape(h, n, nrhs, 0, &ngrp, &nset);
  RF_CHECK(ensure_workspace(h, trsm_ws_bytes(n, ngrp, nset)));
  const TrsmWs w = trsm_ws(h->ws, n, ngrp, nset);
  RF_CHECK(trsm_invert_launch(h, lu_t, n, d_lu, ldlu, w));
  RF_CHECK(getrs_launch(h, lu_t, trans, n, nrhs, d_lu, ldlu, d_b, ldb, w));
  int err = 0;
  RF_HIP(hipMemcpyAsync(&err, w.sync + 1, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  RF_HIP(hipStreamSynchronize(h->stream));
  if (err) {
    set_last_error("triangular solve: dependency wait timed out");
    return REMIFA_ERR_HIP;
  }
  return 0;
}

}  // extern "C"

// ---------------------------------------------------------------- no-allocation solve
// Scratch of remifa_getrs_nopiv_noalloc: a file-scope device array sized for
// the largest order it takes (sync words, the inverted 128 x 128 diagonal
// blocks of L and U, the n x 16 tagged solution words: trsm_ws_bytes(n)).
// Every GPU holds its own copy for the life of the process. Host code never
// uses the array's name as an address: its device address comes from
// hipGetSymbolAddress, once per device (noalloc_scratch).
namespace remifa {
namespace {
constexpr int64_t kNoAllocMaxN = 32768;
constexpr size_t kNoAllocBytes = 256 + 2 * sizeof(float) * NBS * NBS * (kNoAllocMaxN / NBS) +
                                 sizeof(unsigned long long) * kNoAllocMaxN * RC;
static_assert(kNoAllocMaxN % NBS == 0, "whole diagonal blocks");
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {};
}  // namespace

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

// device address of this device's scratch array (looked up on the first call
// for the device, which must be current)
int noalloc_scratch(int device, void** ptr) {
  *ptr = nullptr;
  if (device < 0 || device >= kMaxDevices) {
    set_last_error("device index out of range of the scratch table");
    return REMIFA_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[device]) {
    void* p = nullptr;
    RF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[device] = p;
  }
  *ptr = g_scratch[device];
  return 0;
}

size_t noalloc_scratch_bytes() { return kNoAllocBytes; }
}  // namespace remifa

extern "C" {

int remifa_getrs_nopiv_noalloc(remifa_handle_t h, int lu_t, int trans, int64_t n, int64_t nrhs,
                               const void* d_lu, int64_t ldlu, float* d_b, int64_t ldb) {
  if (!h) return -1;
  if (lu_t != REMIFA_R_32F && lu_t != REMIFA_R_16F) return -2;
  if (n < 0) return -4;
  if (nrhs < 0) return -5;
  if (!d_lu && n > 0) return -6;
  if (ldlu < std::max<int64_t>(n, 1)) return -7;
  if (!d_b && n > 0 && nrhs > 0) return -8;
  if (ldb < std::max<int64_t>(n, 1)) return -9;
  if (n > kNoAllocMaxN) {
    set_last_error("remifa_getrs_nopiv_noalloc: n = " + std::to_string(n) +
                   " exceeds the largest order of its static scratch, " +
                   std::to_string(kNoAllocMaxN));
    return REMIFA_ERR_WORKSPACE;
  }
  if (n == 0 || nrhs == 0) return 0;
  if (!h->scratch) {
    set_last_error("remifa_getrs_nopiv_noalloc: no scratch address for this handle's device");
    return REMIFA_ERR_HIP;
  }
  // the kernels of remifa_getrs_nopiv on the static scratch; the timer is
  // held off (its event pool would grow), the sync words and solution tags
  // are cleared by fill kernels inside getrs_launch, the inverted blocks
  // are rewritten, so nothing of an earlier call's contents is read
  const bool timed = h->timer.enabled;
  h->timer.enabled = false;
  const TrsmWs w = trsm_ws(h->scratch, n);
  int st = trsm_invert_launch(h, lu_t, n, d_lu, ldlu, w);
  if (!st) st = getrs_launch(h, lu_t, trans, n, nrhs, d_lu, ldlu, d_b, ldb, w);
  h->timer.enabled = timed;
  RF_CHECK(st);
  int err = 0;
  RF_HIP(hipMemcpyAsync(&err, w.sync + 1, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  RF_HIP(hipStreamSynchronize(h->stream));
  if (err) {
    set_last_error("triangular solve: dependency wait timed out");
    return REMIFA_ERR_HIP;
  }
  return 0;
}

int remifa_residual_f64(remifa_handle_t h, int64_t n, int64_t nrhs, const float* d_a, int64_t lda,
                        const double* d_x, int64_t ldx, const double* d_b, int64_t ldb,
                        double* d_r, int64_t ldr) {
  if (!h) return -1;
  if (n < 0) return -2;
  if (nrhs < 0) return -3;
  if (!d_a && n > 0) return -4;
  if (lda < std::max<int64_t>(n, 1)) return -5;
  if (!d_x && n > 0 && nrhs > 0) return -6;
  if (ldx < std::max<int64_t>(n, 1)) return -7;
  if (!d_b && n > 0 && nrhs > 0) return -8;
  if (ldb < std::max<int64_t>(n, 1)) return -9;
  if (!d_r && n > 0 && nrhs > 0) return -10;
  if (ldr < std::max<int64_t>(n, 1)) return -11;
  if (n == 0 || nrhs == 0) return 0;
  const bool lean = h->ws_user && resid_part_bytes(n, nrhs, false) > h->ws_bytes;
  RF_CHECK(ensure_workspace(h, resid_part_bytes(n, nrhs, lean)));
  return residual_launch(h, n, nrhs, d_a, lda, d_x, ldx, d_b, ldb, d_r, ldr, (double*)h->ws, 0,
                         lean);
}

static int ir_solve_impl(remifa_handle_t h, int trans, int lu_t, int64_t n, int64_t nrhs,
                         const float* d_a, int64_t lda, const void* d_lu, int64_t ldlu,
                         const double* d_b, int64_t ldb, double* d_x, int64_t ldx, double tol,
                         int maxit, int* iters, double* bwd_err, double* history) {
  if (!h) return -1;
  if (lu_t != REMIFA_R_32F && lu_t != REMIFA_R_16F) return -2;
  if (n < 0) return -3;
  if (nrhs < 0) return -4;
  if (!d_a && n > 0) return -5;
  if (lda < std::max<int64_t>(n, 1)) return -6;
  if (!d_lu && n > 0) return -7;
  if (ldlu < std::max<int64_t>(n, 1)) return -8;
  if (!d_b && n > 0 && nrhs > 0) return -9;
  if (ldb < std::max<int64_t>(n, 1)) return -10;
  if (!d_x && n > 0 && nrhs > 0) return -11;
  if (ldx < std::max<int64_t>(n, 1)) return -12;
  if (maxit < 0) return -14;
  if (iters) *iters = -1;
  if (n == 0 || nrhs == 0) {
    if (iters) *iters = 0;
    if (bwd_err) *bwd_err = 0.0;
    return 0;
  }
  // workspace: solve | fp32 correction (n x nrhs) | residual partials |
  // column sums (n) | norms (||r||, ||b||, ||op(A)||, ||x||: 3 nrhs + 1)
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t b_w = al(sizeof(float) * n * nrhs);
  const size_t b_cs = al(sizeof(double) * n);
  const size_t b_nrm = al(sizeof(double) * (3 * nrhs + 2));
  const size_t fixed = b_w + b_cs + b_nrm;
  // (a caller's workspace that has no room for the wider passes takes the
  // narrow ones)
  bool lean = false;
  int ngrp, nset;
  trsm_shape(h, n, nrhs, fixed + al(resid_part_bytes(n, nrhs, false)), &ngrp, &nset);
  if (h->ws_user && al(trsm_ws_bytes(n, ngrp, nset)) + fixed +
                            al(resid_part_bytes(n, nrhs, false)) > h->ws_bytes)
    lean = true;
  const size_t b_sync = al(trsm_ws_bytes(n, ngrp, nset));
  const size_t b_part = al(resid_part_bytes(n, nrhs, lean));
  RF_CHECK(ensure_workspace(h, b_sync + fixed + b_part));
  char* p = (char*)h->ws;
  const TrsmWs tw = trsm_ws(p, n, ngrp, nset);
  float* w = (float*)(p + b_sync);
  double* part = (double*)(p + b_sync + b_w);
  double* cs = (double*)(p + b_sync + b_w + b_part);
  double* nrm = (double*)(p + b_sync + b_w + b_part + b_cs);
  double* const nrm_x = nrm + 2 * nrhs + 1;
  hipStream_t s = h->stream;
  const dim3 gv((unsigned)ceil_div(n, 256), (unsigned)nrhs);

  // ||op(A)||_1 and ||b||_inf per column (fixed for the whole solve): on
  // the handle's second stream (reading A, an HBM-bound pass) while the
  // diagonal blocks are inverted and the first triangular solves run
  // (latency-bound); joined before the first residual. One stream under
  // graph capture.
  hipStreamCaptureStatus cs_st = hipStreamCaptureStatusNone;
  const bool two = hipStreamIsCapturing(s, &cs_st) == hipSuccess &&
                   cs_st == hipStreamCaptureStatusNone && side_stream(h) == 0;
  hipStream_t sn = s;
  if (two) {
    RF_HIP(hipEventRecord(h->ev_main, s));  // inputs ready
    RF_HIP(hipStreamWaitEvent(h->side, h->ev_main, 0));
    sn = h->side;
  }
  if (trans)
    rowsum_kernel<<<(unsigned)ceil_div(n, 64), 1024, 0, sn>>>(n, d_a, lda, cs);
  else
    colsum_kernel<<<(unsigned)n, 256, 0, sn>>>(n, d_a, lda, cs);
  maxreduce_kernel<<<1, 1024, 0, sn>>>(n, cs, nrm + 2 * nrhs);
  colmax_kernel<<<(unsigned)nrhs, 256, 0, sn>>>(n, d_b, ldb, nrm + nrhs);
  RF_HIP(hipGetLastError());
  if (two) RF_HIP(hipEventRecord(h->ev_side, sn));
  // x0 = op(LU)^-1 b in fp32
  d2f_kernel<<<gv, 256, 0, s>>>(n, (int)nrhs, d_b, ldb, w, n);
  const int st0 = trsm_invert_launch(h, lu_t, n, d_lu, ldlu, tw);
  const int st1 = st0 ? st0
                      : getrs_launch(h, lu_t, trans, n, nrhs, d_lu, ldlu, w, n, tw, nrm,
                                     (int)nrhs, nrm_x, (int)nrhs);
  // (joined also when a launch failed: the workspace may be reused next)
  if (two) RF_HIP(hipStreamWaitEvent(s, h->ev_side, 0));
  RF_CHECK(st1);
  axpy_f2d_kernel<<<gv, 256, 0, s>>>(n, w, n, d_x, ldx, 1, nrm_x);
  RF_HIP(hipGetLastError());

  std::vector<double> hn(3 * nrhs + 1);
  int it = 0, done = -1;
  double worst = 0.0;
  for (;; ++it) {
    // w = fp32(b - op(A) x), ||r||_inf (||x||_inf came with the update of x)
    RF_CHECK(residual_launch(h, n, nrhs, d_a, lda, d_x, ldx, d_b, ldb, nullptr, 0, part, trans,
                             lean, w, nrm));
    RF_HIP(hipMemcpyAsync(hn.data(), nrm, sizeof(double) * hn.size(), hipMemcpyDeviceToHost, s));
    int serr = 0;
    RF_HIP(hipMemcpyAsync(&serr, tw.sync + 1, sizeof(int), hipMemcpyDeviceToHost, s));
    RF_HIP(hipStreamSynchronize(s));
    if (serr) {
      set_last_error("triangular solve: dependency wait timed out");
      return REMIFA_ERR_HIP;
    }
    // tests/errors.hxx:237: ||r||_inf / (||A||_1 ||x||_inf + ||b||_inf)
    worst = 0.0;
    const double anorm = hn[2 * nrhs];
    for (int64_t k = 0; k < nrhs; ++k) {
      double e = hn[k] / (anorm * hn[2 * nrhs + 1 + k] + hn[nrhs + k]);
      if (e != e) {
        worst = e;
        break;
      }
      worst = std::max(worst, e);
    }
    if (history) history[it] = worst;
    if (worst <= tol) {
      done = it;
      break;
    }
    if (it >= maxit || worst != worst) break;
    RF_CHECK(getrs_launch(h, lu_t, trans, n, nrhs, d_lu, ldlu, w, n, tw, nrm, (int)nrhs, nrm_x,
                          (int)nrhs));
    axpy_f2d_kernel<<<gv, 256, 0, s>>>(n, w, n, d_x, ldx, 0, nrm_x);
    RF_HIP(hipGetLastError());
  }
  if (iters) *iters = done;
  if (bwd_err) *bwd_err = worst;
  return 0;
}

int remifa_ir_solve(remifa_handle_t h, int lu_t, int64_t n, int64_t nrhs, const float* d_a,
                    int64_t lda, const void* d_lu, int64_t ldlu, const double* d_b, int64_t ldb,
                    double* d_x, int64_t ldx, double tol, int maxit, int* iters, double* bwd_err,
                    double* history) {
  return ir_solve_impl(h, 0, lu_t, n, nrhs, d_a, lda, d_lu, ldlu, d_b, ldb, d_x, ldx, tol, maxit,
                       iters, bwd_err, history);
}

int remifa_ir_solve_trans(remifa_handle_t h, int lu_t, int64_t n, int64_t nrhs, const float* d_a,
                          int64_t lda, const void* d_lu, int64_t ldlu, const double* d_b,
                          int64_t ldb, double* d_x, int64_t ldx, double tol, int maxit,
                          int* iters, double* bwd_err, double* history) {
  return ir_solve_impl(h, 1, lu_t, n, nrhs, d_a, lda, d_lu, ldlu, d_b, ldb, d_x, ldx, tol, maxit,
                       iters, bwd_err, history);
}

}  // extern "C"
