// Inner factorization of one outer block, one launch per slice of up to 64
// columns: the reference's ib loop (src/lu_nopiv_inner_ll.hxx:197-370,
// src/lu_nopiv_inner_rl.hxx:104-196) for an sw-wide slice.
//
// Input: the sw-wide block column l[0:cm, 0:sw] (its top sw x sw tile is the
// diagonal tile), the sw-tall block row u[0:sw, sw:cm] and the operand copies
// lop / uop of the outer block's earlier slices. Output: the slice's factors
// in place (and their fp16 mirror), its operand copies for the next slices.
//
// What bounds it is the chain of 64 dependent pivots per slice, and, between
// slices, memory round trips and launches; the arithmetic is small. Hence one
// launch per slice in which every workgroup factors the tile itself (as every
// thread block of the reference's panel kernel does, src/lu_nopiv.cu:123-170)
// instead of a tile kernel, a kernel for the rows and columns and two update
// GEMMs that pass their results through memory. Six wavefronts:
//  * waves 2-5 first form the tile minus the earlier slices' products (one
//    32 x 32 quadrant each, MFMA) in LDS;
//  * wave 0 (lane = row) and wave 1 (lane = column) then factor the tile in
//    8-wide panels: wave 0 the panel's columns of L, wave 1 its rows of U.
//    Both hold the panel's 8 x 8 diagonal block and run its pivots (readlane)
//    redundantly, with the same bits, so they meet once per panel only: each
//    publishes its panel (operand-rounded) in LDS, and takes the other's as
//    the MFMA operand of the sums that the later panels need;
//  * waves 2-5 meanwhile form their own vectors (rows of L below the tile,
//    columns of U right of it; 64 per unit, 32 with fp32 operands) minus the
//    earlier slices' products, and solve them against the tile in the same
//    8-wide panels, each as soon as it is published.
// The tile is read by every workgroup, so it is not written in place: it goes
// to a slot, and the next slice's launch (or the final one) copies it to the
// matrix, which nothing else reads there meanwhile.
//
// The arithmetic follows the reference's ib-granular semantics:
//  * within an ib block (the panel kernel, src/lu_nopiv.cu:123-170):
//    reciprocal of the pivot, multiply, fused multiply-subtract, in the
//    factor precision (fp32, or fp16 with one rounding per operation), each
//    entry receiving its updates in pivot order;
//  * across ib blocks (the inner GEMMs): products of operands rounded to the
//    update type, summed from zero (fp32 on the matrix cores, or fp16 in k
//    order for FP16 / TC16) and subtracted, left-looking (one sum over
//    everything to the left) or right-looking (one sum, rounded to the panel
//    precision, per ib block, and per slice for the earlier slices).
#pragma once
#include "slice_common.hpp"

namespace remifa {

struct SliceArgs {
  int64_t cm;       // rows of the slice's block column (columns of its block row)
  int sw, so;       // slice width; its offset in the outer block
  int pre;          // subtract the earlier slices' products here (so > 0)
  int chunk;        // right-looking: width of the earlier slices
  void* l;
  int64_t ldl;
  void* u;
  int64_t ldu;
  int vec;          // columns of u (and of cp) start on 16 bytes
  int store_x;      // write the factors to l / u (else only to the mirror)
  half_t* cp;       // fp16 mirror at the tile's corner (null: none)
  int64_t ldcp;
  void* lop;        // operand copies: row r of L / column c of U of the outer
  void* uop;        // block at r * ldop, k-contiguous
  int64_t ldop;
  int write_op;     // a later slice of the outer block reads them
  int nul, nunits;  // units of rows of L; all units
  float* slot;      // this slice's tile
  const float* prev;  // the slice before's (null: none pending)
  void* pa;         // ... and where it goes
  half_t* pcp;
  int64_t lda, ldpcp;
  int psw;
  int w_half;       // the matrix is fp16 (else fp32)
  int64_t col;      // column of the tile in the matrix (for the pivot check)
};

namespace {

constexpr int UW = 4;               // unit wavefronts
constexpr int SLT = 64 * (2 + UW);  // threads of a workgroup
constexpr int SLOT_HDR = 64;        // floats before a slot's tile (header)

typedef float sf16 __attribute__((ext_vector_type(16)));
typedef _Float16 sh2 __attribute__((ext_vector_type(2)));
typedef _Float16 sh4 __attribute__((ext_vector_type(4)));
typedef _Float16 sh8 __attribute__((ext_vector_type(8)));
typedef short ss4 __attribute__((ext_vector_type(4)));
typedef __bf16 sb8 __attribute__((ext_vector_type(8)));
typedef uint16_t su8 __attribute__((ext_vector_type(8)));
typedef unsigned su2 __attribute__((ext_vector_type(2)));

template <int MODE>
struct SlTypes {
  using X = typename std::conditional<(MODE <= SM_F32_TC), float, half_t>::type;
  using O = typename std::conditional<(MODE == SM_F32), float, uint16_t>::type;
  static constexpr int VG = MODE == SM_F32 ? 1 : 2;  // 32-vector groups of a unit
  // operands go through the matrix cores (else fp16 fma chains)
  static constexpr bool MM = MODE != SM_F16_H;
};

constexpr int XP = SW + 1;  // row pitch of the fp32 tile (lanes on rows: no conflicts)
constexpr int OP = SW + 4;  // operand row pitch: 136-byte (272-byte) rows, conflict-free

template <int MODE>
struct SlLds {
  using X = typename SlTypes<MODE>::X;
  using O = typename SlTypes<MODE>::O;
  float ts[2][SW][XP];  // the updated tile: [0][row][column], [1][column][row]
  float vt[UW][32 * SlTypes<MODE>::VG][XP];   // a unit's vectors [vector][entry]
  __attribute__((aligned(16))) O uo[SW][OP];  // op(U) [column][k]
  __attribute__((aligned(16))) O lo[SW][OP];  // op(L) [row][k]
  __attribute__((aligned(16))) X uf[SW][SW];  // U [k][column]
  __attribute__((aligned(16))) X lf[SW][SW];  // L [k][row]
  __attribute__((aligned(16))) X rk[2][SW];   // reciprocals of the pivots, ones
  int flag[2];  // panels whose operand rows each tile wave has published
  int done[2];  // ... and whose values
};

template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// typed panel arithmetic (the same operations as Sem's, on the stored type)
__device__ __forceinline__ float p_rcp(float x) { return 1.0f / x; }
__device__ __forceinline__ half_t p_rcp(half_t x) { return (half_t)(1.0f / (float)x); }
// The same value wherever rcp_ok(x) holds: one Newton step on the
// hardware estimate with a fused residual is the correctly rounded reciprocal
// of a normal number whose reciprocal is normal (compared with 1.0f / x for
// every float), three dependent instructions instead of eleven on the
// pivots' chain.
__device__ __forceinline__ float p_rcp_fast(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ half_t p_rcp_fast(half_t x) { return (half_t)p_rcp_fast((float)x); }
// (zeros, denormals, huge values, infinities and NaN fail)
__device__ __forceinline__ bool rcp_ok(float x) {
  return ((__builtin_bit_cast(unsigned, x) >> 23) & 0xffu) - 2u <= 250u;
}
__device__ __forceinline__ float p_fnma(float a, float b, float c) {
  return __builtin_fmaf(-a, b, c);
}
__device__ __forceinline__ half_t p_fnma(half_t a, half_t b, half_t c) {
  return __builtin_fmaf16(-a, b, c);
}
__device__ __forceinline__ float p_bcast(float v, int lane) { return bcast_lane(v, lane); }
__device__ __forceinline__ half_t p_bcast(half_t v, int lane) {
  const int b = __builtin_bit_cast(uint16_t, v);
  return __builtin_bit_cast(half_t, (uint16_t)__builtin_amdgcn_readlane(b, lane));
}

// eight consecutive panel values (16-byte aligned)
__device__ __forceinline__ void ld8(const float* p, float (&v)[8]) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
  v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
__device__ __forceinline__ void ld8(const half_t* p, half_t (&v)[8]) {
  const sh8 a = *(const sh8*)p;
#pragma unroll
  for (int c = 0; c < 8; ++c) v[c] = a[c];
}

struct Pair {
  unsigned a, b;
};
// a: low half lanes of v0 | low half lanes of v1 moved up; b: high half lanes
// of v0 moved down | high half lanes of v1
__device__ __forceinline__ Pair swap32(unsigned v0, unsigned v1) {
  const auto r = __builtin_amdgcn_permlane32_swap(v0, v1, false, false);
  return {r[0], r[1]};
}
__device__ __forceinline__ unsigned fbits(float f) { return __builtin_bit_cast(unsigned, f); }
__device__ __forceinline__ float bitsf(unsigned u) { return __builtin_bit_cast(float, u); }

template <int MODE>
__device__ __forceinline__ uint16_t op16(float v) {
  if constexpr (MODE == SM_F16_BF)
    return f32_to_bf16_bits(v);
  else
    return __builtin_bit_cast(uint16_t, (half_t)v);
}
template <int MODE>
__device__ __forceinline__ unsigned op_pack(float a, float b) {
  return (unsigned)op16<MODE>(a) | ((unsigned)op16<MODE>(b) << 16);
}

// D += A B over 8 k-values: D[m][n], lane (n, h) holds rows m = 8 (q / 4) +
// 4 h + q % 4; operands: lane (r, h) holds k = 4 h .. 4 h + 3 of row r
template <int MODE>
__device__ __forceinline__ sf16 mma8(su2 a, su2 b, sf16 c) {
  if constexpr (MODE == SM_F16_BF)
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(ss4, a),
                                                    __builtin_bit_cast(ss4, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(sh4, a),
                                                __builtin_bit_cast(sh4, b), c, 0, 0, 0);
}
// ... over 16 k-values, lane (r, h) holding k = 8 h .. 8 h + 7
template <int MODE>
__device__ __forceinline__ sf16 mma16(su8 a, su8 b, sf16 c) {
  if constexpr (MODE == SM_F16_BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sb8, a),
                                                   __builtin_bit_cast(sb8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(sh8, a),
                                                  __builtin_bit_cast(sh8, b), c, 0, 0, 0);
}

// acc[m][n] += sum over K (a multiple of 8) of rows am[m] (A) and bn[n] (B)
// of the operand copies; am / bn point at this lane's rows (lane % 32), at
// the first k of the range. The rows come straight from memory (L2) into
// fragments: a ring of D steps in flight, since a step's matrix work (32 to
// 128 cycles) is far below the latency of its loads.
template <int MODE, int D, int NM, int NN>
__device__ __forceinline__ void op_sum(sf16 (&acc)[NM][NN],
                                       const typename SlTypes<MODE>::O* const (&am)[NM],
                                       const typename SlTypes<MODE>::O* const (&bn)[NN], int K,
                                       int lh) {
  constexpr bool F = MODE == SM_F32;
  constexpr int ST = F ? 8 : 16;  // k-values of a step
  using V = typename std::conditional<F, float4, su8>::type;
  auto mma = [&](const V(&a)[NM], const V(&b)[NN]) {
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
      for (int j = 0; j < NN; ++j) {
        if constexpr (F) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].x, b[j].x, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].y, b[j].y, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].z, b[j].z, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].w, b[j].w, acc[i][j], 0, 0, 0);
        } else {
          acc[i][j] = mma16<MODE>(a[i], b[j], acc[i][j]);
        }
      }
  };
  const int lo = (ST / 2) * lh;
  auto load = [&](int k, V(&a)[NM], V(&b)[NN]) {
#pragma unroll
    for (int i = 0; i < NM; ++i) a[i] = *(const V*)(am[i] + k + lo);
#pragma unroll
    for (int j = 0; j < NN; ++j) b[j] = *(const V*)(bn[j] + k + lo);
  };
  int k = 0;
  if constexpr (D == 16) {
    // up to D steps' loads at once (addresses past the range repeat its last)
#pragma unroll 1
    for (; k + ST <= K; k += ST * D) {
      const int n = (K - k) / ST < D ? (K - k) / ST : D;
      V a[D][NM], b[D][NN];
#pragma unroll
      for (int s = 0; s < D; ++s) load(k + ST * (s < n ? s : n - 1), a[s], b[s]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < D; ++s) {
        if (s < n) mma(a[s], b[s]);
      }
    }
    k = K / ST * ST;
  } else {
    const int km = K / (ST * D) * (ST * D);
    if (km > 0) {
      V a[D][NM], b[D][NN];
#pragma unroll
      for (int s = 0; s < D; ++s) load(ST * s, a[s], b[s]);
#pragma unroll 1
      for (; k < km; k += ST * D) {
        const int kn = k + ST * D < km ? k + ST * D : k;  // (the last round reloads its own)
#pragma unroll
        for (int s = 0; s < D; ++s) {
          mma(a[s], b[s]);
          load(kn + ST * s, a[s], b[s]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
#pragma unroll 1
  for (; k + ST <= K; k += ST) {
    V a[NM], b[NN];
    load(k, a, b);
    mma(a, b);
  }
  if constexpr (!F) {
    if (k < K) {
      su2 a[NM], b[NN];
#pragma unroll
      for (int i = 0; i < NM; ++i) a[i] = *(const su2*)(am[i] + k + 4 * lh);
#pragma unroll
      for (int j = 0; j < NN; ++j) b[j] = *(const su2*)(bn[j] + k + 4 * lh);
#pragma unroll
      for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NN; ++j) acc[i][j] = mma8<MODE>(a[i], b[j], acc[i][j]);
    }
  }
}

template <int NM, int NN>
__device__ __forceinline__ void acc_zero(sf16 (&acc)[NM][NN]) {
#pragma unroll
  for (int i = 0; i < NM; ++i)
#pragma unroll
    for (int j = 0; j < NN; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;
}

// The cross-block sums of one wavefront's vectors (vector = lane). ROLE 0: a
// unit; 1: the tile's own vectors (of the first 32 only the first 32 entries
// are wanted). The panel loop is a real loop (unrolled it is 60-170 KB of
// code that runs once per launch, and fetching that took longer than running
// it), so the sums slide: register group i always holds the panel i after the
// current one. On the matrix cores they live as 32 x 32 quadrants acc[w][rg]
// (entries 8 P + 32 w .., vectors 32 rg ..; panel P the next one);
// vector-per-lane values come from them with v_permlane32_swap.
template <int MODE, int ROLE>
struct Cross {
  using Ty = SlTypes<MODE>;
  using O = typename Ty::O;
  using X = typename Ty::X;
  static constexpr int NR = ROLE == 1 ? 2 : Ty::VG;
  sf16 acc[Ty::MM ? 2 : 1][Ty::MM ? NR : 1];
  sh2 ah[Ty::MM ? 1 : SW / 2];

  __device__ __forceinline__ void zero() {
    if constexpr (Ty::MM) {
      acc_zero(acc);
    } else {
#pragma unroll
      for (int c = 0; c < SW / 2; ++c) ah[c] = (sh2){(_Float16)0, (_Float16)0};
    }
  }
  // this lane's sums of the panel I after the one the window starts at
  template <int I>
  __device__ __forceinline__ void get(float (&a)[8]) const {
    if constexpr (Ty::MM) {
      constexpr int w = I / 4, q0 = 4 * (I % 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float v0 = (ROLE == 1 && w == 1) ? 0.0f : acc[w][0][q0 + q];
        const float v1 = NR == 2 ? acc[w][NR - 1][q0 + q] : v0;
        const Pair r = swap32(fbits(v0), fbits(v1));
        a[q] = bitsf(r.a);
        a[4 + q] = bitsf(r.b);
      }
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) a[c] = (float)ah[4 * I + c / 2][c % 2];
    }
  }
  // the window moves on by one panel
  __device__ __forceinline__ void slide(int g) {
    if constexpr (Ty::MM) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
#pragma unroll
        for (int q = 0; q < 12; ++q) acc[0][r][q] = acc[0][r][q + 4];
        if ((ROLE == 1 && r == 0) || g > 3) continue;  // (nothing further right)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[0][r][12 + q] = acc[1][r][q];
#pragma unroll
        for (int q = 0; q < 12; ++q) acc[1][r][q] = acc[1][r][q + 4];
      }
    } else {
#pragma unroll
      for (int c = 0; c < SW / 2 - 4; ++c) ah[c] = ah[c + 4];
    }
  }
  // add the products of the finished panel g (p: its entries of this lane's
  // vector) to the panels after it: tab = the other factor's operand rows
  // [entry][k], mf its values [k][entry] (the rows past the tile wrap around;
  // their sums are not used)
  __device__ __forceinline__ void add(const X (&p)[8], const O (*tab)[OP], const X (*mf)[SW],
                                      int g, int l32, int lh) {
    const int e0 = 8 * (g + 1);
    if constexpr (!Ty::MM) {
#pragma unroll
      for (int i = 0; i < 7; ++i) {
        if (g + 1 + i < 8) {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const sh2 xk = {(_Float16)p[k], (_Float16)p[k]};
            const sh8 m = *(const sh8*)&mf[8 * g + k][e0 + 8 * i];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              ah[4 * i + e] = __builtin_elementwise_fma(xk, (sh2){m[2 * e], m[2 * e + 1]},
                                                        ah[4 * i + e]);
          }
        }
      }
    } else {
      const int k0 = 8 * g + 4 * lh;
      const int r0 = (e0 + l32) & (SW - 1), r1 = (e0 + 32 + l32) & (SW - 1);
      if constexpr (MODE == SM_F32) {
        float b[NR][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const Pair r = swap32(fbits(p[j]), fbits(p[4 + j]));
          b[0][j] = bitsf(r.a);
          if constexpr (NR == 2) b[1][j] = bitsf(r.b);
        }
        auto quad = [&](int w, int rg, const float4& a) {
          acc[w][rg] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b[rg][0], acc[w][rg], 0, 0, 0);
          acc[w][rg] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b[rg][1], acc[w][rg], 0, 0, 0);
          acc[w][rg] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b[rg][2], acc[w][rg], 0, 0, 0);
          acc[w][rg] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b[rg][3], acc[w][rg], 0, 0, 0);
        };
        const float4 a0 = *(const float4*)&tab[r0][k0];
        const float4 a1 = *(const float4*)&tab[r1][k0];
        quad(0, NR - 1, a0);
        if (NR == 2 && (ROLE == 0 || g < 3)) quad(0, 0, a0);
        if (g < 3) {
          quad(1, NR - 1, a1);
          if (ROLE == 0 && NR == 2) quad(1, 0, a1);
        }
      } else {
        const su2 lo2 = {op_pack<MODE>((float)p[0], (float)p[1]),
                         op_pack<MODE>((float)p[2], (float)p[3])};
        const su2 hi2 = {op_pack<MODE>((float)p[4], (float)p[5]),
                         op_pack<MODE>((float)p[6], (float)p[7])};
        const Pair s0 = swap32(lo2[0], hi2[0]), s1 = swap32(lo2[1], hi2[1]);
        const su2 b0 = {s0.a, s1.a}, b1 = {s0.b, s1.b};
        const su2 a0 = *(const su2*)&tab[r0][k0];
        const su2 a1 = *(const su2*)&tab[r1][k0];
        acc[0][1] = mma8<MODE>(a0, b1, acc[0][1]);
        if (ROLE == 0 || g < 3) acc[0][0] = mma8<MODE>(a0, b0, acc[0][0]);
        if (g < 3) {
          acc[1][1] = mma8<MODE>(a1, b1, acc[1][1]);
          if constexpr (ROLE == 0) acc[1][0] = mma8<MODE>(a1, b0, acc[1][0]);
        }
      }
    }
  }
};

// Panel g of this lane's vector xl (LDS) into p, after the cross-block sums.
// Left-looking: at the start of an ib block the sums of the finished blocks
// come off its panels; right-looking: the sums of the block that just ended
// come off everything after it.
template <int MODE, bool RL, int IB, int ROLE>
__device__ __forceinline__ void panel_start(Cross<MODE, ROLE>& cr, float* xl, int g,
                                            typename SlTypes<MODE>::X (&p)[8]) {
  using X = typename SlTypes<MODE>::X;
  constexpr int PB = IB / 8;
  constexpr bool HALF = MODE >= SM_F16_TC;
  float x[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) x[c] = xl[8 * g + c];
  if (g % PB == 0) {
    if (g == 0) {
      cr.zero();
      // (left-looking: the entries minus the earlier slices' products are
      // not rounded to fp16 so far)
      if constexpr (HALF && !RL) {
#pragma unroll
        for (int c = 0; c < 8; ++c) x[c] = r16(x[c]);
#pragma unroll
        for (int c = 8; c < IB; ++c) xl[c] = r16(xl[c]);
      }
    } else {
      float a[8];
      cr.template get<0>(a);
#pragma unroll
      for (int c = 0; c < 8; ++c) x[c] = Sem<MODE>::apply(x[c], a[c]);
      constexpr int NP = RL ? 8 : PB;  // panels it reaches
      static_for<NP - 1>([&](auto ii) {
        constexpr int i = decltype(ii)::value + 1;
        if (!RL || g + i < 8) {
          cr.template get<i>(a);
          float* const y = xl + 8 * (g + i);
#pragma unroll
          for (int c = 0; c < 8; ++c) y[c] = Sem<MODE>::apply(y[c], a[c]);
        }
      });
      if constexpr (RL) cr.zero();
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) p[c] = (X)x[c];
}

// The eight pivots k0 .. k0 + 7 of a panel (8 entries p of this lane's row,
// or with COL column); rr: the reciprocals. Nothing is masked: wave 0 keeps
// the multipliers only (the lanes at or above a pivot's row compute values
// nobody reads), and wave 1 the rows of U (lanes left of the pivot's column
// likewise); a pivot reads lane k alone.
template <bool FAST, bool COL, typename X>
__device__ __forceinline__ void panel_pivots(X (&p)[8], X (&rr)[8], int k0) {
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) {
    X v[8];
#pragma unroll
    for (int c = kk; c < 8; ++c) v[c] = p_bcast(p[c], k0 + kk);
    const X r = FAST ? p_rcp_fast(v[kk]) : p_rcp(v[kk]);
    rr[kk] = r;
    if constexpr (!COL) {
      // multipliers of the rows below, then their later columns
      p[kk] = p[kk] * r;
#pragma unroll
      for (int c = kk + 1; c < 8; ++c) p[c] = p_fnma(p[kk], v[c], p[c]);
    } else {
      // the multipliers are column k's entries (lane k) times r
#pragma unroll
      for (int c = kk + 1; c < 8; ++c) p[c] = p_fnma((X)(v[c] * r), p[kk], p[c]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// false if some pivot of the panel is outside p_rcp_fast's range: wave 1's
// lane k0 + kk still holds pivot kk as its entry kk; in wave 0 that entry is
// pivot times reciprocal (1 up to rounding; 0, infinite or NaN outside)
template <bool COL, typename X>
__device__ __forceinline__ bool pivots_ok(const X (&p)[8], int g, int lane) {
  const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4;
  const X q0 = b0 ? p[1] : p[0], q1 = b0 ? p[3] : p[2], q2 = b0 ? p[5] : p[4],
          q3 = b0 ? p[7] : p[6];
  const X h0 = b1 ? q1 : q0, h1 = b1 ? q3 : q2;
  const float f = (float)(b2 ? h1 : h0);  // entry lane % 8
  const bool ok = COL ? rcp_ok(f) : (f > 0.5f && f < 2.0f);
  return __ballot(!ok && (lane >> 3) == g) == 0;
}

// a finished panel's values [k][lane] and reciprocals, for the units
template <bool COL, int MODE, typename X>
__device__ __forceinline__ void put_values(SlLds<MODE>& S, const X (&p)[8], const X (&rr)[8],
                                           int p0, int lane) {
  auto& F = COL ? S.uf : S.lf;
#pragma unroll
  for (int c = 0; c < 8; ++c) F[p0 + c][lane] = p[c];
  if constexpr (!COL) {
    if (lane == 0) {
#pragma unroll
      for (int c = 0; c < 8; ++c) S.rk[0][p0 + c] = rr[c];
    }
  }
}

// wait until the tile waves have published panel g (they always get there:
// they wait for each other's previous panel only)
__device__ __forceinline__ void wait_flag(const int& flag, int g) {
  while (__hip_atomic_load(&flag, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) <= g) {
  }
}

// The tile's factorization by waves 0 (COL = false: lane = row, entries =
// columns) and 1 (COL = true: lane = column, entries = rows).
template <int MODE, bool RL, int IB, bool COL>
__device__ __forceinline__ void tile_wave(SlLds<MODE>& S, int lane) {
  using Ty = SlTypes<MODE>;
  using X = typename Ty::X;
  using O = typename Ty::O;
  const int l32 = lane & 31, lh = lane >> 5;
  float* const xl = S.ts[COL][lane];
  __builtin_amdgcn_s_setprio(3);  // the slice waits for this chain
  Cross<MODE, 1> cr;
#pragma unroll 1
  for (int g = 0; g < 8; ++g) {
    const int p0 = 8 * g, kend = (p0 / IB + 1) * IB;
    X p[8], rr[8];
    panel_start<MODE, RL, IB, 1>(cr, xl, g, p);
    if constexpr (IB < SW) cr.slide(g);
    {
      X s[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) s[c] = p[c];
      panel_pivots<true, COL>(p, rr, p0);
      if (!pivots_ok<COL>(p, g, lane)) {  // (wave-uniform)
#pragma unroll
        for (int c = 0; c < 8; ++c) p[c] = s[c];
        panel_pivots<false, COL>(p, rr, p0);
      }
    }
    // the later panels of the ib block, pivot by pivot
    if constexpr (IB > 8) {
#pragma unroll 1
      for (int c0 = p0 + 8; c0 < kend; c0 += 8) {
        X y[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) y[c] = (X)xl[c0 + c];
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          const int k = p0 + kk;
          X w[8];
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            w[c] = p_bcast(y[c], k);
            if constexpr (COL) w[c] = w[c] * rr[kk];
          }
#pragma unroll
          for (int c = 0; c < 8; ++c)
            y[c] = COL ? p_fnma(w[c], p[kk], y[c]) : p_fnma(p[kk], w[c], y[c]);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) xl[c0 + c] = (float)y[c];
      }
    }
    // publish: operand rows [lane][k] for the other tile wave's sums (and the
    // units'), values [k][lane] and reciprocals for the units
    if (IB < SW && kend < SW) {
      if constexpr (Ty::MM) {
        O* const o = COL ? &S.uo[lane][p0] : &S.lo[lane][p0];
        if constexpr (MODE == SM_F32) {
          *(float4*)o = make_float4(p[0], p[1], p[2], p[3]);
          *(float4*)(o + 4) = make_float4(p[4], p[5], p[6], p[7]);
        } else {
          *(su2*)o = (su2){op_pack<MODE>((float)p[0], (float)p[1]),
                           op_pack<MODE>((float)p[2], (float)p[3])};
          *(su2*)(o + 4) = (su2){op_pack<MODE>((float)p[4], (float)p[5]),
                                 op_pack<MODE>((float)p[6], (float)p[7])};
        }
      } else {
        put_values<COL>(S, p, rr, p0, lane);
      }
      __hip_atomic_store(&S.flag[COL], g + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      wait_flag(S.flag[!COL], g);
      cr.add(p, COL ? S.lo : S.uo, COL ? S.lf : S.uf, g, l32, lh);
      if constexpr (Ty::MM) put_values<COL>(S, p, rr, p0, lane);  // (while the matrix cores work)
    } else {
      put_values<COL>(S, p, rr, p0, lane);
    }
    __hip_atomic_store(&S.done[COL], g + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __builtin_amdgcn_s_setprio(0);
}

// Solve one vector per lane (xl, in LDS) against the tile, panel by panel as
// the tile waves publish it: rows of L
// (tab = op(U) [column][k], mf = U [k][column], pivots scaled by rk) or
// columns of U (tab = op(L), mf = L, not scaled).
// put(p0, p): called with each finished panel.
template <int MODE, bool RL, int IB, typename F>
__device__ __forceinline__ void unit_solve(const SlLds<MODE>& S, float* xl, bool is_l, int lane,
                                           F&& put) {
  using Ty = SlTypes<MODE>;
  using X = typename Ty::X;
  const int l32 = lane & 31, lh = lane >> 5;
  const auto* const tab = is_l ? S.uo : S.lo;
  const X(*const mf)[SW] = is_l ? S.uf : S.lf;
  const X* const rk = S.rk[!is_l];
  Cross<MODE, 0> cr;
#pragma unroll 1
  for (int g = 0; g < 8; ++g) {
    const int p0 = 8 * g, kend = (p0 / IB + 1) * IB;
    X p[8];
    while (true) {
      const int a = __hip_atomic_load(&S.done[0], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
      const int b = __hip_atomic_load(&S.done[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (a > g && b > g) break;  // (see wait_flag)
      __builtin_amdgcn_s_sleep(1);
    }
    X rv[8];
    ld8(rk + p0, rv);
    panel_start<MODE, RL, IB, 0>(cr, xl, g, p);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const X lk = p[kk] * rv[kk];
      p[kk] = lk;
      X m[8];
      ld8(&mf[p0 + kk][p0], m);
#pragma unroll
      for (int c = kk + 1; c < 8; ++c) p[c] = p_fnma(lk, m[c], p[c]);
    }
    if constexpr (IB > 8) {
#pragma unroll 1
      for (int c0 = p0 + 8; c0 < kend; c0 += 8) {
        X y[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) y[c] = (X)xl[c0 + c];
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          X m[8];
          ld8(&mf[p0 + kk][c0], m);
#pragma unroll
          for (int c = 0; c < 8; ++c) y[c] = p_fnma(p[kk], m[c], y[c]);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) xl[c0 + c] = (float)y[c];
      }
    }
    if (IB < SW && kend < SW) {
      cr.slide(g);
      cr.add(p, tab, mf, g, l32, lh);
    }
    put(p0, p);
  }
}

// wave-private exchange through LDS: earlier writes of the wavefront's lanes
// are read by its other lanes
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// T: type of the factored buffers (float for the half-footprint layout's,
// whose matrix is fp16: g.w_half)
template <typename T, int MODE, bool RL, int IB>
__global__ void __launch_bounds__(SLT) slice_kernel(SliceArgs g) {
  using Ty = SlTypes<MODE>;
  using O = typename Ty::O;
  using X = typename Ty::X;
  constexpr int VG = Ty::VG, VPU = 32 * VG;
  __shared__ SlLds<MODE> S;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  T* const l = (T*)g.l;
  T* const u = (T*)g.u;
  const int sw = g.sw, so = g.so;
  const O* const lop = (const O*)g.lop;
  const O* const uop = (const O*)g.uop;

  if (threadIdx.x < 2) S.flag[threadIdx.x] = S.done[threadIdx.x] = 0;
  if (wave == 1) S.rk[1][lane] = (typename Ty::X)1.0f;

  // ---- the tile minus the earlier slices' products, one quadrant per unit
  // wave: lane (n, h) holds rows 32 rg + n, columns 32 cg + 8 (q / 4) + 4 h
  // + q % 4
  if (wave >= 2) {
    const int qd = wave - 2, rg = qd & 1, cg = qd >> 1;
    const int row = 32 * rg + l32;
    float cv[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int col = 32 * cg + 8 * (q >> 2) + 4 * lh + (q & 3);
      cv[q] = (float)l[(row < sw ? row : sw - 1) + (int64_t)(col < sw ? col : sw - 1) * g.ldl];
    }
    if constexpr (Ty::MM) {
      if (g.pre) {
        const O* const am[1] = {uop + (so + 32 * cg + l32) * g.ldop};
        const O* const bn[1] = {lop + (so + row) * g.ldop};
        const int step = RL ? g.chunk : so;
        for (int k0 = 0; k0 < so; k0 += step) {
          sf16 acc[1][1];
          acc_zero(acc);
          const O* const a0[1] = {am[0] + k0};
          const O* const b0[1] = {bn[0] + k0};
          op_sum<MODE, 16, 1, 1>(acc, a0, b0, step, lh);
#pragma unroll
          for (int q = 0; q < 16; ++q) {
            cv[q] -= acc[0][0][q];
            if constexpr (RL && MODE >= SM_F16_TC) cv[q] = r16(cv[q]);
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int col = 32 * cg + 8 * (q >> 2) + 4 * lh + (q & 3);
      const float v = (row < sw && col < sw) ? cv[q] : (row == col ? 1.0f : 0.0f);
      S.ts[0][row][col] = v;
      S.ts[1][col][row] = v;
    }
  }
  __syncthreads();

  if (wave < 2) {
    if (wave == 0)
      tile_wave<MODE, RL, IB, false>(S, lane);
    else
      tile_wave<MODE, RL, IB, true>(S, lane);
    wait_flag(S.done[wave ^ 1], 7);
    // this slice's tile to its slot, the one before to the matrix
    if (blockIdx.x == 0) {
#pragma unroll 8
      for (int c = wave; c < SW; c += 2)
        g.slot[SLOT_HDR + c * SW + lane] =
            (float)(lane > c ? S.lf[c][lane] : S.uf[lane][c]);
      if (wave == 0) {
        // first zero or non-finite pivot as stored, 1-based, 0 if none
        const float v = (float)S.uf[lane][lane];
        const float d = g.w_half ? r16(v) : v;
        const unsigned long long bad =
            __ballot(lane < sw && (d == 0.0f || !__builtin_isfinite(d)));
        if (lane == 0) {
          const int before = g.prev ? ((const int*)g.prev)[0] : 0;
          ((int*)g.slot)[0] =
              before ? before : (bad ? (int)(g.col + __builtin_ctzll(bad) + 1) : 0);
        }
      }
    }
    if (g.prev && blockIdx.x == gridDim.x - 1) {
#pragma unroll 8
      for (int c = wave; c < g.psw; c += 2) {
        const float v = g.prev[SLOT_HDR + c * SW + lane];
        if (lane < g.psw) {
          if (g.w_half)
            ((half_t*)g.pa)[lane + c * g.lda] = (half_t)v;
          else
            ((float*)g.pa)[lane + c * g.lda] = v;
          if (g.pcp) g.pcp[lane + c * g.ldpcp] = (half_t)v;
        }
      }
    }
    return;
  }

  // ---- units (the first of each wave while the tile is factored)
  float(*const vt)[XP] = S.vt[wave - 2];
  const int vl = VG == 2 ? lane : l32;  // this lane's vector of the unit
  float* const xl = vt[vl];
#pragma unroll 1
  for (int un = blockIdx.x + gridDim.x * (wave - 2); un < g.nunits; un += gridDim.x * UW) {
    const bool is_l = un < g.nul;
    const int64_t v0 = sw + (int64_t)(is_l ? un : un - g.nul) * VPU;  // first vector
    const int64_t cl = g.cm - 1;
    // rows of L are read across the rows (one column of the slice at a
    // time), columns of U along the columns; both land in vt[vector][entry]
    // (addresses stay at the last column / vector once past it; a batch of
    // loads is in flight before the first value goes to LDS)
    constexpr int NB = 32;
    if (is_l) {
      const int64_t v = v0 + vl;
      const T* p = l + (v < cl ? v : cl);
#pragma unroll 1
      for (int c0 = 0; c0 < SW; c0 += NB) {
        T y[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          y[c] = *p;
          p += c0 + c < sw - 1 ? g.ldl : 0;
        }
#pragma unroll
        for (int c = 0; c < NB; ++c) xl[c0 + c] = (float)y[c];
      }
    } else {
      const int64_t va = v0 < cl ? v0 : cl;
      const int nv = (int)(cl - va < VPU - 1 ? cl - va : VPU - 1);
      const T* p = u + va * g.ldu + (lane < sw ? lane : sw - 1);
#pragma unroll 1
      for (int c0 = 0; c0 < VPU; c0 += NB) {
        T y[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          y[c] = *p;
          p += c0 + c < nv ? g.ldu : 0;
        }
#pragma unroll
        for (int c = 0; c < NB; ++c) vt[c0 + c][lane] = (float)y[c];
      }
    }
    wave_sync();
    if constexpr (Ty::MM) {
      if (g.pre) {
        const O* const mop = (is_l ? uop : lop) + (so + l32) * g.ldop;
        const O* const vop = is_l ? lop : uop;
        const O* am[2] = {mop, mop + 32 * g.ldop};
        const O* bn[VG];
#pragma unroll
        for (int r = 0; r < VG; ++r) {
          const int64_t v = v0 + 32 * r + l32;
          bn[r] = vop + (so + (v < cl ? v : cl)) * g.ldop;
        }
        const int step = RL ? g.chunk : so;
#pragma unroll 1
        for (int k0 = 0; k0 < so; k0 += step) {
          Cross<MODE, 0> pre;
          pre.zero();
          const O* a0[2] = {am[0] + k0, am[1] + k0};
          const O* b0[VG];
#pragma unroll
          for (int r = 0; r < VG; ++r) b0[r] = bn[r] + k0;
          op_sum<MODE, 4, 2, VG>(pre.acc, a0, b0, step, lh);
          static_for<8>([&](auto pi) {
            constexpr int P = decltype(pi)::value;
            float a[8];
            pre.template get<P>(a);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              float y = xl[8 * P + c] - a[c];
              if constexpr (RL && MODE >= SM_F16_TC) y = r16(y);
              xl[8 * P + c] = y;
            }
          });
        }
      }
    }
#pragma unroll 1
    for (int c = sw; c < SW; ++c) xl[c] = 0.0f;
    // each finished panel goes out while the wave waits for the next one:
    // factors and mirror (rows of L across the lanes; columns of U as one
    // 16-byte run per lane where they are aligned, else through vt at the
    // end), and the operand copy
    const int nv = (int)(g.cm - v0 < VPU ? g.cm - v0 : VPU);
    const bool mine = lane < nv;
    T* const px = is_l ? l + v0 + vl : u + (v0 + vl) * g.ldu;
    half_t* const pc = g.cp + (is_l ? v0 + vl : (v0 + vl) * g.ldcp);
    O* const po = (O*)(is_l ? g.lop : g.uop) + (so + v0 + vl) * g.ldop + so;
    const bool vec = g.vec && sw == SW;
    const bool late = !is_l && !vec;
    unit_solve<MODE, RL, IB>(S, xl, is_l, lane, [&](int p0, const X(&p)[8]) {
      if (late) {
#pragma unroll
        for (int c = 0; c < 8; ++c) xl[p0 + c] = (float)p[c];
      }
      if (!mine || p0 >= sw) return;
      if (g.write_op) {
        if constexpr (MODE == SM_F32) {
          *(float4*)(po + p0) = make_float4(p[0], p[1], p[2], p[3]);
          *(float4*)(po + p0 + 4) = make_float4(p[4], p[5], p[6], p[7]);
        } else {
          su8 w;
#pragma unroll
          for (int e = 0; e < 8; ++e) w[e] = op16<MODE>((float)p[e]);
          *(su8*)(po + p0) = w;
        }
      }
      if (late) return;
      if (is_l) {
        auto put = [&](auto* q, int64_t st) {
          using Q = typename std::remove_pointer<decltype(q)>::type;
          if (p0 + 8 <= sw) {
#pragma unroll
            for (int c = 0; c < 8; ++c, q += st) *q = (Q)p[c];
          } else {
#pragma unroll
            for (int c = 0; c < 8; ++c, q += st)
              if (p0 + c < sw) *q = (Q)p[c];
          }
        };
        if (g.store_x) put(px + p0 * g.ldl, g.ldl);
        if (g.cp) put(pc + p0 * g.ldcp, g.ldcp);
      } else {
        sh8 w;
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = (half_t)p[e];
        if (g.cp) *(sh8*)(pc + p0) = w;
        if (g.store_x) {
          if constexpr (std::is_same<T, float>::value) {
            *(float4*)(px + p0) = make_float4(p[0], p[1], p[2], p[3]);
            *(float4*)(px + p0 + 4) = make_float4(p[4], p[5], p[6], p[7]);
          } else {
            *(sh8*)(px + p0) = w;
          }
        }
      }
    });
    if (late) {
      wave_sync();
      auto put = [&](auto* q, int64_t st) {
        using Q = typename std::remove_pointer<decltype(q)>::type;
#pragma unroll 1
        for (int c0 = 0; c0 < nv; c0 += 16) {
          float y[16];
#pragma unroll
          for (int c = 0; c < 16; ++c) y[c] = vt[c0 + c < nv ? c0 + c : nv - 1][lane];
#pragma unroll
          for (int c = 0; c < 16; ++c) {
            if (c0 + c < nv) *q = (Q)y[c];
            q += st;
          }
        }
      };
      if (lane < sw) {
        if (g.store_x) put(u + lane + v0 * g.ldu, g.ldu);
        if (g.cp) put(g.cp + lane + v0 * g.ldcp, g.ldcp);
      }
      wave_sync();  // (vt is filled again by the next unit)
    }
  }
}

template <typename T, int MODE, bool RL>
int launch_ib(remifa_handle_t h, int ib, const SliceArgs& g, int grid) {
  switch (ib) {
    case 8: slice_kernel<T, MODE, RL, 8><<<grid, SLT, 0, h->stream>>>(g); break;
    case 16: slice_kernel<T, MODE, RL, 16><<<grid, SLT, 0, h->stream>>>(g); break;
    case 32: slice_kernel<T, MODE, RL, 32><<<grid, SLT, 0, h->stream>>>(g); break;
    default: slice_kernel<T, MODE, RL, 64><<<grid, SLT, 0, h->stream>>>(g); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : REMIFA_ERR_HIP;
}

}  // namespace
}  // namespace remifa
