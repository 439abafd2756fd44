// Launches of the slice kernel (slice.hpp; instantiated per arithmetic in
// slice_*.hip) and the final copy of the last tile.
#include <algorithm>

#include "slice.hpp"

namespace remifa {

int slice_f32_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid);
int slice_f32tc_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid);
int slice_f16tc_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid);
int slice_f16h_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid);
int slice_f16bf_launch(remifa_handle_t h, bool rl, int ib, const SliceArgs& g, int grid);

namespace {

// Last slice's tile to the matrix and *info: the first zero or non-finite
// pivot (1-based), from the slots' running value for columns >= c0 (slices)
// and from the matrix's diagonal for the columns before.
template <typename WT>
__global__ void __launch_bounds__(256) slice_finish_kernel(int64_t c0, const WT* __restrict__ a,
                                                           int64_t lda,
                                                           const float* __restrict__ prev, WT* pa,
                                                           half_t* pcp, int64_t ldpcp, int psw,
                                                           int* info) {
  __shared__ int first;
  const int t = threadIdx.x;
  if (t == 0) first = 0x7fffffff;
  if (prev) {
#pragma unroll 8
    for (int e = t; e < SW * SW; e += 256) {
      const int i = e % SW, j = e / SW;
      const float v = prev[SLOT_HDR + e];
      if (i < psw && j < psw) {
        pa[i + j * lda] = (WT)v;
        if (pcp) pcp[i + j * ldpcp] = (half_t)v;
      }
    }
  }
  if (!info) return;  // uniform
  __syncthreads();
  for (int64_t k = t; k < c0; k += 256) {
    const float v = (float)a[k + k * lda];
    if (v == 0.0f || !__builtin_isfinite(v)) atomicMin(&first, (int)(k + 1));
  }
  __syncthreads();
  if (t == 0) {
    const int s = prev ? ((const int*)prev)[0] : 0;
    *info = first != 0x7fffffff ? first : s;
  }
}

// mode from (type of the factored buffers, inner compute type): see SubMode
int slice_mode(int T, int I) {
  if (T == REMIFA_R_32F) return I == REMIFA_FP32 ? SM_F32 : SM_F32_TC;
  if (I == REMIFA_FP16 || I == REMIFA_TC16) return SM_F16_H;
  if (I == REMIFA_BF16_TC32) return SM_F16_BF;
  return SM_F16_TC;
}

size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }
size_t op_size(int T, int I) { return slice_mode(T, I) == SM_F32 ? 4 : 2; }

// leading dimension of the operand copies: whole 128-byte lines per row, and
// not a power of two of them (rows spread over the L2 channels)
int64_t op_ld(int64_t nb) { return (nb + 63) / 64 * 64 + 64; }

}  // namespace

size_t slice_slot_bytes() { return (SLOT_HDR + SW * SW) * sizeof(float); }

// operand copies of an outer block of nb columns (and as many rows) out of m
size_t slice_op_bytes(int T, int I, int64_t m, int64_t nb) {
  return 2 * al256((size_t)(m + SW) * op_ld(nb) * op_size(T, I));
}

// true if the slice kernel can subtract the earlier slices' products itself;
// else the driver runs the update GEMMs (fp16-accumulated sums; bf16 operands
// rounded from the fp16 mirror of fp32 buffers)
bool slice_updates(int T, int I) {
  return slice_mode(T, I) != SM_F16_H && !(T == REMIFA_R_32F && I == REMIFA_BF16_TC32);
}

// One slice at offset so of the outer block (m rows below and including its
// first row): l, u, cp point at the slice's diagonal tile. nb: width of the
// outer block's operand copies ops (null: the driver runs the update GEMMs).
//
// Measured (MI355X): a slice takes 22 us at n = 5001 (fp16 panels, ib = 8, nb
// = 256) where the tile kernel (30), the vector kernel (22) and the update
// GEMMs (20) took 72; 31 against 41 + 20 right-looking at n = 4096, ib = 32.
// Whole factorizations: 6.90 -> 3.32 ms there, 3.82 -> 2.34 right-looking,
// 12.4 -> 8.6 in fp32 at n = 8192, 0.33 -> 0.20 at n = 300.
int slice_launch(remifa_handle_t h, int T, int W, int I, bool rl, int ib, int pw, int64_t m,
                 int64_t nb, int64_t so, int sw, bool last, void* l, int64_t ldl, void* u,
                 int64_t ldu, bool store_x, half_t* cp, int64_t ldcp, void* ops, void* a,
                 int64_t lda, half_t* acp, int64_t ldacp, int64_t col, SlicePending& pend) {
  const int mode = slice_mode(T, I);
  const int64_t cm = m - so;
  if (sw <= 0) return 0;
  if (sw > SW || cm < sw || (ib != 8 && ib != 16 && ib != 32 && ib != 64))
    return REMIFA_ERR_UNSUPPORTED;
  SliceArgs g{};
  g.cm = cm, g.sw = sw, g.so = (int)so, g.chunk = pw;
  g.pre = so > 0 && ops;
  g.l = l, g.ldl = ldl, g.u = u, g.ldu = ldu, g.store_x = store_x;
  g.cp = cp, g.ldcp = ldcp;
  const int64_t es16 = 16 / (int64_t)dtype_size(T);
  g.vec = (!store_x || ((uintptr_t)u % 16 == 0 && ldu % es16 == 0)) &&
          (!cp || ((uintptr_t)cp % 16 == 0 && ldcp % 8 == 0));
  g.ldop = op_ld(nb);
  if (ops) {
    g.lop = ops;
    g.uop = (char*)ops + al256((size_t)(m + SW) * g.ldop * op_size(T, I));
  }
  g.write_op = !last && ops;
  const int vpu = mode == SM_F32 ? 32 : 64;
  g.nul = (int)ceil_div(cm - sw, vpu);
  g.nunits = 2 * g.nul;
  g.slot = pend.slots + (size_t)(pend.next & 1) * (slice_slot_bytes() / sizeof(float));
  if (pend.sw) {
    g.prev = pend.slots + (size_t)((pend.next + 1) & 1) * (slice_slot_bytes() / sizeof(float));
    g.pa = pend.a, g.lda = lda, g.pcp = pend.cp, g.ldpcp = ldacp, g.psw = pend.sw;
  }
  g.col = col;
  g.w_half = W == REMIFA_R_16F;
  // one unit per workgroup first (latency), then more units per wavefront
  const int grid = std::max(1, std::min(g.nunits, h->num_cu));
  const size_t es = dtype_size(T);
  const double rest = (double)(cm - sw);
  timer_begin(h, KC_PANEL, 2.0 * (2.0 * rest * sw) * es + (cp ? 2.0 * rest * sw * 2 : 0.0), 0);
  int st;
  switch (mode) {
    case SM_F32: st = slice_f32_launch(h, rl, ib, g, grid); break;
    case SM_F32_TC: st = slice_f32tc_launch(h, rl, ib, g, grid); break;
    case SM_F16_TC: st = slice_f16tc_launch(h, rl, ib, g, grid); break;
    case SM_F16_H: st = slice_f16h_launch(h, rl, ib, g, grid); break;
    default: st = slice_f16bf_launch(h, rl, ib, g, grid); break;
  }
  timer_end(h);
  if (st) return st;
  if (pend.first_col < 0) pend.first_col = col;
  pend.a = a;
  pend.cp = acp;
  pend.sw = sw;
  ++pend.next;
  return 0;
}

// the pending tile to the matrix, and the pivot check (info may be null)
int slice_finish_launch(remifa_handle_t h, int W, int64_t n, const void* d_a, int64_t lda,
                        int64_t ldacp, const SlicePending& pend, int* info) {
  if (!pend.sw && !info) return 0;
  const float* prev =
      pend.sw ? pend.slots + (size_t)((pend.next + 1) & 1) * (slice_slot_bytes() / sizeof(float))
              : nullptr;
  const int64_t c0 = pend.sw ? pend.first_col : n;
  if (W == REMIFA_R_32F)
    slice_finish_kernel<float><<<1, 256, 0, h->stream>>>(c0, (const float*)d_a, lda, prev,
                                                         (float*)pend.a, pend.cp, ldacp, pend.sw,
                                                         info);
  else
    slice_finish_kernel<half_t><<<1, 256, 0, h->stream>>>(c0, (const half_t*)d_a, lda, prev,
                                                          (half_t*)pend.a, pend.cp, ldacp, pend.sw,
                                                          info);
  RF_HIP(hipGetLastError());
  return 0;
}

}  // namespace remifa
