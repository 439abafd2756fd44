// FP8 update GEMM (included by gemm.hip inside its anonymous namespace,
// after gemm_mfma.hpp). C = alpha A B + beta C with OCP e4m3 operands and
// one power-of-two (E8M0) scale per 32-long K block of every row of A and
// every column of B, on the gfx950 scaled matrix cores
// (v_mfma_scale_f32_32x32x64_f8f6f4), fp32 accumulation.
//
// Operand formats (both K-contiguous, so both fragments are plain 16-byte
// LDS reads):
//   qa[m * ldqa + k]  codes of A (row m, column k), sa[m * ldsa + k / 32]
//   qb[n * ldqb + k]  codes of B (row k, column n), sb[n * ldsb + k / 32]
// A scale byte s stands for 2^(s - 127). The quantizer below produces them
// from column-major fp16 / fp32 matrices: per 32-block, scale 2^(floor(log2
// amax) - 8) (the OCP MX rule for e4m3, emax = 8), codes rounded to nearest
// even with saturation at +-448.
//
// Matrix-core operand layout (32x32x64, 8-bit): lane l holds row l % 32 of
// its operand; bytes 0-15 are K 16 h .. 16 h + 15 and bytes 16-31 are
// K 32 + 16 h .. 32 + 16 h + 15 (h = l / 32), and lane (r + 32 b) supplies
// the scale of row r for the 32-block b. The MFMA computes D^T = B^T A^T as
// the 16-bit kernel does, so the accumulator layout and epilogue match it.

struct Fp8Args {
  int64_t M, N, K;
  const uint8_t* A;
  int64_t lda;
  const uint8_t* SA;
  int64_t ldsa;
  const uint8_t* B;
  int64_t ldb;
  const uint8_t* SB;
  int64_t ldsb;
  float alpha, beta;
  void* C;
  int64_t ldc;
  const void* Cin;  // optional source of the beta term (else C): fp16 or fp32
  int64_t ldcin;
  int cin_half;
  float* W;        // split-K partials [split][N][ldw]
  int64_t ldw;
  int64_t kchunk;  // K range per split (multiple of 128)
  int tiles_m, tiles_n;
};

typedef int v8i32 __attribute__((ext_vector_type(8)));

// v if ok, else zeros (component selects: a select of whole structs would
// turn into an address select and push the staging registers to memory)
__device__ __forceinline__ uint4 keep16(bool ok, uint4 v) {
  return make_uint4(ok ? v.x : 0u, ok ? v.y : 0u, ok ? v.z : 0u, ok ? v.w : 0u);
}

__device__ __forceinline__ v8i32 join16(uint4 lo, uint4 hi) {
  return (v8i32){(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w,
                 (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

// scale bytes of a 128-long K slab (four 32-blocks) of row r, in two steps
// so that nothing waits for the load before the matrix-core work: the word
// (from a clamped, in-bounds address when out of range) and the number of
// its valid blocks; blocks past the K range, and rows past the matrix, then
// read as 2^0 (their codes are 0)
__device__ __forceinline__ uint32_t scale_word(const uint8_t* s, int64_t lds, int64_t r,
                                               int64_t nrows, int64_t kb0, int64_t nkb,
                                               int& valid) {
  const bool ok = r < nrows && kb0 < nkb;
  valid = ok ? (int)(nkb - kb0 < 4 ? nkb - kb0 : 4) : 0;
  return *(const uint32_t*)(s + (ok ? r * lds + kb0 : 0));
}
__device__ __forceinline__ uint32_t scale_mask(uint32_t w, int valid) {
  // bytes >= valid -> 127
  const uint32_t keep = valid >= 4 ? 0xFFFFFFFFu : ((1u << (8 * valid)) - 1u);
  return (w & keep) | (0x7F7F7F7Fu & ~keep);
}

template <typename OutT>
__global__ void __launch_bounds__(256, 2) gemm_fp8_kernel(Fp8Args g) {
  constexpr int BM = 128, BN = 128, BK = 128;  // BK: K per slab (bytes per row)
  constexpr int P = BK + 16;  // LDS row pitch: 16 rows of a fragment read hit distinct banks
  __shared__ __attribute__((aligned(16))) uint8_t As[2][BM * P];
  __shared__ __attribute__((aligned(16))) uint8_t Bs[2][BN * P];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave % 2, wn = wave / 2;  // 2 x 2 waves of 64 x 64
  const int l32 = lane & 31, lh = lane >> 5;

  const int nt = g.tiles_m * g.tiles_n;
  const int tile = xcd_tile(blockIdx.x, nt);
  constexpr int GM = 8;  // grouped raster (as the 16-bit kernel)
  const int gsz = GM * g.tiles_n;
  const int grp = tile / gsz, first = grp * GM;
  const int rows = g.tiles_m - first < GM ? g.tiles_m - first : GM;
  const int tm = first + (tile % gsz) % rows, tn = (tile % gsz) / rows;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t kbeg = (int64_t)blockIdx.z * g.kchunk;
  const int64_t kend = kbeg + g.kchunk < g.K ? kbeg + g.kchunk : g.K;
  const int64_t klen = kend > kbeg ? kend - kbeg : 0;
  const int nk = (int)((klen + BK - 1) / BK);
  const bool split = gridDim.z > 1;
  const int64_t nkb = kend / 32;  // 32-blocks below kend (K is a multiple of 32)

  uint4 ra[4], rb[4];
  bool oka[4], okb[4];
  uint32_t nsa[2], nsb[2];  // scale words of the slab being loaded
  int nva[2], nvb[2];       // and their valid block counts
  uint32_t csa[2], csb[2];  // scale words of the slab being computed

  auto load_slab = [&](int kt) {
    const int64_t k0 = kbeg + (int64_t)kt * BK;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int c = tid + 256 * p;
      const int row = c >> 3, kq = c & 7;
      const int64_t gk = k0 + 16 * kq;
      const int64_t gm = m0 + row, gn = n0 + row;
      const bool ka = gm < g.M && gk < kend, kb = gn < g.N && gk < kend;
      ra[p] = *(const uint4*)(g.A + (ka ? gm * g.lda + gk : 0));
      rb[p] = *(const uint4*)(g.B + (kb ? gn * g.ldb + gk : 0));
      oka[p] = ka;
      okb[p] = kb;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      nsa[i] = scale_word(g.SA, g.ldsa, m0 + wm * 64 + i * 32 + l32, g.M, k0 / 32, nkb, nva[i]);
      nsb[i] = scale_word(g.SB, g.ldsb, n0 + wn * 64 + i * 32 + l32, g.N, k0 / 32, nkb, nvb[i]);
    }
  };
  auto store_tiles = [&](int buf) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int c = tid + 256 * p;
      const int row = c >> 3, kq = c & 7;
      *(uint4*)&As[buf][row * P + 16 * kq] = keep16(oka[p], ra[p]);
      *(uint4*)&Bs[buf][row * P + 16 * kq] = keep16(okb[p], rb[p]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      csa[i] = scale_mask(nsa[i], nva[i]);
      csb[i] = scale_mask(nsb[i], nvb[i]);
    }
  };

  f16v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;

  // one 64-long K step (two 32-blocks): opsel picks scale byte 2 s (+ lh via the shift)
  auto kstep = [&](const uint8_t* as, const uint8_t* bs, int s, auto opsel_tag) {
    constexpr int OPS = decltype(opsel_tag)::value;
    v8i32 xb[2], ya[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint8_t* p = &bs[(wn * 64 + j * 32 + l32) * P + 64 * s + 16 * lh];
      xb[j] = join16(*(const uint4*)p, *(const uint4*)(p + 32));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint8_t* p = &as[(wm * 64 + i * 32 + l32) * P + 64 * s + 16 * lh];
      ya[i] = join16(*(const uint4*)p, *(const uint4*)(p + 32));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            xb[j], ya[i], acc[i][j], 0, 0, OPS, (int)(csb[j] >> (8 * lh)), OPS,
            (int)(csa[i] >> (8 * lh)));
  };
  auto compute = [&](int buf) {
    kstep(As[buf], Bs[buf], 0, std::integral_constant<int, 0>{});
    kstep(As[buf], Bs[buf], 1, std::integral_constant<int, 2>{});
  };

  if (nk > 0) {
    load_slab(0);
    store_tiles(0);
  }
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    // straight-line body (after the last slab the loads are masked, clamped
    // to in-bounds addresses, and land in the buffer nobody reads again): a
    // branch around the stores lets the compiler sink the matrix-core work
    // below them, behind the waits for the loads just issued
    load_slab(kt + 1);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out first
    compute(buf);
    __builtin_amdgcn_sched_barrier(0);
    store_tiles(buf ^ 1);
    __syncthreads();
  }

  // epilogue: lane holds C[m = .. + l32][n = .. + 8*(q/4) + 4*lh + q%4];
  // the beta term's source (C, or Cin in fp16 / fp32) is chosen once per
  // workgroup, outside the loops
  auto epilogue = [&](const auto* __restrict__ src, int64_t lds_) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t m = m0 + wm * 64 + i * 32 + l32;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int64_t nb = n0 + wn * 64 + j * 32 + 4 * lh;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int64_t n = nb + 8 * (q >> 2) + (q & 3);
          if (m >= g.M || n >= g.N) continue;
          if (split) {
            g.W[((int64_t)blockIdx.z * g.N + n) * g.ldw + m] = g.alpha * acc[i][j][q];
          } else {
            const float cv = g.beta != 0.0f ? (float)src[m + n * lds_] : 0.0f;
            ((OutT*)g.C)[m + n * g.ldc] =
                (OutT)__builtin_fmaf(g.alpha, acc[i][j][q], g.beta * cv);
          }
        }
      }
    }
  };
  if (split || !g.Cin)
    epilogue((const OutT*)g.C, g.ldc);
  else if (g.cin_half)
    epilogue((const half_t*)g.Cin, g.ldcin);
  else
    epilogue((const float*)g.Cin, g.ldcin);
}

// ------------------------------------------------------------ 256 x 256 tile
// 16 bytes (4 bytes) per lane: as dma16 of gemm_big.hpp
__device__ __forceinline__ void dma4(const u32x4& rsrc, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dword %0, %1, 0 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(lds_base))
               : "memory", "m0");
}

// One 512-thread workgroup per CU owns a 256 x 256 tile, each wavefront 128 x
// 64 of it; K slabs of 64 come through LDS-DMA requests into a ring of four
// stages, as in gemm_big_kernel. Both operands are K-contiguous: a row is 64
// bytes (four 16-byte units, unit c at c ^ ((row / 4) % 4), so that the 16
// lanes of a read phase hit 16 different bank groups), a fragment two 16-byte
// reads per lane. The scales come with the slab, a 4-byte word per row (the
// four 32-blocks of 128 k-values; the slab uses two of its bytes). Bound by
// the matrix cores and the LDS alike: 1024 cycles of each per slab (half the
// LDS bytes per flop of the 128 x 128 tile). Rows and columns outside the
// matrix repeat its last ones (their products are not stored); a last slab of
// 32 k-values is cleared past them in LDS and its scales there set to 2^0.
// Measured (MI355X) at 8192 x 8192 x 4096: 327 us, 1.68 PFLOP/s (128 x 128
// tiles: 533 us).
template <typename OutT>
__global__ void __launch_bounds__(512) gemm_fp8_big_kernel(Fp8Args g) {
  constexpr int BK = 64, NS = 4, FN = 2, WTN = 64;
  constexpr int OP_ST = 256 * BK;              // bytes of an operand slab
  constexpr int SC = 2 * OP_ST;                // scale words: A's rows, then B's columns
  constexpr int ST = SC + 2 * 256 * 4;         // bytes of a stage
  constexpr int REQ = 5;                       // requests of a wavefront per slab
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * ST];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int l32 = lane & 31, lh = lane >> 5;

  const int nt = g.tiles_m * g.tiles_n;
  const int tile = xcd_tile(blockIdx.x, nt);
  constexpr int GM = 8;  // grouped raster (as the 16-bit kernel)
  const int gsz = GM * g.tiles_n;
  const int grp = tile / gsz, first = grp * GM;
  const int rows = g.tiles_m - first < GM ? g.tiles_m - first : GM;
  const int tm = first + (tile % gsz) % rows, tn = (tile % gsz) / rows;
  const int64_t m0 = (int64_t)tm * 256, n0 = (int64_t)tn * 256;
  const int64_t kbeg = (int64_t)blockIdx.z * g.kchunk;
  const int64_t kend = kbeg + g.kchunk < g.K ? kbeg + g.kchunk : g.K;
  const int nk = kend > kbeg ? (int)((kend - kbeg + BK - 1) / BK) : 0;
  const bool half_slab = kend > kbeg && (kend - kbeg) % BK != 0;  // 32 k-values in the last
  const int mv = g.M - m0 < 256 ? (int)(g.M - m0) : 256;
  const int nv = g.N - n0 < 256 ? (int)(g.N - n0) : 256;

  // lane offsets in bytes from the corner of a slab: two operand requests
  // each, and the scale words of 64 rows (wavefronts 0-3: A, 4-7: B)
  uint32_t offa[2], offb[2];
  auto lane_offsets = [&](bool half) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int p = (wave * 2 + t) * 64 + lane;  // 16-byte position in the slab
      const int r = p / 4;
      int c = (p % 4) ^ ((r / 4) % 4);
      if (half) c &= 1;
      offa[t] = (uint32_t)((int64_t)(r < mv ? r : mv - 1) * g.lda + 16 * c);
      offb[t] = (uint32_t)((int64_t)(r < nv ? r : nv - 1) * g.ldb + 16 * c);
    }
  };
  lane_offsets(false);
  const bool sc_b = wave >= 4;
  const int sr = 64 * (wave & 3) + lane, sv = sc_b ? nv : mv;
  const uint32_t offs = (uint32_t)((int64_t)(sr < sv ? sr : sv - 1) * (sc_b ? g.ldsb : g.ldsa));
  const uint8_t* const sbase = sc_b ? g.SB + n0 * g.ldsb : g.SA + m0 * g.ldsa;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_vptr)lds);
  auto issue = [&](int k, int st) {
    const int64_t kk = kbeg + (int64_t)k * BK;
    const u32x4 ra = big_rsrc(g.A + m0 * g.lda + kk);
    const u32x4 rb = big_rsrc(g.B + n0 * g.ldb + kk);
    const u32x4 rs = big_rsrc(sbase + (kk / 128) * 4);
    const uint32_t as = lds0 + (uint32_t)(st * ST);
#pragma unroll
    for (int t = 0; t < 2; ++t) dma16(ra, offa[t], as + (uint32_t)((wave * 2 + t) * 1024));
#pragma unroll
    for (int t = 0; t < 2; ++t)
      dma16(rb, offb[t], as + (uint32_t)(OP_ST + (wave * 2 + t) * 1024));
    dma4(rs, offs, as + (uint32_t)(SC + wave * 256));
  };

  // fragment addresses (bytes from the stage): rows 32 apart share the swizzle
  const int ra0 = 128 * wm + l32, rb0 = WTN * wn + l32;
  const int fa = (ra0 / 4) % 4, fb = (rb0 / 4) % 4;
  int aoff[2], boff[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    aoff[u] = (ra0 * 4 + ((2 * u + lh) ^ fa)) * 16;
    boff[u] = OP_ST + (rb0 * 4 + ((2 * u + lh) ^ fb)) * 16;
  }

  f16v acc[4][FN];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;

  auto compute = [&](int st, int k) {
    const uint8_t* const base = lds + st * ST;
    const int sh = 8 * (2 * (k & 1) + lh);  // this lane's 32-block of the word
    v8i32 xb[FN], ya[4];
    int sa[4], sb[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      sb[j] = (int)(*(const uint32_t*)(base + SC + 1024 + 4 * (rb0 + 32 * j)) >> sh);
      xb[j] = join16(*(const uint4*)(base + boff[0] + j * 2048),
                     *(const uint4*)(base + boff[1] + j * 2048));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sa[i] = (int)(*(const uint32_t*)(base + SC + 4 * (ra0 + 32 * i)) >> sh);
      ya[i] = join16(*(const uint4*)(base + aoff[0] + i * 2048),
                     *(const uint4*)(base + aoff[1] + i * 2048));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(xb[j], ya[i], acc[i][j], 0, 0,
                                                                    0, sb[j], 0, sa[i]);
  };

  // (a half slab is the last request: its lane offsets replace the others)
  const int nfull = nk - (half_slab ? 1 : 0);
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (p < nk) {
      if (p == nfull) lane_offsets(true);
      issue(p, p);
    }
  int k = 0, st = 0;
  for (; k + NS - 1 < nfull; ++k) {
    vm_wait_barrier<(NS - 2) * REQ>();
    compute(st, k);
    issue(k + NS - 1, st == 0 ? NS - 1 : st - 1);
    st = st == NS - 1 ? 0 : st + 1;
  }
  bool half_pending = half_slab && nk >= NS;
  for (; k < nk; ++k) {
    vm_wait_barrier<0>();
    if (k == nfull) {
      uint8_t* const base = lds + st * ST;
      for (int p = tid; p < 2 * 1024; p += 512) {
        const int r = (p % 1024) / 4;
        if (((p % 4) ^ ((r / 4) % 4)) >= 2) *(uint4*)(base + p * 16) = make_uint4(0, 0, 0, 0);
      }
      const int b = 8 * (2 * (k & 1) + 1);
      uint32_t* const sw = (uint32_t*)(base + SC) + tid;
      *sw = (*sw & ~(0xFFu << b)) | (0x7Fu << b);
      __syncthreads();
    }
    compute(st, k);
    if (half_pending) {
      lane_offsets(true);
      issue(nfull, st == 0 ? NS - 1 : st - 1);
      half_pending = false;
    }
    st = st == NS - 1 ? 0 : st + 1;
  }
  big_epilogue<OutT, FN, WTN>(g, acc, wm, wn, l32, lh, m0, n0, mv, nv);
}

// ---------------------------------------------------------------- quantizer
// For each 32-block the scale exponent 2^(floor(log2 amax) - 8) (2^0 for an
// all-zero or non-finite block) and 32 codes, rounded by the conversion
// instruction (to nearest even, after saturation at +-448); NaNs, which the
// maximum skips, through the bit-level conversion. Codes past K are zero,
// nothing past the last 32-block is written. HBM-bound (3 bytes per fp16
// entry): 16-byte reads and whole-line writes. Measured (MI355X), 8192 x
// 4096 fp16: rows 63 -> 28 us, columns 94 -> 26 us against one lane per 32-block.
__device__ __forceinline__ int quant_exponent(float amax) {
  int se = 0;
  if (amax > 0.0f && amax <= 3.4028235e38f) {
    int e;
    frexpf(amax, &e);
    se = e - 1 - 8;
  }
  return se;
}

// codes of four values
__device__ __forceinline__ uint32_t quant_codes4(const float* v, int se) {
  float y[4];
  bool nan = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y[e] = ldexpf(v[e], -se);
    nan |= y[e] != y[e];
  }
  if (nan) {
    uint32_t x = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) x |= (uint32_t)f32_to_e4m3_bits(y[e]) << (8 * e);
    return x;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = fminf(fmaxf(y[e], -448.0f), 448.0f);
  int x = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], x, true);
}

template <typename T, int N>
struct QVec {
  T e[N];
};

// Columns: element (k, r) at src[k + r * ld] (B operands). Four lanes per
// 32-block, eight values each; the workgroup is blockDim.x lanes along K and
// blockDim.y along the columns, QC columns per thread.
constexpr int QC = 4;
template <typename T>
__global__ void __launch_bounds__(256) quant_fp8_cols_kernel(int64_t R, int64_t K,
                                                             const T* __restrict__ src, int64_t ld,
                                                             uint8_t* __restrict__ q, int64_t ldq,
                                                             uint8_t* __restrict__ s,
                                                             int64_t lds) {
  const int64_t k = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  const int64_t r0 = ((int64_t)blockIdx.y * blockDim.y + threadIdx.y) * QC;
  QVec<T, 8> x[QC];
  if (k + 8 <= K && r0 + QC <= R) {
#pragma unroll
    for (int c = 0; c < QC; ++c) __builtin_memcpy(&x[c], src + k + (r0 + c) * ld, sizeof(x[c]));
  } else {
#pragma unroll
    for (int c = 0; c < QC; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool ok = k + e < K && r0 + c < R;
        x[c].e[e] = ok ? src[k + e + (r0 + c) * ld] : (T)0.0f;
      }
  }
  const bool in = k < (K + 31) / 32 * 32;
#pragma unroll
  for (int c = 0; c < QC; ++c) {
    float v[8], amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = (float)x[c].e[e];
      amax = fmaxf(amax, fabsf(v[e]));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
    amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
    const int se = quant_exponent(amax);
    if (!in || r0 + c >= R) continue;
    *(uint2*)(q + (r0 + c) * ldq + k) = make_uint2(quant_codes4(v, se), quant_codes4(v + 4, se));
    if (threadIdx.x % 4 == 0) s[(r0 + c) * lds + k / 32] = (uint8_t)(se + 127);
  }
}

// Rows: element (r, k) at src[r + k * ld] (A operands), so blocks run across
// the stored columns. A workgroup transposes 64 rows x 128 k-values through
// LDS: lanes read consecutive rows, then each thread owns the 32-block
// (row t % 64, block t / 64), then the codes leave as 128 bytes per row.
template <typename T>
__global__ void __launch_bounds__(256) quant_fp8_rows_kernel(int64_t R, int64_t K,
                                                             const T* __restrict__ src, int64_t ld,
                                                             uint8_t* __restrict__ q, int64_t ldq,
                                                             uint8_t* __restrict__ s,
                                                             int64_t lds) {
  constexpr int V = 16 / (int)sizeof(T);  // rows per read
  constexpr int L = 64 / V;               // lanes per column of the tile
  constexpr int NI = 128 * L / 256;       // reads per thread
  constexpr int QP = 128 + 16;            // pitch of a row's codes
  __shared__ __attribute__((aligned(16))) T tile[128 * 64];
  __shared__ __attribute__((aligned(16))) uint8_t codes[64 * QP];
  const int t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * 64, k0 = (int64_t)blockIdx.y * 128;
  const int64_t kpad = (K + 31) / 32 * 32;
  QVec<T, V> x[NI];
  const bool full = r0 + 64 <= R && k0 + 128 <= K;
  if (full) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
      __builtin_memcpy(&x[i], src + r0 + V * (t % L) + (k0 + t / L + i * (256 / L)) * ld,
                       sizeof(x[i]));
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const int64_t r = r0 + V * (t % L) + e, k = k0 + t / L + i * (256 / L);
        x[i].e[e] = (r < R && k < K) ? src[r + k * ld] : (T)0.0f;
      }
  }
#pragma unroll
  for (int i = 0; i < NI; ++i)
    *(QVec<T, V>*)&tile[(t / L + i * (256 / L)) * 64 + V * (t % L)] = x[i];
  __syncthreads();
  const int r = t % 64, b = t / 64;
  float v[32], amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    v[j] = (float)tile[(32 * b + j) * 64 + r];
    amax = fmaxf(amax, fabsf(v[j]));
  }
  const int se = quant_exponent(amax);
  uint32_t w[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) w[u] = quant_codes4(v + 4 * u, se);
  *(uint4*)&codes[r * QP + 32 * b] = make_uint4(w[0], w[1], w[2], w[3]);
  *(uint4*)&codes[r * QP + 32 * b + 16] = make_uint4(w[4], w[5], w[6], w[7]);
  if (r0 + r < R && k0 + 32 * b < K) s[(r0 + r) * lds + k0 / 32 + b] = (uint8_t)(se + 127);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int rr = t / 8 + 32 * i, u = t % 8;
    if (r0 + rr < R && k0 + 16 * u < kpad)
      *(uint4*)(q + (r0 + rr) * ldq + k0 + 16 * u) = *(const uint4*)&codes[rr * QP + 16 * u];
  }
}
