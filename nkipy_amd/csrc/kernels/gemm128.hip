// MFMA GEMM over 128 x 128 output tiles, for products whose 256 x 256 tiles
// (gemm.hip) do not fill the part: row counts from a few dozen to a few
// thousand.  Same operands, epilogues and arithmetic (bf16 MFMA on exact
// weights, fp32 accumulation, the traced cast points).
//
// 256 threads = 4 waves (2 x 2); each wave owns 64 rows and 32 columns of
// each 64-column half of the tile (4 x 4 tiles of v_mfma_f32_16x16x32_bf16),
// so that a wave holds matching gate / up columns (SwiGLU: half 0 gate, half
// 1 up) or matching halves of one 128-wide head (rotary epilogue).  At most
// 80 KiB of LDS and 256 registers: two workgroups share a CU, and one's MFMAs
// run while the other waits for its fragments.
//
// LDS rings filled by DMA (buffer_load ... lds, tracked by explicit vmcnt
// waits).  A: three blocks of 64 k, 128 rows x 128 B (whole lines per move: a
// ring of 32-deep stages, half a line per row and move, measured 60.9 against
// 45.4 us at 128 x 6144 x 4096 bf16 NN).  B: fp8 NT three blocks of 64 k (128
// rows x 64 B); bf16 NT four phases of 32 k (128 rows x 64 B); bf16 NN four
// phases (two column halves of 32 k rows x 128 B, read transposed with
// ds_read_b64_tr_b16).  72 / 80 KiB.
// 16-byte chunks are XOR-swizzled by row (A and B^T as in gemm.hip; an NN
// row's chunk c sits at c ^ 4 ((k >> 1) & 1): the four k rows of a transpose
// read cover distinct banks).
// One barrier per block (fp8) or phase: after it every wave's moves of the
// data read next have landed and every wave's reads of the slot refilled next
// are done.
//
// KH (the form taken when at most 256 workgroups run, one per CU): eight waves,
// the two groups of four computing alternate 32 k of every 64-k block of rings
// twice as deep, their sums added through LDS at the end.  One wave per SIMD
// leaves its matrix pipe idle while it issues moves and fragment reads (the
// four-wave form takes 0.55 us a block at one workgroup per CU, 2.3 times its
// MFMA time, whatever the ring depth); two waves overlap: fp8 NT, K 4096, 1000
// x 4096 43.0 -> 36.9 us, K 14336, 128 x 4096 126 -> 102.  With two workgroups
// per CU the four-wave form is the faster one (2000 x 4096 65 against 73).
//
// Few rows (_kh64, _kh32; the first also for more rows while its tiles are at
// most one per CU: 170 x 6144 x 4096 fp8 38 -> 28 us): the same eight
// waves over 64 or 32 rows (2 or 1 MFMA row tiles per wave).  24 rows padded to
// 128 leave the matrix pipes, not the weight stream, as the bound (0.55 us a
// block, 15 KB/us a CU); the smaller tile and the deeper ring its A stage
// leaves room for (nine 64-k blocks fp8, six bf16) put the stream back.
//
// K ranges (grid y, *_splitk): fp32 partial planes for the reduction of
// gemv.hip.
#include "gemm_common.h"

typedef __attribute__((address_space(3))) uint8_t lds_b;

// MI: MFMA row tiles per wave; 4 (128 rows), with KH also 2 and 1
template <bool NT, bool FP8, bool SWIGLU, typename TC, bool ROPE, bool KH, int MI = 4>
__device__ __forceinline__ void gemm128_body(const GemmArgs &a) {
  static_assert(NT || !FP8, "no fp8 NN form");
  static_assert(MI == 4 || (KH && (MI == 2 || MI == 1)), "few-row tiles take the eight-wave form");
  // (RING must hold the 64 KiB the KH groups exchange)
  static_assert(!ROPE || (!SWIGLU && sizeof(TC) == 2), "the rotary epilogue writes bf16 projections");
  constexpr int NW = KH ? 8 : 4;              // waves
  // A ring: blocks of 64 k (32-row tiles stage 64 rows, a move per wave)
  constexpr int SA = MI == 4 ? 16384 : 8192;
  constexpr int RA = KH ? (MI == 4 ? (FP8 ? 6 : 4) : (FP8 ? 9 : 6)) : 3;
  // B ring: blocks of 64 k (fp8, KH), else phases of 32 k
  constexpr int RB = KH || FP8 ? RA : 4, SB = KH && !FP8 ? 16384 : 8192;
  constexpr int NAM = SA / 1024 / NW, NBM = SB / 1024 / NW;  // 1 KiB moves per wave: A block, B block / phase
  // KH, bf16 NT: B^T rows of 128 B, as A's
  constexpr bool BL = KH && NT && !FP8;

  int tm, tn;
  gemm_tile(a, tm, tn);
  const int64_t m0 = (int64_t)tm * (32 * MI);
  const int64_t n0 = (int64_t)tn * (SWIGLU ? 64 : 128);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = KH ? wave >> 2 : 0;  // KH: the half of each block this wave computes
  const int wm = (wave >> 1) & 1, wn = wave & 1;
  const int l16 = lane & 15, g4 = lane >> 4;

  f32x4 acc[MI][4];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  const int64_t brows = NT ? a.N : a.K;
  const i32x4_t ra = rsrc_words(a.A, a.M * a.lda * 2);
  const i32x4_t rb0 = rsrc_words(a.B0, brows * a.ldb * (FP8 ? 1 : 2));
  const i32x4_t rb1 = rsrc_words(SWIGLU ? a.B1 : a.B0, brows * a.ldb * (FP8 ? 1 : 2));

  // DMA sources.  Rows past M (A), past N (NT B) and k rows past K (NN B) lie
  // past the resource's end and read zeros; chunks past K (A, NT B) or past N
  // (NN B) are sent out of range.
  // A: move j: rows 8 (NW j + wave) + l / 8, slot l % 8; the slot's logical
  // chunk is the same for every j.
  const int ac = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
  const uint32_t abase = (uint32_t)(((m0 + 8 * wave + (lane >> 3)) * a.lda + ac * 8) * 2);
  const uint32_t astr = (uint32_t)(8 * NW * a.lda * 2);
  // B: tile half 0 and half 1 (64 B^T rows, or 64 columns) of the lane's row
  // NT: rows of 64 B, 16 per move: 4 waves cover a half (KH, fp8: wave / 4 is
  // the half), rows of 128 B (BL), 8 per move: 8 waves cover a half.  NN: move
  // j is half j, wave w its k rows 8 w + l / 8.
  const int bc = BL ? ac : NT ? (lane & 3) ^ ((lane >> 4) & 3) : (lane & 7) ^ (((lane >> 4) & 1) << 2);
  constexpr int BCK = FP8 ? 16 : 8;  // k per 16-byte chunk of an NT row
  uint32_t b0v, b1v;
  if constexpr (NT) {
    const int64_t r0 = n0 + (BL ? 8 * wave + (lane >> 3) : 16 * (wave & 3) + (lane >> 2));
    b0v = (uint32_t)(FP8 ? r0 * a.ldb + bc * 16 : (r0 * a.ldb + bc * 8) * 2);
    b1v = SWIGLU ? b0v : b0v + (uint32_t)(64 * a.ldb * (FP8 ? 1 : 2));
  } else {
    const int64_t c0 = n0 + bc * 8, c1 = SWIGLU ? c0 : c0 + 64;
    const int64_t kr = 8 * wave + (lane >> 3);
    b0v = c0 < a.N ? (uint32_t)((kr * a.ldb + c0) * 2) : OOB;
    b1v = c1 < a.N ? (uint32_t)((kr * a.ldb + c1) * 2) : OOB;
  }

  __shared__ __attribute__((aligned(1024))) uint8_t RING[RA * SA + RB * SB];
  const uint32_t ringa = lds_addr(RING), ringb = ringa + RA * SA;
  // (k past the end: zeros, no memory read)
  auto issue_a = [&](int st, int64_t k0) __attribute__((always_inline)) {
    const uint32_t la = ringa + st * SA;
    const uint32_t va = k0 + ac * 8 < a.K ? abase : OOB;
#pragma unroll
    for (int j = 0; j < NAM; ++j) dma16_asm_so(ra, la + (NW * j + wave) * 1024, va, j * astr + (uint32_t)k0 * 2);
  };
  auto issue_b = [&](int st, int64_t k0) __attribute__((always_inline)) {
    const uint32_t lb = ringb + st * SB;
    if constexpr (NT) {
      const bool kin = k0 + bc * BCK < a.K;
      const uint32_t ko = (uint32_t)k0 * (FP8 ? 1 : 2);
      if constexpr (KH && FP8) {
        dma16_asm_so(kg ? rb1 : rb0, lb + wave * 1024, kin ? (kg ? b1v : b0v) : OOB, ko);
      } else {
        dma16_asm_so(rb0, lb + wave * 1024, kin ? b0v : OOB, ko);
        dma16_asm_so(rb1, lb + (NW + wave) * 1024, kin ? b1v : OOB, ko);
      }
    } else {
      // (32 k rows of a half: 4 KiB; KH: the block's second 32 k follow both halves)
      const uint32_t ko = (uint32_t)k0 * (uint32_t)(a.ldb * 2);
      const uint32_t lw = lb + (wave & 3) * 1024 + kg * 8192;
      dma16_asm_so(rb0, lw, b0v, ko);
      dma16_asm_so(rb1, lw + 4096, b1v, ko);
    }
  };

  // Fragment offsets within a stage.  A tile i: rows 16 MI wm + 16 i + l16; B
  // tile j: tile columns 32 wn + brel[j] + l16 (half j / 2).  The row swizzles
  // only see l16.  A block's second 32 k: A chunk 4 + g (offset bit 6), fp8 B
  // chunk 2 + g / 2 (offset bit 5).
  constexpr int brel[4] = {0, 16, 64, 80};
  const uint32_t aoff = ((16 * MI * wm + l16) * 128 + ((g4 ^ swz_a64(l16)) << 4)) ^ (kg ? 64u : 0u);
  uint32_t boff;  // tile 0
  if constexpr (FP8) {
    boff = ((32 * wn + l16) * 64 + (((g4 >> 1) ^ swz_b64(l16)) << 4) + 8 * (g4 & 1)) ^ (kg ? 32u : 0u);
  } else if constexpr (BL) {
    boff = ((32 * wn + l16) * 128 + ((g4 ^ swz_a64(l16)) << 4)) ^ (kg ? 64u : 0u);
  } else if constexpr (NT) {
    boff = (32 * wn + l16) * 64 + ((g4 ^ hswz(l16)) << 4);
  } else {
    // lane (g, i): k rows 8 g + 4 s + i / 4, columns c + 4 (i % 4) of the
    // half; the column's chunk is 4 wn + 2 (j % 2) + (i % 4) / 2, so tiles 0
    // and 1 differ in chunk bit 1 (offset bit 5)
    boff = (8 * g4 + (l16 >> 2)) * 128 + (((4 * wn + ((l16 & 3) >> 1)) ^ (((l16 >> 3) & 1) << 2)) << 4) +
           (l16 & 1) * 8 + kg * 8192;
  }

  typedef __attribute__((address_space(3))) const uint8_t lds_u8;
  typedef __attribute__((address_space(3))) const bf16x8_t lds_bf16x8;
  typedef __attribute__((address_space(3))) const unsigned long long lds_u64;
  // fragments of the 32 k of half h of an A block and its B (fp8: the same
  // half of the B block)
  auto load = [&](lds_u8 *sta, lds_u8 *stb, int h, bf16x8_t (&af)[MI], bf16x8_t (&bf)[4])
      __attribute__((always_inline)) {
    lds_u8 *pa = sta + (h ? aoff ^ 64u : aoff);
    lds_u8 *pb = stb + (FP8 && h ? boff ^ 32u : boff);
#pragma unroll
    for (int i = 0; i < MI; ++i) af[i] = *reinterpret_cast<lds_bf16x8 *>(pa + i * 2048);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (FP8) {
        const unsigned long long q = *reinterpret_cast<lds_u64 *>(pb + brel[j] * 64);
        const uint4 w = e4m3x8_to_bf16x8(make_uint2((uint32_t)q, (uint32_t)(q >> 32)));
        bf[j] = *reinterpret_cast<const bf16x8_t *>(&w);
      } else if constexpr (NT) {
        bf[j] = *reinterpret_cast<lds_bf16x8 *>(pb + brel[j] * (BL ? 128 : 64));
      } else {
        lds_u8 *pj = stb + (j >> 1) * 4096 + ((j & 1) ? boff ^ 32u : boff);
        s16x4 v[2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
          v[s] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(pj + s * 512));
        bf[j] = __builtin_shufflevector(__builtin_bit_cast(__attribute__((ext_vector_type(4))) __bf16, v[0]),
                                        __builtin_bit_cast(__attribute__((ext_vector_type(4))) __bf16, v[1]),
                                        0, 1, 2, 3, 4, 5, 6, 7);
      }
    }
  };
  // C^T tiles (B fragment as the A operand): lane (g, i) of tile (i', j) holds
  // output row 16 i' + i and columns (tile column) + 4 g + 0..3
  auto mma = [&](const bf16x8_t (&af)[MI], const bf16x8_t (&bf)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j], af[i], acc[i][j], 0, 0, 0);
  };

  // "at most N moves outstanding, every LDS read in registers", then the barrier
  auto sync = [&](auto ntag) __attribute__((always_inline)) {
    constexpr int N = decltype(ntag)::value;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
    barrier_no_fence();
  };
  const int nblk = (int)((a.K + 63) / 64);
  lds_u8 *const RA0 = (lds_u8 *)RING, *const RB0 = RA0 + RA * SA;
  // Phases of 32 k, q = 2 t + h (half h of block t).  Phase q reads the
  // fragments of phase q + 1 from LDS while its own, read a phase earlier, feed
  // the MFMAs.
  bf16x8_t af[2][MI], bf[2][4];
  int sa = 0;  // ring slot of block t (fp8: of its B block too)
  auto next = [](int s) __attribute__((always_inline)) { return s == RA - 1 ? 0 : s + 1; };
  if constexpr (KH) {
    // the two groups of four waves take alternate 32 k of every block; block
    // t + 1's fragments are read while block t's feed the MFMAs, and block t +
    // RA moves into the slot whose fragments are in registers.  A SwiGLU pair over NT weights: tile column tn starts at its own place
    // in K and wraps around.  Its tiles run one K loop each in step, and rows a
    // power of two apart at the same k sit on the same memory channels (24 rows
    // of 2 x 14336 x 4096 fp8: 31.0 us in step, 28.4 spread; with K ranges, which
    // spread by themselves, 3% slower).
    const int rot = NT && SWIGLU ? (int)((int64_t)tn * nblk / a.tiles_n) : 0;
    auto issue = [&](int t, int st) __attribute__((always_inline)) {
      const int u = NT && SWIGLU && t < nblk ? (t + rot < nblk ? t + rot : t + rot - nblk) : t;
      issue_a(st, (int64_t)u * 64);
      issue_b(st, (int64_t)u * 64);
    };
#pragma unroll
    for (int t = 0; t < RA; ++t) issue(t, t);
    sync(Int<(RA - 1) * (NAM + NBM)>{});
    load(RA0, RB0, 0, af[0], bf[0]);
    auto step = [&](int t, int c) __attribute__((always_inline)) {
      sync(Int<(RA - 2) * (NAM + NBM)>{});  // block t + 1 landed
      issue(t + RA, sa);
      sa = next(sa);
      lds_u8 *pa = RA0 + sa * SA, *pb = RB0 + sa * SB;
      asm volatile("" : "+s"(pa), "+s"(pb));
      load(pa, pb, 0, af[1 - c], bf[1 - c]);  // (past the last block: never used)
      mma(af[c], bf[c]);
    };
    for (int t = 0; t < nblk; t += 2) {
      step(t, 0);
      if (t + 1 < nblk) step(t + 1, 1);
    }
  } else if constexpr (FP8) {
    // in issue order: A0 B0 A1 B1 .., then per block, once its fragments are
    // in registers, A(t + RA) B(t + RA) into its slot
#pragma unroll
    for (int t = 0; t < RA; ++t) {
      issue_a(t, t * 64);
      issue_b(t, t * 64);
    }
    sync(Int<(RA - 1) * (NAM + NBM)>{});
    load(RA0, RB0, 0, af[0], bf[0]);
    for (int t = 0; t < nblk; ++t) {
      lds_u8 *pa = RA0 + sa * SA, *pb = RB0 + sa * SB;
      asm volatile("" : "+s"(pa), "+s"(pb));
      load(pa, pb, 1, af[1], bf[1]);
      mma(af[0], bf[0]);
      sync(Int<(RA - 2) * (NAM + NBM)>{});  // block t + 1 landed
      issue_a(sa, (int64_t)(t + RA) * 64);
      issue_b(sa, (int64_t)(t + RA) * 64);
      sa = next(sa);
      pa = RA0 + sa * SA;
      pb = RB0 + sa * SB;
      asm volatile("" : "+s"(pa), "+s"(pb));
      load(pa, pb, 0, af[0], bf[0]);  // (past the last block: never used)
      mma(af[1], bf[1]);
    }
  } else {
    // in issue order: A0 B0, then A(u) right before B(2 u - 1), through
    // B(RB - 1); then in phase q (h = 1: A(t + RA)) B(q + RB), into the slots
    // whose fragments are in registers, which continues that order.  Phase q
    // needs B(q + 1) and A((q + 1) / 2) landed: B(q + 2) .. B(q + RB - 1) and
    // the RA - 2 blocks of A among them may be outstanding.
    issue_a(0, 0);
#pragma unroll
    for (int q = 0; q < RB; ++q) {
      if (q & 1) issue_a((q + 1) / 2, (q + 1) / 2 * 64);
      issue_b(q, q * 32);
    }
    sync(Int<(RA - 1) * NAM + (RB - 1) * NBM>{});
    load(RA0, RB0, 0, af[0], bf[0]);
    int sb = 0;  // B slot of phase 2 t
    for (int t = 0; t < nblk; ++t) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        sync(Int<(RA - 2) * NAM + (RB - 2) * NBM>{});
        if (h == 1) {
          issue_a(sa, (int64_t)(t + RA) * 64);
          sa = next(sa);
        }
        issue_b(sb + h, (int64_t)t * 64 + (h + RB) * 32);
        if (h == 1) sb = sb == RB - 2 ? 0 : sb + 2;
        lds_u8 *pa = RA0 + sa * SA, *pb = RB0 + (h == 1 ? sb : sb + 1) * SB;
        asm volatile("" : "+s"(pa), "+s"(pb));
        load(pa, pb, 1 - h, af[1 - h], bf[1 - h]);  // (past the last phase: never used)
        mma(af[h], bf[h]);
      }
    }
  }
  wait_vmem();  // no LDS DMA outlives the workgroup
  // KH: the groups add their halves' sums through the (idle) ring, group g
  // keeping the g-th half of the A tiles (one tile: group 0 keeps it)
  constexpr int NI = KH && MI > 1 ? MI / 2 : MI;
  f32x4 out[NI][4];
  if constexpr (KH) {
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    sync(Int<0>{});
    lds_f32x4 *X = (lds_f32x4 *)RING + (threadIdx.x & 255);
    constexpr int HI = MI > 1 ? NI : 0;  // first tile of group 1
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) X[((kg * NI + i) * 4 + j) * 256] = kg ? acc[i][j] : acc[HI + i][j];
    sync(Int<0>{});
    if (MI == 1 && kg) return;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 o = X[(((1 - kg) * NI + i) * 4 + j) * 256];
#pragma unroll
        for (int e = 0; e < 4; ++e) out[i][j][e] = (kg ? acc[HI + i][j][e] : acc[i][j][e]) + o[e];
      }
  } else {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) out[i][j] = acc[i][j];
  }

  // ---- epilogue: rows 16 MI wm + 16 i + l16, columns 32 wn + brel[j] + 4 g ..
  const bool vec = (a.flags & GEMM_VEC) != 0;
  const int64_t rbase = m0 + 16 * MI * wm + (MI > 1 ? 8 * MI * kg : 0) + l16;
  auto put4 = [&](int64_t row, int64_t col, const float (&v)[4]) __attribute__((always_inline)) {
    if (vec && col + 3 < a.N) {
      OutT<TC>::store4(a.C, row * a.ldc + col, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < a.N) OutT<TC>::store(a.C, row * a.ldc + col + e, v[e]);
    }
  };
  if constexpr (SWIGLU) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t col = n0 + 32 * wn + 16 * j + 4 * g4;
      if (col >= a.N) continue;
      float sg[4], su[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = (a.flags & GEMM_SCALE) && col + e < a.N;
        sg[e] = in ? a.scale0[col + e] : 1.f;
        su[e] = in ? a.scale1[col + e] : 1.f;
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int64_t row = rbase + 16 * i;
        if (row >= a.M) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = out[i][j][e] * sg[e], u = out[i][j + 2][e] * su[e];
          // silu(g) = g / (1 + exp(-g)) from the hardware 2^x and reciprocal
          const float ex = __builtin_amdgcn_exp2f(g * -1.44269504088896341f);
          v[e] = g * __builtin_amdgcn_rcpf(1.0f + ex) * u;
        }
        put4(row, col, v);
      }
    }
    return;
  }
  if constexpr (ROPE) {
    if (n0 < (int64_t)a.rope_nq + a.rope_nk) {
      // the tile is one head: lane holds frequencies d of both halves (tiles
      // j and j + 2); the arithmetic of gemm.hip's rotary epilogue
      const bool isq = n0 < a.rope_nq;
      uint16_t *dst = reinterpret_cast<uint16_t *>(isq ? a.rope_q : a.rope_k);
      const int64_t ldd = isq ? a.rope_nq : a.rope_nk, c0 = isq ? n0 : n0 - a.rope_nq;
      const bool scaled = (a.flags & GEMM_SCALE) != 0;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int d = 32 * wn + 16 * j + 4 * g4;
        float s0[4], s1[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s0[e] = scaled ? a.scale0[n0 + d + e] : 1.f;
          s1[e] = scaled ? a.scale0[n0 + 64 + d + e] : 1.f;
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int64_t row = rbase + 16 * i;
          if (row >= a.M) continue;
          const int64_t to = (int64_t)((int32_t)row % a.rope_seq) * a.rope_ts + d;
          const float4 c = *reinterpret_cast<const float4 *>(a.rope_cos + to);
          const float4 s = *reinterpret_cast<const float4 *>(a.rope_sin + to);
          const float cv[4] = {c.x, c.y, c.z, c.w}, sv[4] = {s.x, s.y, s.z, s.w};
          float y0[4], y1[4];
          {
#pragma clang fp contract(off)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float x0 = bf16_to_f32(f32_to_bf16(out[i][j][e] * s0[e]));
              const float x1 = bf16_to_f32(f32_to_bf16(out[i][j + 2][e] * s1[e]));
              y0[e] = x0 * cv[e] - x1 * sv[e];
              y1[e] = x0 * sv[e] + x1 * cv[e];
            }
          }
          OutT<bf16>::store4(dst, row * ldd + c0 + d, y0);
          OutT<bf16>::store4(dst, row * ldd + c0 + 64 + d, y1);
        }
      }
      return;
    }
  }
  // loads of a tile column (its factors, the residual's elements this lane
  // then writes) before its stores: C may be the residual buffer
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t col = n0 + 32 * wn + brel[j] + 4 * g4;
    if (col >= a.N) continue;
    float sc[4], bi[4], r4[NI][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = col + e < a.N;
      sc[e] = ((a.flags & GEMM_SCALE) && in) ? a.scale0[col + e] : 1.f;
      bi[e] = ((a.flags & GEMM_BIAS) && in) ? bf16_to_f32(reinterpret_cast<const uint16_t *>(a.bias)[col + e]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int64_t row = rbase + 16 * i;
#pragma unroll
      for (int e = 0; e < 4; ++e) r4[i][e] = 0.f;
      if (!(a.flags & GEMM_RESID) || row >= a.M) continue;
      if (vec && col + 3 < a.N) {
        OutT<TC>::load4(a.resid, row * a.ldc + col, r4[i]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < a.N) r4[i][e] = OutT<TC>::load(a.resid, row * a.ldc + col + e);
      }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int64_t row = rbase + 16 * i;
      if (row >= a.M) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = epilogue(a.flags, out[i][j][e] * sc[e], bi[e], r4[i][e]);
      put4(row, col, v);
    }
  }
}

// each with four waves (two workgroups per CU) and with eight (_kh; _kh64 and
// _kh32 for at most 64 and 32 rows)
#define NK_GEMM128(NT, FP8, SW, TC, ROPE, name)                                    \
  extern "C" __global__ __launch_bounds__(256, 2) void name(GemmArgs a) {          \
    gemm128_body<NT, FP8, SW, TC, ROPE, false>(a);                                 \
  }                                                                                \
  extern "C" __global__ __launch_bounds__(512, 1) void name##_kh(GemmArgs a) {   \
    gemm128_body<NT, FP8, SW, TC, ROPE, true>(a);                                  \
  }                                                                                \
  extern "C" __global__ __launch_bounds__(512, 1) void name##_kh64(GemmArgs a) {   \
    gemm128_body<NT, FP8, SW, TC, ROPE, true, 2>(a);                               \
  }                                                                                \
  extern "C" __global__ __launch_bounds__(512, 1) void name##_kh32(GemmArgs a) {   \
    gemm128_body<NT, FP8, SW, TC, ROPE, true, 1>(a);                               \
  }
NK_GEMM128(false, false, false, bf16, false, nk_gemm128_nn_bf16_bf16)
NK_GEMM128(false, false, false, float, false, nk_gemm128_nn_bf16_f32)
NK_GEMM128(false, false, true, bf16, false, nk_gemm128_swiglu_nn_bf16_bf16)
NK_GEMM128(false, false, false, bf16, true, nk_gemm128_nn_bf16_bf16_rope)
NK_GEMM128(true, false, false, bf16, false, nk_gemm128_nt_bf16_bf16)
NK_GEMM128(true, false, false, float, false, nk_gemm128_nt_bf16_f32)
NK_GEMM128(true, false, true, bf16, false, nk_gemm128_swiglu_nt_bf16_bf16)
NK_GEMM128(true, false, false, bf16, true, nk_gemm128_nt_bf16_bf16_rope)
NK_GEMM128(true, true, false, bf16, false, nk_gemm128_nt_e4m3_bf16)
NK_GEMM128(true, true, false, float, false, nk_gemm128_nt_e4m3_f32)
NK_GEMM128(true, true, true, bf16, false, nk_gemm128_swiglu_nt_e4m3_bf16)
NK_GEMM128(true, true, false, bf16, true, nk_gemm128_nt_e4m3_bf16_rope)

// K-range entries: workgroup (tile, s) computes the tile's fp32 partial sum
// over K range s, handed the range as its operands: A and B advanced to the
// range's first k, K = the range's length, C = the range's partial plane
// (flags: at most GEMM_VEC, so the epilogue stores the plain sums).  The
// buffer ranges then end where the range ends (rows of NN B, columns of A and
// NT B past it read zeros, as at a real K end), and the ranges' planes are
// added in order by the reduction kernel of gemv.hip, which applies the
// epilogue.
template <bool NT, int BSZ>
__device__ __forceinline__ GemmArgs splitk_args(const GemmArgs &a) {
  GemmArgs s = a;
  const int64_t k0 = (int64_t)blockIdx.y * a.kc;
  s.K = min((int64_t)a.kc, a.K - k0);
  s.A = reinterpret_cast<const uint16_t *>(a.A) + k0;
  s.B0 = reinterpret_cast<const uint8_t *>(a.B0) + (NT ? k0 * BSZ : k0 * a.ldb * BSZ);
  s.C = reinterpret_cast<float *>(a.C) + (int64_t)blockIdx.y * a.M * a.ldc;
  return s;
}

// (the eight-wave forms under the 8-wave kernels' names: for at most 64 rows
// without a suffix)
#define NK_GEMM128_SPLITK(NT, FP8, tag)                                                              \
  extern "C" __global__ __launch_bounds__(256, 2) void nk_gemm128_##tag##_f32_splitk(GemmArgs a) {   \
    gemm128_body<NT, FP8, false, float, false, false>(splitk_args<NT, FP8 ? 1 : 2>(a));              \
  }                                                                                                  \
  extern "C" __global__ __launch_bounds__(512, 1) void nk_gemm8k_##tag##_f32_splitk128(GemmArgs a) {  \
    gemm128_body<NT, FP8, false, float, false, true>(splitk_args<NT, FP8 ? 1 : 2>(a));               \
  }                                                                                                 \
  extern "C" __global__ __launch_bounds__(512, 1) void nk_gemm8k_##tag##_f32_splitk(GemmArgs a) {     \
    gemm128_body<NT, FP8, false, float, false, true, 2>(splitk_args<NT, FP8 ? 1 : 2>(a));            \
  }                                                                                                 \
  extern "C" __global__ __launch_bounds__(512, 1) void nk_gemm8k_##tag##_f32_splitk32(GemmArgs a) {   \
    gemm128_body<NT, FP8, false, float, false, true, 1>(splitk_args<NT, FP8 ? 1 : 2>(a));            \
  }
NK_GEMM128_SPLITK(false, false, nn_bf16)
NK_GEMM128_SPLITK(true, false, nt_bf16)
NK_GEMM128_SPLITK(true, true, nt_e4m3)
