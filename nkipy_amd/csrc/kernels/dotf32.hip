// Batched product of strided float operands in fp32 on the matrix cores:
// C[b, m, n] = sum_k A[b, m, k] B[b, k, n], fp32 multiply-adds
// (v_mfma_f32_16x16x4_f32), C contiguous.
//
// The fallback product of a NumPy kernel's fp32 arrays (the fused GEMM
// kernels take bf16 and fp8), so operands come through arbitrary strides as
// fp32, fp16 or bf16, widened exactly on the way into LDS.  Bound by the
// matrix cores' fp32 rate for large products, by latency for small ones: the
// one-output-per-thread kernel (nk_dot) ran 200 x 6144 x 1024 at 12 TFLOP/s
// (208 us) on the vector units, 38 us here with its reduction; 1024 x 4096 x
// 4096 reaches 131 TFLOP/s of the 153 a large library product does.
//
// 256 threads = 4 waves (2 x 2) on a 64 x 64 tile, each wave 32 x 32 as 2 x 2
// MFMA tiles; K in stages of 32, two LDS buffers per operand (36 KiB: four
// workgroups per CU).  A lane reads four
// consecutive k of its row (16 bytes) for four MFMAs: instruction s takes k =
// 4 g + s of a 16-k group in both operands, a permutation of the 16 the sum
// does not see.  The next stage's global loads are issued before the current
// stage's products.  Load modes per operand, chosen by the host: 4 elements at
// a time along k (1) or along rows / columns (2) where strides, sizes and
// alignment allow, else element by element (0); one kernel per pair of modes
// and element widths (nk_dot_f32_<f|h><mode A>_<f|h><mode B>).
// fp32 pairs also come over 32 x 128 tiles (the four waves side by side; 46 KiB:
// three workgroups per CU) for up to 32 rows, which 64-row tiles pad to twice
// the matrix work: one row of a feed-forward of 2048 / 6144 78 -> 63 us.
// K ranges (grid z = batch x ksplit) write fp32 planes [range][batch m][n] for
// the reduction of gemv.hip when the tiles leave CUs idle.
#include "common.h"

using namespace nk;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct DotF32Args {
  const void *A;
  const void *B;
  void *C;
  int64_t batch, M, N, K;
  int64_t sab, sam, sak;  // A strides (elements)
  int64_t sbb, sbk, sbn;  // B strides
  int32_t a_dtype, b_dtype, c_dtype;  // 0 fp32, 1 fp16, 2 bf16
  int32_t a_mode, b_mode;
  int32_t ksplit, kc;     // K ranges of kc (a multiple of 32); ksplit 1: C direct
  int32_t c_vec;          // fp32 C: rows take aligned 16-byte stores
  int32_t a_bytes, b_bytes;  // one batch's span of each operand (< 2 GiB)
};

constexpr int KS = 32;
// LDS layouts: modes 0 and 1 [rows][32 k + 4], mode 2 as it lies in memory,
// [32 k][rows + 4]: 16-byte writes, and both kinds of read (16 rows x 16
// bytes, 16 rows x four k) spread over all banks
constexpr int PITCH = KS + 4;
constexpr uint32_t FAR = 0x80000000u;  // past every operand (each spans less than 2 GiB): reads zeros

// One operand's stage (R rows x 32 k): this thread's R / 32 4-element pieces as
// raw words.  MODE 1: row t / 8 + 32 u, k 4 (t % 8); MODE 2 (64 rows): k t / 16
// + 16 u, rows 4 (t % 16); MODE 0: as MODE 1, element by element.  HALF: 16-bit
// elements.  Loads go through a buffer resource with out-of-range pieces sent
// past its end, so no load sits behind a branch and all stay in flight until
// the pieces are widened on their way into LDS.
template <int MODE, bool HALF, int ROWS>
struct Operand {
  static constexpr int ES = HALF ? 2 : 4;
  static constexpr int U = ROWS / 32, R4 = ROWS / 4, KSTEP = 256 / R4, KPITCH = ROWS + 4;
  static constexpr int WORDS = ROWS * PITCH > KS * KPITCH ? ROWS * PITCH : KS * KPITCH;
  __amdgpu_buffer_rsrc_t r;
  uint32_t off[U], kstep, estep;
  int kofs[U], dt;
  uint32_t w[U][4];

  __device__ __forceinline__ void init(const void *p, int64_t bytes, int dtype, int64_t r0, int64_t R, int64_t sr,
                                       int64_t sk) {
    const int t = threadIdx.x;
    r = buf_rsrc(p, (uint32_t)bytes);
    dt = dtype;
    kstep = (uint32_t)(sk * ES);
    estep = (uint32_t)((MODE == 2 ? sr : sk) * ES);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = r0 + (MODE == 2 ? 4 * (t % R4) : (t >> 3) + 32 * u);
      kofs[u] = MODE == 2 ? t / R4 + KSTEP * u : 4 * (t & 7);
      off[u] = row < R ? (uint32_t)((row * sr + kofs[u] * sk) * ES) : FAR;
    }
  }
  // k0: first k of the stage, k1: end of the range
  __device__ __forceinline__ void fetch(int64_t k0, int64_t k1) {
    const uint32_t so = __builtin_amdgcn_readfirstlane((uint32_t)k0 * kstep);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (MODE == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t o = k0 + kofs[u] + e < k1 ? off[u] + e * estep : FAR;
          w[u][e] = HALF ? __builtin_amdgcn_raw_buffer_load_b16(r, o, so, 0)
                         : __builtin_amdgcn_raw_buffer_load_b32(r, o, so, 0);
        }
      } else {
        const uint32_t o = k0 + kofs[u] < k1 ? off[u] : FAR;
        if constexpr (HALF) {
          const nk_u32x2 q = __builtin_amdgcn_raw_buffer_load_b64(r, o, so, 0);
          w[u][0] = q[0];
          w[u][1] = q[1];
        } else {
          const nk_u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(r, o, so, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[u][e] = q[e];
        }
      }
    }
  }
  __device__ __forceinline__ void put(float *S) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      f32x4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (HALF) {
          const uint32_t h = MODE == 0 ? w[u][e] & 0xffffu : (e & 1) ? w[u][e >> 1] >> 16 : w[u][e >> 1] & 0xffffu;
          v[e] = dt == 2 ? __uint_as_float(h << 16) : f16_to_f32((uint16_t)h);
        } else {
          v[e] = __uint_as_float(w[u][e]);
        }
      }
      if constexpr (MODE == 2) {
        *reinterpret_cast<f32x4_t *>(S + (t / R4 + KSTEP * u) * KPITCH + 4 * (t % R4)) = v;
      } else {
        *reinterpret_cast<f32x4_t *>(S + ((t >> 3) + 32 * u) * PITCH + 4 * (t & 7)) = v;
      }
    }
  }
  // four k (16 h + 4 g + 0..3) of a row of the staged operand
  __device__ __forceinline__ f32x4_t frag(const float *S, int row, int h, int g) const {
    if constexpr (MODE == 2) {
      f32x4_t v;
#pragma unroll
      for (int s = 0; s < 4; ++s) v[s] = S[(16 * h + 4 * g + s) * KPITCH + row];
      return v;
    } else {
      return *reinterpret_cast<const f32x4_t *>(S + row * PITCH + 16 * h + 4 * g);
    }
  }
};

// TM x TN: 64 x 64 (waves 2 x 2) or 32 x 128 (waves 1 x 4)
template <int MA, bool HA, int MB, bool HB, int TM, int TN>
__device__ __forceinline__ void dot_f32_body(const DotF32Args &a) {
  using OpA = Operand<MA, HA, TM>;
  using OpB = Operand<MB, HB, TN>;
  __shared__ __attribute__((aligned(16))) float SA[2][OpA::WORDS], SB[2][OpB::WORDS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int WN = TN / 32;
  const int wm = wave / WN, wn = wave % WN, l16 = lane & 15, g = lane >> 4;
  const int64_t b = blockIdx.z / (uint32_t)a.ksplit;
  const int sp = blockIdx.z % (uint32_t)a.ksplit;
  const int64_t m0 = (int64_t)blockIdx.y * TM, n0 = (int64_t)blockIdx.x * TN;
  const int64_t k0 = (int64_t)sp * a.kc, k1 = min(k0 + a.kc, a.K);
  OpA oa;
  OpB ob;
  oa.init((const uint8_t *)a.A + b * a.sab * oa.ES, a.a_bytes, a.a_dtype, m0, a.M, a.sam, a.sak);
  ob.init((const uint8_t *)a.B + b * a.sbb * ob.ES, a.b_bytes, a.b_dtype, n0, a.N, a.sbn, a.sbk);

  f32x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f;

  oa.fetch(k0, k1);
  ob.fetch(k0, k1);
  int cur = 0;
  for (int64_t k = k0; k < k1; k += KS, cur ^= 1) {
    // (the buffer written here was last read before the previous barrier)
    oa.put(SA[cur]);
    ob.put(SB[cur]);
    lds_barrier();  // (leaves the loads issued next in flight)
    oa.fetch(k + KS, k1);  // (past the range: zeros)
    ob.fetch(k + KS, k1);
#pragma unroll
    for (int h = 0; h < KS / 16; ++h) {
      f32x4_t af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        af[i] = oa.frag(SA[cur], 32 * wm + 16 * i + l16, h, g);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bf[j] = ob.frag(SB[cur], 32 * wn + 16 * j + l16, h, g);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][s], af[i][s], acc[i][j], 0, 0, 0);
    }
  }
  // lane: row 16 i + l16, columns 16 j + 4 g + 0..3
  const int64_t plane = a.batch * a.M * a.N;
  float *part = (float *)a.C + sp * plane;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t m = m0 + 32 * wm + 16 * i + l16;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t n = n0 + 32 * wn + 16 * j + 4 * g;
      const int64_t o = (b * a.M + m) * a.N + n;
      if (a.c_vec && n < a.N) {
        *reinterpret_cast<f32x4_t *>(part + o) = acc[i][j];
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= a.N) break;
        if (a.c_dtype == 0) part[o + e] = acc[i][j][e];
        else if (a.c_dtype == 1) ((uint16_t *)a.C)[o + e] = f32_to_f16(acc[i][j][e]);
        else ((uint16_t *)a.C)[o + e] = f32_to_bf16(acc[i][j][e]);
      }
    }
  }
}

#define NK_DOT(MA, ta, HA, MB, tb, HB)                                                               \
  extern "C" __global__ __launch_bounds__(256, 4) void nk_dot_f32_##ta##MA##_##tb##MB(DotF32Args a) { \
    dot_f32_body<MA, HA, MB, HB, 64, 64>(a);                                                              \
  }
#define NK_DOT_B(MA, ta, HA)                                                           \
  NK_DOT(MA, ta, HA, 0, f, false) NK_DOT(MA, ta, HA, 1, f, false) NK_DOT(MA, ta, HA, 2, f, false) \
  NK_DOT(MA, ta, HA, 0, h, true) NK_DOT(MA, ta, HA, 1, h, true) NK_DOT(MA, ta, HA, 2, h, true)
NK_DOT_B(0, f, false)
NK_DOT_B(1, f, false)
NK_DOT_B(2, f, false)
NK_DOT_B(0, h, true)
NK_DOT_B(1, h, true)
NK_DOT_B(2, h, true)
#define NK_DOT_WIDE(MA, MB)                                                                            \
  extern "C" __global__ __launch_bounds__(256, 3) void nk_dot_f32_f##MA##_f##MB##_wide(DotF32Args a) { \
    dot_f32_body<MA, false, MB, false, 32, 128>(a);                                                    \
  }
NK_DOT_WIDE(0, 0) NK_DOT_WIDE(0, 1) NK_DOT_WIDE(0, 2)
NK_DOT_WIDE(1, 0) NK_DOT_WIDE(1, 1) NK_DOT_WIDE(1, 2)
NK_DOT_WIDE(2, 0) NK_DOT_WIDE(2, 1) NK_DOT_WIDE(2, 2)
