// Shared by the MFMA GEMM kernels (gemm.hip, gemm128.hip): the argument
// struct and flags, epilogue arithmetic, output element access, LDS moves and
// waits and the XCD-aware tile walk.
#pragma once

#include "common.h"

using namespace nk;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Tile rows per group of the XCD-local walk.  Measured on MI355X (us, 8-wave
// kernel, GROUP_M 1 / 2 / 4 / 8): NT bf16 16384x6144x4096 731 / 709 / 685 /
// 771, NT fp8 same shape 692 / 694 / 668 / 730, NN 4096x4096x14336 353 /
// 352 / 351 / 358, fp8 SwiGLU 16384x14336x4096 unchanged.
#define GROUP_M 4

enum {
  GEMM_BIAS = 1,      // + bias[col] (bf16)
  GEMM_SCALE = 2,     // * scale[col] (fp32), per output column (fp8 weights)
  GEMM_RESID = 4,     // + residual[row][col] (same dtype as C)
  GEMM_VEC = 8,       // C / residual rows allow aligned 4-element vector access
  GEMM_RND_BIAS = 16, // round the (scaled) product to bf16 before the bias add
  GEMM_RND_RESID = 32,// round to bf16 before the residual add
  GEMM_ROWS16 = 64,   // bf16 C / residual rows take aligned 16-byte chunks (N, ldc
                      // multiples of 8) and a residual is added to a rounded value:
                      // the 8-wave kernels may stage the output tile through LDS
};
// The rounding flags keep the cast points of the traced NumPy code: e.g.
// ``z + (x @ w).astype(bf16)`` rounds the product before the add.

struct GemmArgs {
  const void *A;       // M x K
  const void *B0;      // NN: K x N ; NT: N x K
  const void *B1;      // swiglu: up weight (same layout as B0)
  void *C;             // M x N (swiglu: M x N_out)
  const void *bias;    // N, bf16
  const float *scale0; // N, fp32 (scales of B0 columns)
  const float *scale1; // N, fp32 (scales of B1 columns, swiglu)
  const void *resid;   // M x N, C dtype
  int64_t M, N, K;     // N = output columns
  int64_t lda, ldb, ldc;
  int32_t tiles_m, tiles_n;
  int32_t flags;
  int32_t group_m;     // tile rows per group of the tile walk; 0: GROUP_M
  // rotary embedding of the q / k columns (the *_rope kernels only)
  const float *rope_cos;  // fp32 [position][64], row stride rope_ts
  const float *rope_sin;
  void *rope_q;           // M x rope_nq bf16: rotated columns 0 .. rope_nq-1
  void *rope_k;           // M x rope_nk bf16: rotated columns rope_nq ..
  int64_t rope_ts;
  int32_t rope_seq;       // row m sits at position m % rope_seq
  int32_t rope_nq, rope_nk, rope_pad;
  // split-K entries (*_splitk): K ranges of kc (a multiple of 64), range
  // blockIdx.y; fp32 partial sums of range s at C + s * M * ldc
  int32_t ksplit, kc;
};

// ---------------------------------------------------------------------------
// element helpers
// ---------------------------------------------------------------------------
// fp8 -> bf16 staging uses nk::e4m3x8_to_bf16x8 (common.h)

// (product + bias) + residual with the optional bf16 roundings in between
__device__ __forceinline__ float epilogue(int flags, float prod, float bias, float resid) {
  if (flags & GEMM_RND_BIAS) prod = bf16_to_f32(f32_to_bf16(prod));
  float v = prod + bias;
  if (flags & GEMM_RND_RESID) v = bf16_to_f32(f32_to_bf16(v));
  return v + resid;
}

template <typename TC> struct OutT;
template <> struct OutT<bf16> {
  static __device__ __forceinline__ void store(void *C, int64_t i, float v) {
    reinterpret_cast<uint16_t *>(C)[i] = f32_to_bf16(v);
  }
  static __device__ __forceinline__ float load(const void *C, int64_t i) {
    return bf16_to_f32(reinterpret_cast<const uint16_t *>(C)[i]);
  }
  static __device__ __forceinline__ void store4(void *C, int64_t i, const float (&v)[4]) {
    *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(C) + i) =
        make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  }
  static __device__ __forceinline__ void load4(const void *C, int64_t i, float (&v)[4]) {
    const uint2 w = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(C) + i);
    v[0] = __uint_as_float(w.x << 16);
    v[1] = __uint_as_float(w.x & 0xffff0000u);
    v[2] = __uint_as_float(w.y << 16);
    v[3] = __uint_as_float(w.y & 0xffff0000u);
  }
};
template <> struct OutT<float> {
  static __device__ __forceinline__ void store(void *C, int64_t i, float v) {
    reinterpret_cast<float *>(C)[i] = v;
  }
  static __device__ __forceinline__ float load(const void *C, int64_t i) {
    return reinterpret_cast<const float *>(C)[i];
  }
  static __device__ __forceinline__ void store4(void *C, int64_t i, const float (&v)[4]) {
    *reinterpret_cast<float4 *>(reinterpret_cast<float *>(C) + i) = make_float4(v[0], v[1], v[2], v[3]);
  }
  static __device__ __forceinline__ void load4(const void *C, int64_t i, float (&v)[4]) {
    const float4 w = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(C) + i);
    v[0] = w.x;
    v[1] = w.y;
    v[2] = w.z;
    v[3] = w.w;
  }
};

// Operands are read through buffer resources: 32-bit offsets from one base
// (no per-load 64-bit addresses), and an offset past the end (OOB) reads
// zeros, which pads the M / N / K edges without branches.
#define OOB 0x80000000u
#define BUF_WORD3 0x00020000  // gfx9 buffer resource word 3 (raw, untyped)

__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)
// vmcnt(N): all but the N most recent vector memory loads have completed
// (loads retire in issue order)
template <int N>
__device__ __forceinline__ void wait_vmem_but() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// Workgroup barrier without __syncthreads()'s release fence, which would
// wait for every outstanding load (vmcnt(0)), including the DMA of the tile
// after next.  Ordering is explicit instead: each wave waits (vmcnt) for the
// DMAs the next tile needs before the barrier, and every LDS read of a stage
// has been consumed by an MFMA before the barrier that precedes the stage's
// refill.  The empty asm statements keep the compiler from moving memory
// accesses across the barrier.
__device__ __forceinline__ void barrier_no_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Output tile of this workgroup, XCD aware: consecutive workgroup ids are
// dealt to the 8 XCDs round robin, so ids are remapped so that each XCD
// receives a contiguous run of tiles, walked in groups of GROUP_M tile rows.
__device__ __forceinline__ void gemm_tile(const GemmArgs &a, int &tm, int &tn) {
  const int ntiles = a.tiles_m * a.tiles_n;
  int pid = blockIdx.x;
  if ((ntiles & 7) == 0) pid = (pid & 7) * (ntiles >> 3) + (pid >> 3);
  const int gm = a.group_m > 0 ? a.group_m : GROUP_M;
  const int in_group = gm * a.tiles_n;
  const int group = pid / in_group;
  const int first_m = group * gm;
  const int gsize = min(a.tiles_m - first_m, gm);
  tm = first_m + (pid % in_group) % gsize;
  tn = (pid % in_group) / gsize;
}

template <int N> struct Int {
  static constexpr int value = N;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 16-byte chunk swizzle of a 64-byte row: chunk c of row r at c ^ hswz(r)
__device__ __forceinline__ int hswz(int row) { return (row >> 2) & 3; }
// 64-deep stages: 128-byte rows of 8 chunks, 64-byte rows of 4 chunks
__device__ __forceinline__ int swz_a64(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int swz_b64(int r) { return (r >> 2) & 3; }

// LDS DMA as in dma16_asm, with a uniform (SGPR) part of the offset: voff + soff
__device__ __forceinline__ void dma16_asm_so(i32x4_t r, uint32_t lds, uint32_t voff, uint32_t soff) {
  const uint32_t m = __builtin_amdgcn_readfirstlane(lds);
  const uint32_t so = __builtin_amdgcn_readfirstlane(soff);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %3 offen lds"
               :: "v"(voff), "s"(r), "s"(m), "s"(so) : "memory", "m0");
}
