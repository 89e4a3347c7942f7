// Generic fallback kernels for graph nodes no fused pattern covers.
//
// nk_ew_program: one thread per output element evaluates a short register
//   program (loads with arbitrary strides -- broadcast, transpose, slice and
//   reverse are stride patterns -- constants, iota, unary / binary / select /
//   compare ops).  Registers are double; every instruction rounds its result
//   to the dtype of the graph node it implements, so chained ops see the same
//   intermediate roundings as NumPy in the node dtype.
// nk_reduce:   one workgroup per output element, any set of reduced axes.
// nk_dot:      batched C = A * B with arbitrary operand strides, LDS tiles,
//              fp32 accumulation.  Fallback only: the fused GEMM kernels are
//              the fast path.
// nk_gather / nk_scatter: take, take_along_axis, scatter / put along axis.
// nk_cumsum:   sequential scan per line.
//
// Index operands are clamped into range (never a fault on bad indices).

#include "common.h"

using namespace nk;

enum DType : int32_t {
  DT_F32 = 0, DT_F16 = 1, DT_BF16 = 2, DT_E4M3 = 3, DT_I8 = 4, DT_I16 = 5,
  DT_I32 = 6, DT_I64 = 7, DT_U8 = 8, DT_U16 = 9, DT_U32 = 10, DT_U64 = 11,
  DT_BOOL = 12, DT_F64 = 13,
};

__device__ __forceinline__ double load_any(const void *p, int64_t i, int dt) {
  switch (dt) {
    case DT_F32: return (double)((const float *)p)[i];
    case DT_F16: return (double)f16_to_f32(((const uint16_t *)p)[i]);
    case DT_BF16: return (double)bf16_to_f32(((const uint16_t *)p)[i]);
    case DT_E4M3: return (double)e4m3_to_f32(((const uint8_t *)p)[i]);
    case DT_I8: return (double)((const int8_t *)p)[i];
    case DT_I16: return (double)((const int16_t *)p)[i];
    case DT_I32: return (double)((const int32_t *)p)[i];
    case DT_I64: return (double)((const int64_t *)p)[i];
    case DT_U8: return (double)((const uint8_t *)p)[i];
    case DT_U16: return (double)((const uint16_t *)p)[i];
    case DT_U32: return (double)((const uint32_t *)p)[i];
    case DT_U64: return (double)((const uint64_t *)p)[i];
    case DT_BOOL: return ((const uint8_t *)p)[i] ? 1.0 : 0.0;
    case DT_F64: return ((const double *)p)[i];
  }
  return 0.0;
}

// E4M3FN encode, round to nearest even, saturating to +-448.
__device__ __forceinline__ uint8_t f32_to_e4m3(float f) {
  uint32_t u = __float_as_uint(f);
  uint8_t sign = (u >> 24) & 0x80;
  float a = fabsf(f);
  if (a != a) return 0x7f;
  if (a >= 448.f) return sign | 0x7e;
  if (a < 0.0009765625f) {  // below half the smallest subnormal (2^-10)
    return sign;
  }
  int e;
  float m = frexpf(a, &e);  // a = m * 2^e, m in [0.5, 1)
  int exp = e - 1 + 7;      // biased exponent of the 1.xxx form
  uint32_t code;
  if (exp <= 0) {
    // subnormal: value = k * 2^-9, k = 0..7
    float k = rintf(a * 512.f);
    code = (uint32_t)k;  // k == 8 rolls into the smallest normal (0x08)
  } else {
    float q = rintf((m * 2.f - 1.f) * 8.f);  // mantissa 0..8
    uint32_t mant = (uint32_t)q;
    if (mant == 8) { mant = 0; exp += 1; }
    code = ((uint32_t)exp << 3) | mant;
    if (code > 0x7e) code = 0x7e;
  }
  return sign | (uint8_t)code;
}

__device__ __forceinline__ double round_to_dtype(double v, int dt) {
  switch (dt) {
    case DT_F32: return (double)(float)v;
    case DT_F16: return (double)f16_to_f32(f32_to_f16((float)v));
    case DT_BF16: return (double)bf16_to_f32(f32_to_bf16((float)v));
    case DT_E4M3: return (double)e4m3_to_f32(f32_to_e4m3((float)v));
    case DT_I8: return (double)(int8_t)(int64_t)v;
    case DT_I16: return (double)(int16_t)(int64_t)v;
    case DT_I32: return (double)(int32_t)(int64_t)v;
    case DT_I64: return (double)(int64_t)v;
    case DT_U8: return (double)(uint8_t)(int64_t)v;
    case DT_U16: return (double)(uint16_t)(int64_t)v;
    case DT_U32: return (double)(uint32_t)(int64_t)v;
    case DT_U64: return (double)(uint64_t)v;
    case DT_BOOL: return v != 0.0 ? 1.0 : 0.0;
  }
  return v;
}

__device__ __forceinline__ void store_any(void *p, int64_t i, int dt, double v) {
  switch (dt) {
    case DT_F32: ((float *)p)[i] = (float)v; break;
    case DT_F16: ((uint16_t *)p)[i] = f32_to_f16((float)v); break;
    case DT_BF16: ((uint16_t *)p)[i] = f32_to_bf16((float)v); break;
    case DT_E4M3: ((uint8_t *)p)[i] = f32_to_e4m3((float)v); break;
    case DT_I8: ((int8_t *)p)[i] = (int8_t)(int64_t)v; break;
    case DT_I16: ((int16_t *)p)[i] = (int16_t)(int64_t)v; break;
    case DT_I32: ((int32_t *)p)[i] = (int32_t)(int64_t)v; break;
    case DT_I64: ((int64_t *)p)[i] = (int64_t)v; break;
    case DT_U8: ((uint8_t *)p)[i] = (uint8_t)(int64_t)v; break;
    case DT_U16: ((uint16_t *)p)[i] = (uint16_t)(int64_t)v; break;
    case DT_U32: ((uint32_t *)p)[i] = (uint32_t)(int64_t)v; break;
    case DT_U64: ((uint64_t *)p)[i] = (uint64_t)v; break;
    case DT_BOOL: ((uint8_t *)p)[i] = v != 0.0 ? 1 : 0; break;
    case DT_F64: ((double *)p)[i] = v; break;
  }
}

// ---------------------------------------------------------------------------
// Elementwise program
// ---------------------------------------------------------------------------
#define EW_MAX_RANK 6
#define EW_MAX_IN 8
#define EW_MAX_INSTR 40
#define EW_REGS 16

enum EwOp : int16_t {
  OP_LOAD = 0, OP_CONST, OP_IOTA,
  // unary
  OP_NEG = 10, OP_ABS, OP_EXP, OP_LOG, OP_SQRT, OP_RSQRT, OP_SIN, OP_COS, OP_TAN,
  OP_ATAN, OP_TANH, OP_CEIL, OP_FLOOR, OP_RINT, OP_TRUNC, OP_SIGN, OP_NOT, OP_LOG1P,
  OP_EXPM1, OP_ISFINITE, OP_ISNAN, OP_LOGISTIC, OP_LOG2, OP_COPY,
  // binary
  OP_ADD = 40, OP_SUB, OP_MUL, OP_DIV, OP_POW, OP_MAX, OP_MIN, OP_AND, OP_OR, OP_XOR,
  OP_REM, OP_FLOORDIV, OP_ATAN2,
  // compare
  OP_EQ = 60, OP_NE, OP_LT, OP_LE, OP_GT, OP_GE,
  // ternary
  OP_SELECT = 70,
};

struct EwInput {
  const void *ptr;
  int64_t strides[EW_MAX_RANK];  // in elements, over the output index space
  int32_t dtype;
  int32_t pad;
};

struct EwInstr {
  int16_t op;
  int8_t dst, a, b, c;
  int8_t dtype;  // result dtype (rounding) ; for OP_LOAD: unused
  int8_t flags;  // bit0: operands are integers (integer semantics)
  double imm;    // OP_CONST value; OP_IOTA dimension; OP_LOAD input index
};

struct EwArgs {
  void *out;
  int64_t out_offset;                // elements
  int64_t out_strides[EW_MAX_RANK];  // elements
  int64_t shape[EW_MAX_RANK];
  int64_t total;
  int32_t rank, n_in, n_instr, out_dtype;
  int32_t result_reg, pad;
  int64_t nthreads;  // grid size * 256 (grid-stride loop step)
  EwInput in[EW_MAX_IN];
  EwInstr prog[EW_MAX_INSTR];
};

__device__ __forceinline__ double floor_mod(double a, double b, bool isint) {
  if (isint) {
    int64_t x = (int64_t)a, y = (int64_t)b;
    if (y == 0) return 0.0;
    int64_t r = x % y;
    if (r != 0 && ((r < 0) != (y < 0))) r += y;
    return (double)r;
  }
  double r = fmod(a, b);
  if (r != 0.0 && ((r < 0.0) != (b < 0.0))) r += b;
  return r;
}

__device__ __forceinline__ double floor_div(double a, double b, bool isint) {
  if (isint) {
    int64_t x = (int64_t)a, y = (int64_t)b;
    if (y == 0) return 0.0;
    int64_t q = x / y;
    if ((x % y != 0) && ((x < 0) != (y < 0))) q -= 1;
    return (double)q;
  }
  return floor(a / b);
}

extern "C" __global__ __launch_bounds__(256) void nk_ew_program(EwArgs a) {
  const int64_t stride = a.nthreads;
  for (int64_t lin = (int64_t)blockIdx.x * 256 + threadIdx.x; lin < a.total; lin += stride) {
    int64_t idx[EW_MAX_RANK];
    int64_t rem = lin;
    for (int d = a.rank - 1; d >= 0; --d) {
      idx[d] = rem % a.shape[d];
      rem /= a.shape[d];
    }
    double r[EW_REGS];
    for (int k = 0; k < a.n_instr; ++k) {
      const EwInstr &I = a.prog[k];
      const bool isint = I.flags & 1;
      double x = r[I.a & (EW_REGS - 1)];
      double y = r[I.b & (EW_REGS - 1)];
      double v = 0.0;
      switch (I.op) {
        case OP_LOAD: {
          const EwInput &in = a.in[(int)I.imm];
          int64_t off = 0;
          for (int d = 0; d < a.rank; ++d) off += idx[d] * in.strides[d];
          v = load_any(in.ptr, off, in.dtype);
          break;
        }
        case OP_CONST: v = I.imm; break;
        case OP_IOTA: v = (double)idx[(int)I.imm]; break;
        case OP_NEG: v = -x; break;
        case OP_ABS: v = fabs(x); break;
        case OP_EXP: v = exp(x); break;
        case OP_LOG: v = log(x); break;
        case OP_SQRT: v = sqrt(x); break;
        case OP_RSQRT: v = 1.0 / sqrt(x); break;
        case OP_SIN: v = sin(x); break;
        case OP_COS: v = cos(x); break;
        case OP_TAN: v = tan(x); break;
        case OP_ATAN: v = atan(x); break;
        case OP_TANH: v = tanh(x); break;
        case OP_CEIL: v = ceil(x); break;
        case OP_FLOOR: v = floor(x); break;
        case OP_RINT: v = rint(x); break;
        case OP_TRUNC: v = trunc(x); break;
        case OP_SIGN: v = (x > 0.0) ? 1.0 : ((x < 0.0) ? -1.0 : x); break;
        case OP_NOT: v = (I.dtype == DT_BOOL) ? (x != 0.0 ? 0.0 : 1.0) : (double)(~(int64_t)x); break;
        case OP_LOG1P: v = log1p(x); break;
        case OP_EXPM1: v = expm1(x); break;
        case OP_ISFINITE: v = isfinite(x) ? 1.0 : 0.0; break;
        case OP_ISNAN: v = isnan(x) ? 1.0 : 0.0; break;
        case OP_LOGISTIC: v = 1.0 / (1.0 + exp(-x)); break;
        case OP_LOG2: v = log2(x); break;
        case OP_COPY: v = x; break;
        case OP_ADD: v = x + y; break;
        case OP_SUB: v = x - y; break;
        case OP_MUL: v = x * y; break;
        case OP_DIV:
          if (isint) v = (y == 0.0) ? 0.0 : (double)((int64_t)x / (int64_t)y);
          else v = x / y;
          break;
        case OP_POW: v = pow(x, y); break;
        case OP_MAX: v = (x != x || y != y) ? (x + y) : fmax(x, y); break;
        case OP_MIN: v = (x != x || y != y) ? (x + y) : fmin(x, y); break;
        case OP_AND: v = (double)((int64_t)x & (int64_t)y); break;
        case OP_OR: v = (double)((int64_t)x | (int64_t)y); break;
        case OP_XOR: v = (double)((int64_t)x ^ (int64_t)y); break;
        case OP_REM: v = floor_mod(x, y, isint); break;
        case OP_FLOORDIV: v = floor_div(x, y, isint); break;
        case OP_ATAN2: v = atan2(x, y); break;
        case OP_EQ: v = x == y; break;
        case OP_NE: v = x != y; break;
        case OP_LT: v = x < y; break;
        case OP_LE: v = x <= y; break;
        case OP_GT: v = x > y; break;
        case OP_GE: v = x >= y; break;
        case OP_SELECT: v = (x != 0.0) ? y : r[I.c & (EW_REGS - 1)]; break;
      }
      r[I.dst & (EW_REGS - 1)] = round_to_dtype(v, I.dtype);
    }
    int64_t off = a.out_offset;
    for (int d = 0; d < a.rank; ++d) off += idx[d] * a.out_strides[d];
    store_any(a.out, off, a.out_dtype, r[a.result_reg & (EW_REGS - 1)]);
  }
}

// ---------------------------------------------------------------------------
// Elementwise program over float types, four elements per thread.
//
// nk_ew_program interprets in double, one element per thread, at 247 registers
// (two waves per SIMD): its time is the interpretation, 16 instructions over
// 614400 elements 38 us.  Programs whose values are all fp32 / fp16 / bf16 /
// bool and whose operations are listed below run here instead: registers are
// fp32, each instruction is decoded once for four consecutive elements of the
// innermost dimension, inputs contiguous there load as one vector, and the
// dimensions come collapsed from the host (usually one or two).  The results
// are the other kernel's bit for bit: an fp32 sum, difference, product, quotient
// or root equals the double one rounded to fp32 (53 >= 2 * 24 + 2 bits; and 24
// >= 2 * 11 + 2 for fp16 by way of fp32), and the transcendental functions are
// evaluated in double here too and narrowed in one rounding (ewf_narrow).
// That program, a SiLU with its product over 200 x 3072 fp32: 38 us there, 9.4
// us here (0.8 TB/s; the double exp of each element bounds it).
// ---------------------------------------------------------------------------
#define EWF_MAX_RANK 6
struct EwfInput {
  const void *ptr;
  int32_t strides[EWF_MAX_RANK];  // elements, over the collapsed dimensions
  int32_t dtype;
  int32_t mode;                   // innermost: 0 broadcast, 1 aligned vector of 4, 2 strided
};
struct EwfInstr {
  uint8_t op, dst, a, b, c, dtype;
  uint8_t pad[2];
  float imm;  // OP_CONST value; OP_LOAD input index
};
struct EwfArgs {
  void *out;
  int32_t out_strides[EWF_MAX_RANK];
  uint32_t shape[EWF_MAX_RANK];
  uint32_t total, step;           // elements, elements per grid pass
  int32_t rank, n_instr, out_dtype, out_mode, result_reg;
  int32_t rows4;                  // the innermost dimension is a multiple of 4
  EwfInput in[EW_MAX_IN];
  EwfInstr prog[EW_MAX_INSTR];
};
typedef float f32v16 __attribute__((ext_vector_type(16)));

// four elements at offsets o: all loads in flight before the first is widened
__device__ __forceinline__ void ewf_gather(const void *p, const int32_t (&o)[4], int dt, float (&v)[4]) {
  if (dt == DT_F32) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = ((const float *)p)[o[e]];
  } else if (dt == DT_BOOL) {
    uint8_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = ((const uint8_t *)p)[o[e]];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = h[e] ? 1.f : 0.f;
  } else {
    uint16_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = ((const uint16_t *)p)[o[e]];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = dt == DT_BF16 ? bf16_to_f32(h[e]) : f16_to_f32(h[e]);
  }
}
__device__ __forceinline__ float ewf_round(float v, int dt) {
  if (dt == DT_BF16) return bf16_to_f32(f32_to_bf16(v));
  if (dt == DT_F16) return f16_to_f32(f32_to_f16(v));
  if (dt == DT_BOOL) return v != 0.f ? 1.f : 0.f;
  return v;
}
// A double result as the fp32 that ewf_round narrows.  nk_ew_program's double
// reaches fp16 in one rounding (the compiler contracts its two conversions); on
// the way to fp16 this one is rounded to odd (toward zero, an inexact one with
// its last bit set), which keeps the fp16 rounding from seeing a tie that the
// double is not on: exp(0.02269) lies 2.7e-8 below the middle of two fp16
// values and its nearest fp32 is that middle.  bf16 results are the same either
// way, for every operand of that type.
template <bool F16FN>
__device__ __forceinline__ float ewf_narrow(double d, int dt) {
  if (F16FN) {
    // fp32 keeps the upper 23 of 52 fraction bits: the 29 below become one (by
    // a mask: a branch on dt spills registers)
    const uint32_t m = dt == DT_F16 ? 0x1fffffffu : 0u;
    const uint64_t u = (uint64_t)__double_as_longlong(d);
    const uint32_t lo = (uint32_t)u;
    const uint32_t odd = (lo | ((lo & m) + m)) & ~m;
    d = __longlong_as_double((long long)((u & 0xffffffff00000000ull) | odd));
  }
  const float f = (float)d;
  // one element's function at a time: interleaved, the four need 37 registers
  // more than there are at four waves per SIMD
  if (F16FN) __builtin_amdgcn_sched_barrier(0);
  return f;
}
__device__ __forceinline__ void ewf_store1(void *p, int32_t i, int dt, float v) {
  if (dt == DT_F32) ((float *)p)[i] = v;
  else if (dt == DT_BF16) ((uint16_t *)p)[i] = f32_to_bf16(v);
  else if (dt == DT_F16) ((uint16_t *)p)[i] = f32_to_f16(v);
  else ((uint8_t *)p)[i] = v != 0.f ? 1 : 0;
}

// F16FN: some function's result is fp16.  A kernel of its own, so that the other
// programs' code stays without the mask and the barriers.  The SiLU program
// above in fp16 over 4096 x 4096, a call: 175 us, 163..178 us without the
// narrowing, 1065 us in nk_ew_program (200 x 3072: 30 / 30 / 64 us).
template <bool F16FN>
__device__ __forceinline__ void ewf_body(const EwfArgs &a) {
  for (uint64_t lin0 = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4; lin0 < a.total; lin0 += a.step) {
    const uint32_t lin = (uint32_t)lin0;
    const uint32_t n = min(4u, a.total - lin);
    // offset of element e of a strided operand (uniform branch: rows of whole
    // fours need one decomposition)
    auto offset = [&](const int32_t *st, uint32_t l) __attribute__((always_inline)) {
      int32_t off = 0;
      uint32_t rem = l;
      for (int d = a.rank - 1; d > 0; --d) {
        const uint32_t q = rem / a.shape[d];
        off += (int32_t)(rem - q * a.shape[d]) * st[d];
        rem = q;
      }
      return off + (int32_t)rem * st[0];
    };
    f32v16 r[4];
    for (int k = 0; k < a.n_instr; ++k) {
      const EwfInstr &I = a.prog[k];
      float x[4], y[4], v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = r[e][I.a & 15];
        y[e] = r[e][I.b & 15];
      }
#define EWF(OP, EXPR)                            \
  case OP:                                       \
    _Pragma("unroll") for (int e = 0; e < 4; ++e) v[e] = (EXPR); \
    break;
      switch (I.op) {
        case OP_LOAD: {
          const EwfInput &in = a.in[(int)I.imm];
          if (a.rows4) {
            const int32_t o = offset(in.strides, lin);
            if (in.mode == 1) {
              if (in.dtype == DT_F32) {
                const float4 q = *reinterpret_cast<const float4 *>((const float *)in.ptr + o);
                v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
              } else if (in.dtype == DT_BOOL) {
                const uint32_t q = *reinterpret_cast<const uint32_t *>((const uint8_t *)in.ptr + o);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ((q >> (8 * e)) & 0xff) ? 1.f : 0.f;
              } else {
                const uint2 q = *reinterpret_cast<const uint2 *>((const uint16_t *)in.ptr + o);
                const uint32_t h[4] = {q.x & 0xffffu, q.x >> 16, q.y & 0xffffu, q.y >> 16};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  v[e] = in.dtype == DT_BF16 ? bf16_to_f32((uint16_t)h[e]) : f16_to_f32((uint16_t)h[e]);
              }
            } else {
              const int32_t s = in.strides[a.rank - 1];  // 0: broadcast
              const int32_t at[4] = {o, o + s, o + 2 * s, o + 3 * s};
              ewf_gather(in.ptr, at, in.dtype, v);
            }
          } else {
            int32_t at[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) at[e] = offset(in.strides, lin + min((uint32_t)e, n - 1));
            ewf_gather(in.ptr, at, in.dtype, v);
          }
          break;
        }
        EWF(OP_CONST, I.imm)
        EWF(OP_NEG, -x[e])
        EWF(OP_ABS, fabsf(x[e]))
        EWF(OP_EXP, ewf_narrow<F16FN>(exp((double)x[e]), I.dtype))
        EWF(OP_LOG, ewf_narrow<F16FN>(log((double)x[e]), I.dtype))
        EWF(OP_SQRT, (float)sqrt((double)x[e]))
        EWF(OP_RSQRT, ewf_narrow<F16FN>(1.0 / sqrt((double)x[e]), I.dtype))
        EWF(OP_TANH, ewf_narrow<F16FN>(tanh((double)x[e]), I.dtype))
        EWF(OP_CEIL, ceilf(x[e]))
        EWF(OP_FLOOR, floorf(x[e]))
        EWF(OP_RINT, rintf(x[e]))
        EWF(OP_TRUNC, truncf(x[e]))
        EWF(OP_SIGN, (x[e] > 0.f) ? 1.f : ((x[e] < 0.f) ? -1.f : x[e]))
        EWF(OP_ISFINITE, isfinite(x[e]) ? 1.f : 0.f)
        EWF(OP_ISNAN, isnan(x[e]) ? 1.f : 0.f)
        EWF(OP_LOGISTIC, ewf_narrow<F16FN>(1.0 / (1.0 + exp(-(double)x[e])), I.dtype))
        EWF(OP_COPY, x[e])
        EWF(OP_ADD, x[e] + y[e])
        EWF(OP_SUB, x[e] - y[e])
        EWF(OP_MUL, x[e] * y[e])
        EWF(OP_DIV, (float)((double)x[e] / (double)y[e]))
        EWF(OP_MAX, (x[e] != x[e] || y[e] != y[e]) ? (x[e] + y[e]) : fmaxf(x[e], y[e]))
        EWF(OP_MIN, (x[e] != x[e] || y[e] != y[e]) ? (x[e] + y[e]) : fminf(x[e], y[e]))
        EWF(OP_EQ, x[e] == y[e] ? 1.f : 0.f)
        EWF(OP_NE, x[e] != y[e] ? 1.f : 0.f)
        EWF(OP_LT, x[e] < y[e] ? 1.f : 0.f)
        EWF(OP_LE, x[e] <= y[e] ? 1.f : 0.f)
        EWF(OP_GT, x[e] > y[e] ? 1.f : 0.f)
        EWF(OP_GE, x[e] >= y[e] ? 1.f : 0.f)
        EWF(OP_SELECT, x[e] != 0.f ? y[e] : r[e][I.c & 15])
        default: EWF(OP_NOT, x[e] != 0.f ? 0.f : 1.f)
      }
#undef EWF
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e][I.dst & 15] = ewf_round(v[e], I.dtype);
    }
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = r[e][a.result_reg & 15];
    if (a.rows4) {
      const int32_t at = offset(a.out_strides, lin);
      if (a.out_mode == 1 && a.out_dtype == DT_F32) {
        *reinterpret_cast<float4 *>((float *)a.out + at) = make_float4(o[0], o[1], o[2], o[3]);
      } else if (a.out_mode == 1 && a.out_dtype == DT_BF16) {
        *reinterpret_cast<uint2 *>((uint16_t *)a.out + at) =
            make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      } else if (a.out_mode == 1 && a.out_dtype == DT_F16) {
        *reinterpret_cast<uint2 *>((uint16_t *)a.out + at) =
            make_uint2((uint32_t)f32_to_f16(o[0]) | ((uint32_t)f32_to_f16(o[1]) << 16),
                       (uint32_t)f32_to_f16(o[2]) | ((uint32_t)f32_to_f16(o[3]) << 16));
      } else {
        const int32_t s = a.out_strides[a.rank - 1];
#pragma unroll
        for (int e = 0; e < 4; ++e) ewf_store1(a.out, at + e * s, a.out_dtype, o[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if ((uint32_t)e < n) ewf_store1(a.out, offset(a.out_strides, lin + e), a.out_dtype, o[e]);
    }
  }
}

extern "C" __global__ __launch_bounds__(256, 4) void nk_ew_f32(EwfArgs a) { ewf_body<false>(a); }
extern "C" __global__ __launch_bounds__(256, 4) void nk_ew_f32_f16fn(EwfArgs a) { ewf_body<true>(a); }

// ---------------------------------------------------------------------------
// SwiGLU over a fp32 product's partial planes: with P the sum of the planes in
// the order of gemv.hip's reduction (four interleaved sums), out[m][j] = (g * (1 / (1 + exp(-g)))) * u, g = P[m][og + j], u = P[m][ou
// + j].  The planes' reduction and the program of nk_ew_f32 in one launch, bit
// for bit theirs (fp32 values, exp rounded from double).  Latency bounds the
// small sizes, of which the interpreter's decode and dependent loads were most;
// all loads of a thread's four outputs are in flight together here.  200 x 3072
// from two planes 5.0 us, the two launches it replaces 4.9 + 9.3; 2 x 3072
// from eight 4.0, 4.0 + 8.9.
// ---------------------------------------------------------------------------
struct SwigluPlanesArgs {
  const float *P;
  float *out;
  int64_t plane;  // elements of a plane
  int32_t rows, F, N, ks, og, ou;
};
extern "C" __global__ __launch_bounds__(64) void nk_swiglu_planes_f32(SwigluPlanesArgs a) {
  const uint32_t i = blockIdx.x * 64 + threadIdx.x, f4 = (uint32_t)a.F / 4;
  const uint32_t r = i / f4, j = 4 * (i % f4);
  if (r >= (uint32_t)a.rows) return;
  const float *p = a.P + (int64_t)r * a.N + j;
  float g4[4][4], u4[4][4];  // (0 + x is x but for x = -0: one plane is copied)
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) g4[q][e] = u4[q][e] = 0.f;
  for (int s0 = 0; s0 < a.ks; s0 += 4) {
    float4 x[4], y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t s = min(s0 + q, a.ks - 1) * a.plane;
      x[q] = *reinterpret_cast<const float4 *>(p + s + a.og);
      y[q] = *reinterpret_cast<const float4 *>(p + s + a.ou);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (s0 + q >= a.ks) break;
      const float xv[4] = {x[q].x, x[q].y, x[q].z, x[q].w}, yv[4] = {y[q].x, y[q].y, y[q].z, y[q].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        g4[q][e] = a.ks == 1 ? xv[e] : g4[q][e] + xv[e];
        u4[q][e] = a.ks == 1 ? yv[e] : u4[q][e] + yv[e];
      }
    }
  }
  float g[4], u[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    g[e] = a.ks == 1 ? g4[0][e] : (g4[0][e] + g4[1][e]) + (g4[2][e] + g4[3][e]);
    u[e] = a.ks == 1 ? u4[0][e] : (u4[0][e] + u4[1][e]) + (u4[2][e] + u4[3][e]);
  }
  float o[4];
  {
#pragma clang fp contract(off)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = 1.f + (float)exp((double)-g[e]);
      o[e] = g[e] * (1.f / d) * u[e];
    }
  }
  *reinterpret_cast<float4 *>(a.out + (int64_t)r * a.F + j) = make_float4(o[0], o[1], o[2], o[3]);
}

// ---------------------------------------------------------------------------
// Reduction: one workgroup per output element.
// ---------------------------------------------------------------------------
#define RED_MAX_RANK 6
enum RedOp : int32_t { RED_ADD = 0, RED_MAX, RED_MIN, RED_MUL, RED_AND, RED_OR, RED_ARGMAX, RED_ARGMIN };

struct ReduceArgs {
  const void *in;
  void *out;
  int64_t out_shape[RED_MAX_RANK];
  int64_t out_strides[RED_MAX_RANK];  // input strides of the kept axes
  int64_t red_shape[RED_MAX_RANK];
  int64_t red_strides[RED_MAX_RANK];  // input strides of the reduced axes
  int64_t n_out, n_red;
  int32_t out_rank, red_rank, op, in_dtype, out_dtype, acc_f32;
};

__device__ __forceinline__ double red_init(int op) {
  switch (op) {
    case RED_ADD: case RED_OR: return 0.0;
    case RED_MUL: case RED_AND: return 1.0;
    case RED_MAX: case RED_ARGMAX: return -INFINITY;
    default: return INFINITY;
  }
}

__device__ __forceinline__ double red_comb(int op, double a, double b) {
  switch (op) {
    case RED_ADD: return a + b;
    case RED_MUL: return a * b;
    case RED_MAX: return (a != a || b != b) ? a + b : fmax(a, b);
    case RED_MIN: return (a != a || b != b) ? a + b : fmin(a, b);
    case RED_AND: return (a != 0.0 && b != 0.0) ? 1.0 : 0.0;
    case RED_OR: return (a != 0.0 || b != 0.0) ? 1.0 : 0.0;
  }
  return a;
}

extern "C" __global__ __launch_bounds__(256) void nk_reduce(ReduceArgs a) {
  __shared__ double sv[256];
  __shared__ int64_t si[256];
  const int64_t o = blockIdx.x;
  if (o >= a.n_out) return;
  int64_t base = 0, rem = o;
  for (int d = a.out_rank - 1; d >= 0; --d) {
    base += (rem % a.out_shape[d]) * a.out_strides[d];
    rem /= a.out_shape[d];
  }
  const bool arg = a.op == RED_ARGMAX || a.op == RED_ARGMIN;
  const bool amax = a.op == RED_ARGMAX;
  double acc = red_init(a.op);
  int64_t best = a.n_red;  // sentinel: no element seen
  for (int64_t j = threadIdx.x; j < a.n_red; j += 256) {
    int64_t off = base, r2 = j;
    for (int d = a.red_rank - 1; d >= 0; --d) {
      off += (r2 % a.red_shape[d]) * a.red_strides[d];
      r2 /= a.red_shape[d];
    }
    double v = load_any(a.in, off, a.in_dtype);
    if (arg) {
      // first occurrence wins; a NaN beats any number (NumPy semantics)
      bool take = best == a.n_red ||
                  (acc == acc && (v != v || (amax ? v > acc : v < acc)));
      if (take) { acc = v; best = j; }
    } else {
      acc = red_comb(a.op, acc, v);
      if (a.acc_f32) acc = (double)(float)acc;
    }
  }
  sv[threadIdx.x] = acc;
  si[threadIdx.x] = best;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      double x = sv[threadIdx.x], y = sv[threadIdx.x + s];
      if (arg) {
        int64_t ix = si[threadIdx.x], iy = si[threadIdx.x + s];
        bool take_y = false;
        if (iy < a.n_red) {
          if (ix >= a.n_red) take_y = true;
          else if (x != x) take_y = (y != y) && iy < ix;
          else if (y != y) take_y = true;
          else if (amax ? y > x : y < x) take_y = true;
          else if (y == x && iy < ix) take_y = true;
        }
        if (take_y) { sv[threadIdx.x] = y; si[threadIdx.x] = iy; }
      } else {
        double z = red_comb(a.op, x, y);
        sv[threadIdx.x] = a.acc_f32 ? (double)(float)z : z;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (arg) store_any(a.out, o, a.out_dtype, (double)si[0]);
    else store_any(a.out, o, a.out_dtype, sv[0]);
  }
}

// ---------------------------------------------------------------------------
// Generic batched dot: C[b, m, n] = sum_k A[b, m, k] * B[b, k, n]
// ---------------------------------------------------------------------------
struct DotArgs {
  const void *A;
  const void *B;
  void *C;
  int64_t batch, M, N, K;
  int64_t sab, sam, sak;  // A strides (elements)
  int64_t sbb, sbk, sbn;  // B strides
  int32_t a_dtype, b_dtype, c_dtype, pad;
};

#define DT_TILE 16
extern "C" __global__ __launch_bounds__(256) void nk_dot(DotArgs a) {
  __shared__ float As[DT_TILE][DT_TILE + 1];
  __shared__ float Bs[DT_TILE][DT_TILE + 1];
  const int64_t b = blockIdx.z;
  const int tx = threadIdx.x % DT_TILE, ty = threadIdx.x / DT_TILE;
  const int64_t m = (int64_t)blockIdx.y * DT_TILE + ty;
  const int64_t n = (int64_t)blockIdx.x * DT_TILE + tx;
  float acc = 0.f;
  for (int64_t k0 = 0; k0 < a.K; k0 += DT_TILE) {
    int64_t ka = k0 + tx, kb = k0 + ty;
    As[ty][tx] = (m < a.M && ka < a.K) ? (float)load_any(a.A, b * a.sab + m * a.sam + ka * a.sak, a.a_dtype) : 0.f;
    Bs[ty][tx] = (kb < a.K && n < a.N) ? (float)load_any(a.B, b * a.sbb + kb * a.sbk + n * a.sbn, a.b_dtype) : 0.f;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < DT_TILE; ++k) acc = fmaf(As[ty][k], Bs[k][tx], acc);
    __syncthreads();
  }
  if (m < a.M && n < a.N) store_any(a.C, (b * a.M + m) * a.N + n, a.c_dtype, (double)acc);
}

// ---------------------------------------------------------------------------
// Gather / scatter along one axis.  Operands are viewed as (O, A, N):
// O = product of the axes before `axis`, A = the axis, N = the axes after.
//   mode 0 take:            out[o, i, n] = in[o, idx[i], n]           (I = #idx)
//   mode 1 take_along_axis: out[o, i, n] = in[o, idx[o, i, n], n]
//   mode 2 scatter:         out[o, idx[i], n] = upd[o, i, n]
//   mode 3 put_along_axis:  out[o, idx[o, i, n], n] = upd[o, i, n]
// Modes 2/3 expect `out` to already hold the operand.
// ---------------------------------------------------------------------------
struct GatherArgs {
  const void *src;  // in (modes 0/1) or updates (modes 2/3)
  const int32_t *idx;
  void *out;
  int64_t O, A, I, N;
  int64_t nthreads;  // grid size * 256
  int32_t mode, dtype;
};

extern "C" __global__ __launch_bounds__(256) void nk_gather(GatherArgs a) {
  const int64_t total = a.O * a.I * a.N;
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += a.nthreads) {
    const int64_t n = t % a.N;
    const int64_t i = (t / a.N) % a.I;
    const int64_t o = t / (a.N * a.I);
    int64_t j = (a.mode == 0 || a.mode == 2) ? a.idx[i] : a.idx[t];
    if (j < 0) j += a.A;
    const bool ok = j >= 0 && j < a.A;
    if (a.mode <= 1) {
      j = j < 0 ? 0 : (j >= a.A ? a.A - 1 : j);
      store_any(a.out, t, a.dtype, load_any(a.src, (o * a.A + j) * a.N + n, a.dtype));
    } else if (ok) {
      store_any(a.out, (o * a.A + j) * a.N + n, a.dtype, load_any(a.src, t, a.dtype));
    }
  }
}

// ---------------------------------------------------------------------------
// Inclusive cumulative sum along an axis viewed as (O, A, N).
// ---------------------------------------------------------------------------
struct CumsumArgs {
  const void *in;
  void *out;
  int64_t O, A, N;
  int32_t in_dtype, out_dtype, acc_f32, pad;
};

extern "C" __global__ __launch_bounds__(256) void nk_cumsum(CumsumArgs a) {
  const int64_t line = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (line >= a.O * a.N) return;
  const int64_t o = line / a.N, n = line % a.N;
  double acc = 0.0;
  for (int64_t i = 0; i < a.A; ++i) {
    const int64_t off = (o * a.A + i) * a.N + n;
    acc += load_any(a.in, off, a.in_dtype);
    if (a.acc_f32) acc = (double)(float)acc;
    store_any(a.out, off, a.out_dtype, acc);
  }
}

// ---------------------------------------------------------------------------
// Streaming copy of n16 16-byte words (plan flat copies; also the plain copy
// kernel of known size that calibrates the HBM traffic counters).
// ---------------------------------------------------------------------------
struct Copy16Args {
  const uint4 *src;
  uint4 *dst;
  int64_t n16;
  int64_t nthreads;  // grid size * 256
};

extern "C" __global__ __launch_bounds__(256) void nk_copy16(Copy16Args a) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n16; i += a.nthreads)
    nt_store16(a.dst + i, nt_load16(a.src + i));
}

// fp8 E4M3FN codes -> bf16 with the decode the GEMM staging uses (8 codes per
// thread).  Weight preparation and the exhaustive check of the decode.
struct DecodeE4m3Args {
  const uint2 *src;
  uint4 *dst;
  int64_t n8;
  int64_t nthreads;
};

extern "C" __global__ __launch_bounds__(256) void nk_decode_e4m3_bf16(DecodeE4m3Args a) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n8; i += a.nthreads)
    a.dst[i] = e4m3x8_to_bf16x8(a.src[i]);
}

// Row-wise top-k (indices) along the last axis: one workgroup per row.
// Round r selects, among the elements that come after round r-1's pick in
// the order (value descending, index ascending) -- ascending values when
// `largest` is 0 -- the first one; each round is one pass over the row, so
// the input is never modified.  k is small (sampling); rows must not hold
// NaN.
struct TopkArgs {
  const void *in;
  uint32_t *idx;  // rows x k
  int64_t rows;
  int64_t n;
  int32_t k;
  int32_t largest;
  int32_t dtype;
  int32_t pad;
};

extern "C" __global__ __launch_bounds__(256) void nk_topk(TopkArgs a) {
  __shared__ double sv[256];
  __shared__ int64_t si[256];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const int64_t base = row * a.n;
  const double sgn = a.largest ? 1.0 : -1.0;
  double pv = 0.0;
  int64_t pi = -1;  // previous pick (none before round 0)
  for (int r = 0; r < a.k; ++r) {
    double bv = -INFINITY;
    int64_t bi = a.n;
    for (int64_t j = tid; j < a.n; j += 256) {
      const double v = sgn * load_any(a.in, base + j, a.dtype);
      const bool after = pi < 0 || v < pv || (v == pv && j > pi);
      if (after && (v > bv || (v == bv && j < bi))) {
        bv = v;
        bi = j;
      }
    }
    sv[tid] = bv;
    si[tid] = bi;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (tid < s) {
        const double ov = sv[tid + s];
        const int64_t oi = si[tid + s];
        if (ov > sv[tid] || (ov == sv[tid] && oi < si[tid])) {
          sv[tid] = ov;
          si[tid] = oi;
        }
      }
      __syncthreads();
    }
    pv = sv[0];
    pi = si[0] < a.n ? si[0] : a.n - 1;  // a row shorter than k repeats its last pick
    if (tid == 0) a.idx[row * a.k + r] = (uint32_t)pi;
    __syncthreads();
  }
}

// Row-wise top-k of long rows, in two launches (nk_topk walks a row with one
// workgroup: 250 us for 8 rows of 151936, one memory round trip per 256
// elements; 5.4 + 4.0 us in this form, launches mostly).  A segment of TK_SEG elements is held in registers by one
// workgroup, which picks its k best; one workgroup per row then picks the k
// best of the segments' picks.  Elements are compared as 64-bit keys: the
// value mapped to an unsigned order (largest first; -0 as +0) above the
// complement of the index, so a larger key is a larger value or, among equals,
// a smaller index, and no two are equal: the picks and their order are those
// of nk_topk.  A NaN's key is 0, which no pick takes before any number, as
// there.  fp32, fp16 and bf16 rows.
#define TK_PER 16
#define TK_SEG (256 * TK_PER)
struct TopkSegArgs {
  const void *in;
  uint64_t *keys;  // rows x nseg x k
  uint32_t *idx;   // rows x k
  int64_t n;
  int32_t nseg, k, largest, dtype;
};

__device__ __forceinline__ uint64_t topk_key(float v, float sgn, uint32_t i) {
  const float x = sgn * v + 0.f;
  const uint32_t u = __float_as_uint(x);
  const uint32_t o = (u & 0x80000000u) ? ~u : u | 0x80000000u;
  return x != x ? 0 : ((uint64_t)o << 32) | (uint32_t)~i;
}
// the workgroup's largest key (all 256 threads get it)
__device__ __forceinline__ uint64_t topk_max(uint64_t m, uint64_t *sv) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t x = __shfl_xor((unsigned long long)m, o, 64);
    m = x > m ? x : m;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sv[threadIdx.x >> 6] = m;
  __syncthreads();
  const uint64_t a = sv[0] > sv[1] ? sv[0] : sv[1], b = sv[2] > sv[3] ? sv[2] : sv[3];
  return a > b ? a : b;
}

extern "C" __global__ __launch_bounds__(256) void nk_topk_segments(TopkSegArgs a) {
  __shared__ uint64_t sv[4];
  const int64_t row = blockIdx.x / (uint32_t)a.nseg;
  const int seg = blockIdx.x % (uint32_t)a.nseg;
  const int64_t base = row * a.n;
  const float sgn = a.largest ? 1.f : -1.f;
  const int esz = a.dtype == DT_F32 ? 4 : 2;
  const uint8_t *p = (const uint8_t *)a.in + base * esz;
  const bool vec = ((uintptr_t)p & 15) == 0;
  uint64_t key[TK_PER];
  // thread t: elements 8 t .. 8 t + 7 of each half of the segment
#pragma unroll
  for (int h = 0; h < TK_PER / 8; ++h) {
    const int64_t j0 = (int64_t)seg * TK_SEG + h * 2048 + threadIdx.x * 8;
    float v[8];
    if (vec && j0 + 8 <= a.n) {
      if (a.dtype == DT_F32) Vec8<float>::load((const float *)p + j0, v);
      else if (a.dtype == DT_BF16) Vec8<bf16>::load((const bf16 *)p + j0, v);
      else Vec8<f16>::load((const f16 *)p + j0, v);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = j0 + e < a.n ? (float)load_any(p, j0 + e, a.dtype) : __builtin_nanf("");
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) key[h * 8 + e] = topk_key(v[e], sgn, (uint32_t)(j0 + e));
  }
  uint64_t prev = ~0ull;
  uint64_t *out = a.keys + (int64_t)blockIdx.x * a.k;
  for (int r = 0; r < a.k; ++r) {
    uint64_t m = 0;
#pragma unroll
    for (int e = 0; e < TK_PER; ++e) m = key[e] < prev && key[e] > m ? key[e] : m;
    prev = topk_max(m, sv);
    if (threadIdx.x == 0) out[r] = prev;
  }
}

extern "C" __global__ __launch_bounds__(256) void nk_topk_merge(TopkSegArgs a) {
  __shared__ uint64_t sv[4];
  const int64_t row = blockIdx.x;
  const int cnt = a.nseg * a.k;
  const uint64_t *in = a.keys + row * cnt;
  uint64_t prev = ~0ull;
  for (int r = 0; r < a.k; ++r) {
    uint64_t m = 0;
    for (int j = threadIdx.x; j < cnt; j += 256) {
      const uint64_t x = in[j];
      m = x < prev && x > m ? x : m;
    }
    prev = topk_max(m, sv);
    // nothing left but NaN: the last element, as nk_topk
    if (threadIdx.x == 0) a.idx[row * a.k + r] = prev ? (uint32_t)~(uint32_t)prev : (uint32_t)(a.n - 1);
  }
}
