// What the GEMM kernels of gemm.hip and gemm_split.hip share: the operand formats and their MFMA steps, the epilogue
// chain and the stores of accumulator blocks, the LDS swizzles and the order in which workgroups take output tiles.
#pragma once
#include <type_traits>

#include "common.h"

namespace krn {

// Epilogue operations. Codes 0-5 take a float32 scalar or a row/column vector; 6-8 are the activations of krn's
// `lib.matmul` (reference src/krn/lib/lib_kernels.py:31-48, formulas of compiler/emit.py:112-114). A vector's
// element kind rides in bits 4-5 of the code: 0 float32, 1 f16, 2 bf16.
enum Op : int {
  MUL_SCALAR = 0, MUL_ROW = 1, MUL_COL = 2, ADD_SCALAR = 3, ADD_ROW = 4, ADD_COL = 5, RELU = 6, GELU = 7, SILU = 8
};
constexpr int VEC_KIND_SHIFT = 4;

struct Epilogue {
  int out_kind;          // F32, F16, BF16 or I32 (I32 only for an int8 product with no operations)
  int nops;              // elementwise operations applied in order, each rounded to float32
  int op[4];
  float scalar[4];
  const void* vec[4];    // per-row (length M) or per-column (length N) vectors
};

__device__ __forceinline__ float activation(int op, float x) {
  if (op == RELU) return x < 0.0f ? 0.0f : x;
  if (op == GELU) return __fmul_rn(__fmul_rn(0.5f, x), __fadd_rn(1.0f, erff(__fmul_rn(x, 0.7071067811865476f))));
  return __fdiv_rn(x, __fadd_rn(1.0f, expf(-x)));  // SILU
}

enum Format : int { FMT_BF16 = 0, FMT_F16 = 1, FMT_I8 = 2, FMT_FP8 = 3 };

typedef short v4s16 __attribute__((ext_vector_type(4)));  // the result type of ds_read_b64_tr_b16

template <int FMT>
struct Mfma;

template <>
struct Mfma<FMT_BF16> {
  typedef f32x16 Acc;
  static constexpr int kBytes = 32;  // bytes of K one instruction consumes per row
  __device__ static void step(Acc& c, const u32x4* a, const u32x4* b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[0]), __builtin_bit_cast(bf16x8, b[0]),
                                               c, 0, 0, 0);
  }
};

template <>
struct Mfma<FMT_F16> {
  typedef f32x16 Acc;
  static constexpr int kBytes = 32;
  __device__ static void step(Acc& c, const u32x4* a, const u32x4* b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[0]), __builtin_bit_cast(f16x8, b[0]), c,
                                              0, 0, 0);
  }
};

template <>
struct Mfma<FMT_I8> {
  typedef i32x16 Acc;
  static constexpr int kBytes = 32;
  __device__ static void step(Acc& c, const u32x4* a, const u32x4* b) {
    c = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a[0]), __builtin_bit_cast(i32x4, b[0]), c, 0,
                                             0, 0);
  }
};

template <>
struct Mfma<FMT_FP8> {
  typedef f32x16 Acc;
  static constexpr int kBytes = 64;
  __device__ static void step(Acc& c, const u32x4* a, const u32x4* b) {
    i32x8 av, bv;
    i32x4 a0 = __builtin_bit_cast(i32x4, a[0]), a1 = __builtin_bit_cast(i32x4, a[1]);
    i32x4 b0 = __builtin_bit_cast(i32x4, b[0]), b1 = __builtin_bit_cast(i32x4, b[1]);
    av = (i32x8){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
    bv = (i32x8){b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
    // format 0 = e4m3 for both operands; E8M0 scale 127 = 2^0
    c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, c, 0, 0, 0, 127, 0, 127);
  }
};

// The 16x16 forms, which consume twice the K per instruction for 16-bit and int8 operands. On gfx950 they sustain
// more throughput than the 32x32 forms under the same power limit (MFMA-only loops on random operands: bf16
// 16x16x32 0.93 of the per-clock peak at 1.71 GHz against 0.84 at 1.62 GHz for 32x32x16). Operand lane L holds row
// (or column) L & 15 and 16 bytes of K from (L >> 4) * 16; accumulator lane L holds column L & 15 of rows
// 4 (L >> 4) .. + 3.
template <int FMT>
struct Mfma16;

template <>
struct Mfma16<FMT_BF16> {
  typedef f32x4 Acc;
  __device__ static void step(Acc& c, u32x4 a, u32x4 b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                0, 0);
  }
  // the same as assembly with the accumulator tied to one AGPR tuple (the allocator otherwise moves 4-register
  // accumulators between AGPRs and VGPRs around the loop)
  __device__ static void step_agpr(Acc& c, u32x4 a, u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};

template <>
struct Mfma16<FMT_F16> {
  typedef f32x4 Acc;
  __device__ static void step(Acc& c, u32x4 a, u32x4 b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                               0);
  }
  __device__ static void step_agpr(Acc& c, u32x4 a, u32x4 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};

template <>
struct Mfma16<FMT_I8> {
  typedef i32x4 Acc;
  __device__ static void step_agpr(Acc& c, u32x4 a, u32x4 b) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};

template <>
struct Mfma16<FMT_FP8> {
  typedef f32x4 Acc;
  // v_mfma_scale_f32_16x16x128_f8f6f4 on e4m3 operands (format 0) with unit E8M0 scales (127 = 2^0, in `one`)
  __device__ static void step_agpr(Acc& c, i32x8 a, i32x8 b, int one) {
    asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %3 op_sel_hi:[0,0,0]"
                 : "+a"(c)
                 : "v"(a), "v"(b), "v"(one));
  }
};

template <typename V>
struct Elem;
template <>
struct Elem<f32x16> {
  typedef float T;
};
template <>
struct Elem<i32x16> {
  typedef int T;
};

template <typename V16, typename V4>
__device__ __forceinline__ V16 join16(const V4& s00, const V4& s01, const V4& s10, const V4& s11) {
  V16 t;
#pragma unroll
  for (int R = 0; R < 2; ++R)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t x0 = __builtin_bit_cast(uint32_t, R ? s10[q] : s00[q]);
      const uint32_t x1 = __builtin_bit_cast(uint32_t, R ? s11[q] : s01[q]);
      const auto p = __builtin_amdgcn_permlane16_swap(x0, x1, false, false);
      const auto w = __builtin_amdgcn_permlane32_swap(p[0], p[1], false, false);
      t[8 * R + q] = __builtin_bit_cast(typename Elem<V16>::T, (uint32_t)w[0]);
      t[8 * R + 4 + q] = __builtin_bit_cast(typename Elem<V16>::T, (uint32_t)w[1]);
    }
  return t;
}

// Store one 32x32 accumulator block (the C layout of a 32x32 MFMA: lane holds column lane & 31 and rows
// (r/4)*8 + (lane/32)*4 + r%4) through a per-wave LDS patch with a 36-word row stride, so that each lane then owns
// 16 consecutive elements of one row: lane l takes row l/2, columns (l&1)*16 .. +16, applies the epilogue and
// writes them with 16-byte stores. Everything indexed by the register array is unrolled, so the accumulators stay
// in registers; the patch is then read with 16-byte LDS loads.
constexpr int PATCH_STRIDE = 36;
constexpr int PATCH_WORDS = 32 * PATCH_STRIDE;

// Register half: copy one accumulator block into the wave's patch. Small and fully unrolled, so that the
// accumulator index is a constant and the accumulators never leave registers.
template <bool INT, typename V>
__device__ __forceinline__ void patch_put(const V& block, uint32_t* patch, int lane) {
  const int half = lane >> 5, r32 = lane & 31;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if constexpr (INT)
      patch[((r >> 2) * 8 + half * 4 + (r & 3)) * PATCH_STRIDE + r32] = (uint32_t)block[r];
    else
      patch[((r >> 2) * 8 + half * 4 + (r & 3)) * PATCH_STRIDE + r32] = __float_as_uint(block[r]);
  }
}

// Entry i of a vector of float32 (`kind` 0) or 16-bit values (1 = f16, 2 = bf16) as raw bits, and their value
__device__ __forceinline__ uint32_t vec_bits(const void* v, int kind, int64_t i) {
  return kind == 0 ? static_cast<const uint32_t*>(v)[i] : static_cast<const uint16_t*>(v)[i];
}

__device__ __forceinline__ float bits_value(int kind, uint32_t b) {
  return kind == 0 ? __uint_as_float(b) : kind == 1 ? h2f((uint16_t)b) : bf2f((uint16_t)b);
}

// Columns n .. n + 7 from raw bits, zero from N on; one branch on the kind for all eight
__device__ __forceinline__ void decode8(int kind, const uint32_t* b, int64_t n, int64_t N, float* s) {
  if (kind == 0) {
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = __uint_as_float(b[c]);
  } else if (kind == 1) {
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = h2f((uint16_t)b[c]);
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = bf2f((uint16_t)b[c]);
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) s[c] = n + c < N ? s[c] : 0.0f;
}

// The vector operands of a 32 x 32 block's epilogue, fetched ahead by every lane of the storing wave: for a per-row
// operation i the entry of the lane's row (row0 + lane / 2, as the memory half stores), for a per-column one the
// entry of column col0 + lane % 32. Every load is unconditional (a 32-bit and a 16-bit one per operation, the unused
// ones reading the valid address `dummy`) and only raw bits are kept, so that no branch merge or decode waits on
// these loads before the epilogue.
struct EpiPre {
  uint32_t w32[4], w16[4];
};

__device__ __forceinline__ void epi_prefetch(EpiPre& p, const Epilogue& e, const void* dummy, int64_t row0,
                                             int64_t col0, int64_t M, int64_t N, int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int op = e.op[i] & ((1 << VEC_KIND_SHIFT) - 1), kind = e.op[i] >> VEC_KIND_SHIFT;
    const bool row = i < e.nops && op < RELU && op % 3 == 1, col = i < e.nops && op < RELU && op % 3 == 2;
    const int64_t at = row ? min(row0 + (lane >> 1), M - 1) : col ? min(col0 + (lane & 31), N - 1) : 0;
    p.w32[i] = static_cast<const uint32_t*>((row || col) && kind == 0 ? e.vec[i] : dummy)[(row || col) && kind == 0 ? at : 0];
    p.w16[i] = static_cast<const uint16_t*>((row || col) && kind != 0 ? e.vec[i] : dummy)[(row || col) && kind != 0 ? at : 0];
  }
}

typedef u32x4 u32x4_any __attribute__((aligned(1)));  // a 16-byte access at any address

// Memory half: the patch through the epilogue to C. ACT = false: the caller has checked that no operation is an
// activation, and their code (erff, expf and a divide for each of 16 values) stays out. PRE: the vector operands
// were fetched ahead by `epi_prefetch` (one value per lane and operation) and reach the lanes that need them by
// cross-lane permutes; the whole wave must then be active. ANY: whole pieces of rows that start at no 16-byte address
// are stored with 16-byte stores all the same, instead of element by element.
template <bool INT, bool ACT = true, bool PRE = false, bool ANY = false>
__device__ __forceinline__ void patch_store_inline(uint32_t* patch, void* C, int64_t ldc, int64_t row0, int64_t col0,
                                                   int64_t M, int64_t N, const Epilogue& e, int lane,
                                                   const EpiPre* pre = nullptr) {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the patch is written before any lane reads it
  __builtin_amdgcn_wave_barrier();
  const int rr = lane >> 1, c0 = (lane & 1) * 16;
  uint32_t bits[16];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(patch + rr * PATCH_STRIDE + c0 + 4 * q);
    bits[4 * q] = w[0], bits[4 * q + 1] = w[1], bits[4 * q + 2] = w[2], bits[4 * q + 3] = w[3];
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();  // the next block may overwrite the patch
  const int64_t m = row0 + rr, n = col0 + c0;
  const bool live = m < M;
  if (!PRE && !live) return;
  const bool inside = n + 16 <= N;
  const bool whole = inside && (ldc % 8) == 0 && (uintptr_t)C % 16 == 0;
  if (INT && e.out_kind == I32) {
    if (!live) return;
    int32_t* out = static_cast<int32_t*>(C) + m * ldc + n;
    if (whole && (ldc % 4) == 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        reinterpret_cast<u32x4*>(out)[q] = u32x4{bits[4 * q], bits[4 * q + 1], bits[4 * q + 2], bits[4 * q + 3]};
    } else if (ANY && inside) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        reinterpret_cast<u32x4_any*>(out)[q] = u32x4{bits[4 * q], bits[4 * q + 1], bits[4 * q + 2], bits[4 * q + 3]};
    } else {
      for (int c = 0; c < 16 && n + c < N; ++c) out[c] = (int32_t)bits[c];
    }
    return;
  }
  float v[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) v[c] = INT ? (float)(int32_t)bits[c] : __uint_as_float(bits[c]);
  auto apply = [&](int i, auto row_value, auto col_values) {
    const int op = e.op[i] & ((1 << VEC_KIND_SHIFT) - 1);
    if (op >= RELU) {
      if constexpr (ACT) {
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = activation(op, v[c]);
      }
    } else if (op % 3 == 0) {
#pragma unroll
      for (int c = 0; c < 16; ++c) v[c] = op < 3 ? __fmul_rn(v[c], e.scalar[i]) : __fadd_rn(v[c], e.scalar[i]);
    } else if (op % 3 == 1) {
      const float s = row_value();
#pragma unroll
      for (int c = 0; c < 16; ++c) v[c] = op < 3 ? __fmul_rn(v[c], s) : __fadd_rn(v[c], s);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // eight columns at a time keeps the store's register use small
        float s[8];
        col_values(s, h * 8);
#pragma unroll
        for (int c = 0; c < 8; ++c)
          v[h * 8 + c] = op < 3 ? __fmul_rn(v[h * 8 + c], s[c]) : __fadd_rn(v[h * 8 + c], s[c]);
      }
    }
  };
  if constexpr (PRE) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i < e.nops) {
        const int kind = e.op[i] >> VEC_KIND_SHIFT;
        const uint32_t mine = kind == 0 ? pre->w32[i] : pre->w16[i];
        apply(i, [&] { return bits_value(kind, mine); }, [&](float* s, int c8) {
          uint32_t b[8];  // column n + c was fetched by lane c0 + c; all permutes out before any result is used
#pragma unroll
          for (int c = 0; c < 8; ++c) b[c] = (uint32_t)__shfl((int)mine, c0 + c8 + c);
          decode8(kind, b, n + c8, N, s);
        });
      }
    }
    if (!live) return;
  } else {
    for (int i = 0; i < e.nops; ++i) {
      const int kind = e.op[i] >> VEC_KIND_SHIFT;
      apply(i, [&] { return bits_value(kind, vec_bits(e.vec[i], kind, m)); }, [&](float* s, int c8) {
        uint32_t b[8];  // clamped indices: the loads issue back to back
#pragma unroll
        for (int c = 0; c < 8; ++c) b[c] = vec_bits(e.vec[i], kind, min(n + c8 + c, N - 1));
        decode8(kind, b, n + c8, N, s);
      });
    }
  }
  if (e.out_kind == F32) {
    float* out = static_cast<float*>(C) + m * ldc + n;
    if (whole) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        reinterpret_cast<f32x4*>(out)[q] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    } else if (ANY && inside) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        reinterpret_cast<u32x4_any*>(out)[q] =
            __builtin_bit_cast(u32x4, f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]});
    } else {
      for (int c = 0; c < 16 && n + c < N; ++c) out[c] = v[c];
    }
    return;
  }
  uint32_t h[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    h[c] = e.out_kind == BF16 ? f2bf2(v[2 * c], v[2 * c + 1])
                              : ((uint32_t)f2h(v[2 * c]) | ((uint32_t)f2h(v[2 * c + 1]) << 16));
  uint16_t* out = static_cast<uint16_t*>(C) + m * ldc + n;
  if (whole) {
    // C is written once and not read here: non-temporal stores keep it from displacing operand panels in L2
    // (bf16 8192^3 +0.3 %, fp8 +1.5 %, bf16 M = 4096 +2 %)
    __builtin_nontemporal_store(u32x4{h[0], h[1], h[2], h[3]}, reinterpret_cast<u32x4*>(out));
    __builtin_nontemporal_store(u32x4{h[4], h[5], h[6], h[7]}, reinterpret_cast<u32x4*>(out) + 1);
  } else if (ANY && inside) {  // rows of C at any alignment
    reinterpret_cast<u32x4_any*>(out)[0] = u32x4{h[0], h[1], h[2], h[3]};
    reinterpret_cast<u32x4_any*>(out)[1] = u32x4{h[4], h[5], h[6], h[7]};
  } else {
    for (int c = 0; c < 16 && n + c < N; ++c) out[c] = (uint16_t)(h[c >> 1] >> ((c & 1) * 16));
  }
}

template <bool INT>
__device__ __noinline__ void patch_store(uint32_t* patch, void* C, int64_t ldc, int64_t row0, int64_t col0, int64_t M,
                                         int64_t N, const Epilogue& e, int lane) {
  patch_store_inline<INT>(patch, C, ldc, row0, col0, M, N, e, lane);
}

// One accumulator block to C through the out-of-line store: the tiles' loops over their blocks must unroll
// completely, and an inlined store in each copy would not fit. (The skinny kernel, with at most four blocks and the
// vectors fetched ahead, inlines the store instead.)
template <bool INT, typename V>
__device__ __forceinline__ void store_block(const V& block, uint32_t* patch, void* C, int64_t ldc, int64_t row0,
                                            int64_t col0, int64_t M, int64_t N, const Epilogue& e, int lane) {
  patch_put<INT>(block, patch, lane);
  patch_store<INT>(patch, C, ldc, row0, col0, M, N, e, lane);
}

// The direct epilogue: whole 32 x 32 blocks straight from the MFMA accumulator layout to 16-bit C, without the LDS
// patch, for epilogues of at most two operations that are float32 scalars or row/column vectors (no activation):
// the headline bf16 product, the fp8 product's `acc * (scale_a * scale_b)`, the W8A8 dequantisation
// `acc * scale_a[m] * scale_w[n]`. Lane L holds column c = L & 31 at rows R(r) = (r / 4) * 8 + (L / 32) * 4 + r % 4;
// neighbouring lanes hold columns c and c ^ 1 of the same rows. The operations and their rounding are the patch
// path's, so the result is the same bit for bit.
constexpr int DIRECT_OPS = 2;

__device__ __forceinline__ bool direct_epilogue(const Epilogue& e) {
  if (e.out_kind != BF16 && e.out_kind != F16) return false;
  if (e.nops > DIRECT_OPS) return false;
  for (int i = 0; i < e.nops; ++i)
    if ((e.op[i] & ((1 << VEC_KIND_SHIFT) - 1)) >= RELU) return false;
  return true;
}

// The vector operands of a wave's TM x TN blocks, fetched for all blocks at once before any is stored: for a per-row
// operation the 16 rows R(r) of each row block, for a per-column one the lane's column of each column block.
template <int TM, int TN>
struct DirectVectors {
  float row[DIRECT_OPS][TM][16];
  float col[DIRECT_OPS][TN];
};

template <int TM, int TN>
__device__ __forceinline__ void direct_vectors(DirectVectors<TM, TN>& dv, const Epilogue& e, int64_t row0,
                                               int64_t col0, int lane) {
  const int c = lane & 31, half = lane >> 5;
#pragma unroll
  for (int q = 0; q < DIRECT_OPS; ++q) {
    if (q >= e.nops) break;
    const int op = e.op[q] & ((1 << VEC_KIND_SHIFT) - 1), kind = e.op[q] >> VEC_KIND_SHIFT;
    // every element is assigned on every path, so the arrays stay in registers
    const bool per_row = op % 3 == 1, per_col = op % 3 == 2;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        dv.row[q][i][r] =
            per_row ? bits_value(kind, vec_bits(e.vec[q], kind, row0 + i * 32 + (r >> 2) * 8 + half * 4 + (r & 3)))
                    : 0.0f;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      dv.col[q][j] = per_col ? bits_value(kind, vec_bits(e.vec[q], kind, col0 + j * 32 + c)) : 0.0f;
  }
}

// One block's 16 accumulators through the epilogue operations, in float32 (the patch path's operations and
// rounding).
template <bool INT, int TM, int TN, typename V>
__device__ __forceinline__ void direct_ops(float (&v)[16], const V& block, const DirectVectors<TM, TN>& dv, int i,
                                           int j, const Epilogue& e) {
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = INT ? (float)(int32_t)block[r] : (float)block[r];
#pragma unroll
  for (int q = 0; q < DIRECT_OPS; ++q) {
    if (q >= e.nops) break;
    const int op = e.op[q] & ((1 << VEC_KIND_SHIFT) - 1);
    const bool mul = op < 3;
    if (op % 3 == 0) {
      const float s = e.scalar[q];
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = mul ? __fmul_rn(v[r], s) : __fadd_rn(v[r], s);
    } else if (op % 3 == 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = mul ? __fmul_rn(v[r], dv.row[q][i][r]) : __fadd_rn(v[r], dv.row[q][i][r]);
    } else {
      const float s = dv.col[q][j];
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = mul ? __fmul_rn(v[r], s) : __fadd_rn(v[r], s);
    }
  }
}

// One block (i, j): one DPP swap per register pair (2k, 2k + 1) gives the even lane both columns c, c + 1 of row
// R(2k) and the odd lane both of row R(2k + 1); each store instruction writes 64-byte row segments (half lines).
template <bool INT, bool BF, int TM, int TN, typename V>
__device__ __forceinline__ void store_block_direct(const V& block, const DirectVectors<TM, TN>& dv, int i, int j,
                                                   __amdgpu_buffer_rsrc_t out, uint32_t lane_off, int64_t ldc,
                                                   const Epilogue& e, int lane) {
  float v[16];
  direct_ops<INT>(v, block, dv, i, j, e);
  const int odd = lane & 1;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float send = odd ? v[2 * k] : v[2 * k + 1];
    const float recv = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), 0xB1, 0xF, 0xF, true));
    const float lo = odd ? recv : v[2 * k], hi = odd ? v[2 * k + 1] : recv;
    const uint32_t pair = BF ? f2bf2(lo, hi) : ((uint32_t)f2h(lo) | ((uint32_t)f2h(hi) << 16));
    // register 2k + odd holds row ((2k + odd) >> 2) * 8 + half * 4 + ((2k + odd) & 3): the lane's part
    // (half * 4 + odd) is in lane_off, the rest is a scalar offset
    const int step = (k >> 1) * 8 + (k & 1) * 2 + i * 32;
    const int soff = __builtin_amdgcn_readfirstlane((int)(((int64_t)step * ldc + j * 32) * 2));
    __builtin_amdgcn_raw_buffer_store_b32(pair, out, (int)lane_off, soff, 2 /* nt */);
  }
}

// A wave's TM x TN accumulator blocks to C. When the wave's whole region lies inside C and the epilogue is one the
// direct path takes, every block goes straight from registers; otherwise each block goes through the LDS patch (all
// operations, ragged edges, int32 and float32 outputs).

// A block of accumulators held in AGPRs (the four-wave loop's 256 of them), copied to VGPRs right before it is
// stored, by ordered reads; left to itself the compiler copies all of them at the end of the loop and spills most of
// them to private memory.
template <typename V>
__device__ __forceinline__ V agpr_block(const V& x) {
  V y;
#pragma unroll
  for (int r = 0; r < (int)(sizeof(V) / 4); ++r)
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(y[r]) : "a"(x[r]) : "memory");
  return y;
}

// `fetch(i, j)` hands over block (i, j) in the 32x32 accumulator layout.
template <bool INT, int TM, int TN, typename Fetch>
__device__ __forceinline__ void store_tile_by(Fetch fetch, uint32_t* patch, void* C, int64_t ldc, int64_t row0,
                                              int64_t col0, int64_t M, int64_t N, const Epilogue& e, int lane) {
  const bool direct = direct_epilogue(e) && (ldc % 2) == 0 && (uintptr_t)C % 4 == 0 && row0 + 32 * TM <= M &&
                      col0 + 32 * TN <= N && (int64_t)32 * TM * ldc * 2 <= 0x7fffffff;
  if (direct) {
    DirectVectors<TM, TN> dv;
    direct_vectors(dv, e, row0, col0, lane);
    // the wave's region of C as a buffer resource; each lane stores a column pair at (c & ~1) of rows
    // half * 4 + odd, plus wave-uniform steps
    const int c = lane & 31;
    // (readfirstlane returns int: each word goes through uint32_t, so the low word is never sign-extended into
    // the high one)
    const uint64_t base = (uint64_t)(static_cast<uint16_t*>(C) + row0 * ldc + col0);
    const uint32_t base_lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)base);
    const uint32_t base_hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
    const void* region = (const void*)(((uint64_t)base_hi << 32) | (uint64_t)base_lo);
    const __amdgpu_buffer_rsrc_t out = panel_rsrc(region, (int64_t)32 * TM * ldc * 2);
    // block by block: row half * 4 + (c & 1), column pair c & ~1 (measured 3 % faster for W8A8 on the eight-wave
    // int8 loop, whose registers are tighter, than pairs of blocks stored as whole lines)
    const uint32_t lane_off = (uint32_t)((((lane >> 5) * 4 + (c & 1)) * ldc + (c & ~1)) * 2);
#define KRN_DIRECT(BF)                                                                                       \
  _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int j = 0; j < TN; ++j)              \
      store_block_direct<INT, BF>(fetch(i, j), dv, i, j, out, lane_off, ldc, e, lane);
    if (e.out_kind == BF16) {
      KRN_DIRECT(true)
    } else {
      KRN_DIRECT(false)
    }
#undef KRN_DIRECT
    return;
  }
  // The out-of-line store takes the epilogue by address. Passing the kernel argument itself would copy it to private
  // memory at kernel entry, in every wave, whichever path the wave takes (80 bytes a lane, 42 MB per bf16 8192^3
  // launch); this copy is made only on this path.
  const Epilogue local = e;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) store_block<INT>(fetch(i, j), patch, C, ldc, row0 + i * 32, col0 + j * 32, M, N, local, lane);
}

template <bool INT, int TM, int TN, typename Acc>
__device__ __forceinline__ void store_tile(const Acc (&acc)[TM][TN], uint32_t* patch, void* C, int64_t ldc,
                                           int64_t row0, int64_t col0, int64_t M, int64_t N, const Epilogue& e,
                                           int lane) {
  store_tile_by<INT, TM, TN>([&](int i, int j) { return acc[i][j]; }, patch, C, ldc, row0, col0, M, N, e, lane);
}

// Register half of the patch path for a block held transposed: `block` is the 32x32 accumulator layout of the
// transpose of a C block (lane holds C row lane & 31 and C columns (r/4)*8 + (lane/32)*4 + r%4), written into the
// patch in C's row-major order.
template <bool INT, typename V>
__device__ __forceinline__ void patch_put_t(const V& block, uint32_t* patch, int lane) {
  const int half = lane >> 5, r32 = lane & 31;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t bits = INT ? (uint32_t)block[r] : __float_as_uint(block[r]);
    patch[r32 * PATCH_STRIDE + (r >> 2) * 8 + half * 4 + (r & 3)] = bits;
  }
}

// The four-wave loop's 8 x 8 blocks of 16 x 16, computed transposed (B A^T, so that C's rows lie along the lanes):
// lane L of block (i, j) holds row 16 i + (L & 15) of the wave's 128 x 128 region and its columns
// 16 j + 4 (L >> 4) .. + 3, one per register. The four lanes L & 15 + 16 s that share a row exchange 8-byte pieces
// (two permlane swaps per word), so that each holds 16 contiguous columns of one block and writes them as two
// 16-byte pieces: per store instruction 64 bytes of each of 16 rows. The untransposed 32x32 layout needs a DPP
// exchange and three selects per register for whole-line pieces; 8-byte pieces without the exchange were slower
// (quarter lines). `ops` applies the epilogue's operations to one block's four values (Quad16Generic,
// Quad16RowCol below), with the patch path's rounding. 32-bit outputs have their own direct store
// (store32t_direct); everything else (ragged edges, activations, more than two operations) goes through the patch:
// four blocks are joined into the 32x32 layout of the transposed block and written into the patch transposed.
// Against the 32x32 direct store (same box, bench legs): bf16 8192^3 equal, fp8 8192^3 0.440 -> 0.424 ms,
// W8A8 M = 4096 0.272 -> 0.247 ms; write-back instead of non-temporal stores: bf16 1.5 % slower.
template <bool INT, bool BF, typename V4, typename Ops>
__device__ __forceinline__ void store16t_direct(const V4 (&acc)[8][8], Ops ops, void* C, int64_t ldc, int64_t row0,
                                                int64_t col0, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const uint64_t base = (uint64_t)(static_cast<uint16_t*>(C) + row0 * ldc + col0);
  const uint32_t base_lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)base);
  const uint32_t base_hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
  const void* region = (const void*)(((uint64_t)base_hi << 32) | (uint64_t)base_lo);
  const __amdgpu_buffer_rsrc_t out = panel_rsrc(region, (int64_t)128 * ldc * 2);
  // after the exchange below, lane group g holds the 16 columns of block 4 jj + g of its row: two 16-byte pieces
  const uint32_t lane_off = (uint32_t)((r16 * ldc + 16 * g) * 2);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      uint32_t w[4][2];  // [block jb][word]: columns 16 (4 jj + jb) + 4 g + 2 word .. + 1
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        const int j = 4 * jj + jb;
        const V4 b = agpr_block(acc[i][j]);
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = INT ? (float)(int32_t)b[c] : (float)b[c];
        ops(v, i, j);
        w[jb][0] = BF ? f2bf2(v[0], v[1]) : ((uint32_t)f2h(v[0]) | ((uint32_t)f2h(v[1]) << 16));
        w[jb][1] = BF ? f2bf2(v[2], v[3]) : ((uint32_t)f2h(v[2]) | ((uint32_t)f2h(v[3]) << 16));
      }
      // a 4 x 4 transpose of 8-byte pieces over the four lane groups (16-lane rows) that share a C row: piece
      // (group s, block jb) goes to group jb, slot s. permlane16_swap(x, y) leaves [x0 y0 x2 y2] in x and
      // [x1 y1 x3 y3] in y (16-lane rows), permlane32_swap(x, y) [x0 x1 y0 y1] and [x2 x3 y2 y3].
      uint32_t t[4][2];  // [slot s][word]: columns 16 (4 jj + g) + 4 s + 2 word .. + 1
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const auto p01 = __builtin_amdgcn_permlane16_swap(w[0][x], w[1][x], false, false);
        const auto p23 = __builtin_amdgcn_permlane16_swap(w[2][x], w[3][x], false, false);
        const auto q02 = __builtin_amdgcn_permlane32_swap(p01[0], p23[0], false, false);
        const auto q13 = __builtin_amdgcn_permlane32_swap(p01[1], p23[1], false, false);
        t[0][x] = q02[0];
        t[2][x] = q02[1];
        t[1][x] = q13[0];
        t[3][x] = q13[1];
      }
      const int soff = __builtin_amdgcn_readfirstlane((int)(((int64_t)16 * i * ldc + 64 * jj) * 2));
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{t[0][0], t[0][1], t[1][0], t[1][1]}, out, (int)lane_off, soff,
                                             2 /* nt */);
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{t[2][0], t[2][1], t[3][0], t[3][1]}, out, (int)lane_off + 16,
                                             soff, 2 /* nt */);
    }
}

// The direct store's operations on one block's four values (row 16 i + (lane & 15), columns 16 j + 4 (lane >> 4)
// + c). Generic: any chain of at most two scalar, row and column multiplies and adds, as two fused multiply-adds
// each (x * s + (-0) = x * s or x * 1 + s = x + s, and the identity x * 1 + (-0) for the other of the pair: each exact
// or rounded once, signed zeros included, so the result is the patch path's bit for bit).
struct Quad16Generic {
  float rm[DIRECT_OPS][8], ra[DIRECT_OPS][8], cm[DIRECT_OPS][8][4], ca[DIRECT_OPS][8][4];
  int nops;
  __device__ void operator()(float (&v)[4], int i, int j) const {
#pragma unroll
    for (int q = 0; q < DIRECT_OPS; ++q) {
      if (q >= nops) break;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        v[c] = __builtin_fmaf(__builtin_fmaf(v[c], rm[q][i], ra[q][i]), cm[q][j][c], ca[q][j][c]);
    }
  }
};

__device__ __forceinline__ void quad16_generic(Quad16Generic& qv, const Epilogue& e, int64_t row0, int64_t col0,
                                               int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  qv.nops = e.nops;
  // per operation: the multiplier and addend of a fused multiply-add per row block (row and scalar operations) and
  // per column of each column block (column operations); the other of the two is the identity x * 1 + (-0), exact
  // for every x, so each operation is two fused multiply-adds and no selection
#pragma unroll
  for (int q = 0; q < DIRECT_OPS; ++q) {
    if (q >= e.nops) break;
    const int op = e.op[q] & ((1 << VEC_KIND_SHIFT) - 1), kind = e.op[q] >> VEC_KIND_SHIFT;
    const bool mul = op < 3, col = op % 3 == 2;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float s = col ? bits_value(kind, vec_bits(e.vec[q], kind, col0 + 16 * j + 4 * g + c)) : 0.0f;
        qv.cm[q][j][c] = col && mul ? s : 1.0f;
        qv.ca[q][j][c] = col && !mul ? s : -0.0f;
      }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float s = col ? 0.0f
                          : op % 3 == 1 ? bits_value(kind, vec_bits(e.vec[q], kind, row0 + 16 * i + r16)) : e.scalar[q];
      qv.rm[q][i] = !col && mul ? s : 1.0f;
      qv.ra[q][i] = !col && !mul ? s : -0.0f;
    }
  }
}

// W8A8's dequantisation `acc * scale_a[m] * scale_w[n]` (a row multiply, then a column multiply, float32 vectors):
// the lane's 8 row and 32 column values, fetched before the loop's last slices, and two multiplies per value.
struct Quad16RowCol {
  float r[8], c[8][4];
  __device__ void operator()(float (&v)[4], int i, int j) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = __fmul_rn(__fmul_rn(v[q], r[i]), c[j][q]);
      // opaque to the compiler, which would otherwise fuse the last multiply into the f16 conversion (a mixed
      // multiply-add with a +0 addend, rounded once: -0 becomes +0 and the float32 rounding is skipped)
      asm("" : "+v"(v[q]));
    }
  }
};

__device__ __forceinline__ bool quad16_is_rowcol(const Epilogue& e) {
  return e.nops == 2 && e.op[0] == MUL_ROW && e.op[1] == MUL_COL;  // kind 0: float32 vectors
}

__device__ __forceinline__ void quad16_rowcol(Quad16RowCol& rc, const Epilogue& e, int64_t row0, int64_t col0,
                                              int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const float* rv = static_cast<const float*>(e.vec[0]);
  const float* cv = static_cast<const float*>(e.vec[1]);
#pragma unroll
  for (int i = 0; i < 8; ++i) rc.r[i] = rv[row0 + 16 * i + r16];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int c = 0; c < 4; ++c) rc.c[j][c] = cv[col0 + 16 * j + 4 * g + c];
}

// Whether a wave's 128 x 128 region at (row0, col0) takes the direct store.
__device__ __forceinline__ bool quad16_direct(const Epilogue& e, const void* C, int64_t ldc, int64_t row0,
                                              int64_t col0, int64_t M, int64_t N) {
  return direct_epilogue(e) && (ldc % 4) == 0 && (uintptr_t)C % 8 == 0 && row0 + 128 <= M && col0 + 128 <= N &&
         (int64_t)128 * ldc * 2 <= 0x7fffffff;
}

// 32-bit outputs (int32 from an int8 product with no operations, float32 with at most two scalar, row and column
// operations) of the transposed blocks: a lane's four values are 16 contiguous bytes of one row, so each block is
// one 16-byte store per lane (64 bytes of each of 16 rows per instruction), no exchange between lanes.
__device__ __forceinline__ bool quad16_direct32(const Epilogue& e, const void* C, int64_t ldc, int64_t row0,
                                                int64_t col0, int64_t M, int64_t N) {
  bool ops_ok = e.nops <= DIRECT_OPS;
  for (int i = 0; i < e.nops; ++i) ops_ok &= (e.op[i] & ((1 << VEC_KIND_SHIFT) - 1)) < RELU;
  const bool kind = (e.out_kind == I32 && e.nops == 0) || (e.out_kind == F32 && ops_ok);
  return kind && (ldc % 4) == 0 && (uintptr_t)C % 16 == 0 && row0 + 128 <= M && col0 + 128 <= N &&
         (int64_t)128 * ldc * 4 <= 0x7fffffff;
}

template <bool INT, typename V4, typename Ops>
__device__ __forceinline__ void store32t_direct(const V4 (&acc)[8][8], Ops ops, bool raw_int, void* C, int64_t ldc,
                                                int64_t row0, int64_t col0, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const uint64_t base = (uint64_t)(static_cast<uint32_t*>(C) + row0 * ldc + col0);
  const uint32_t base_lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)base);
  const uint32_t base_hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
  const void* region = (const void*)(((uint64_t)base_hi << 32) | (uint64_t)base_lo);
  const __amdgpu_buffer_rsrc_t out = panel_rsrc(region, (int64_t)128 * ldc * 4);
  const uint32_t lane_off = (uint32_t)((r16 * ldc + 4 * g) * 4);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const V4 b = agpr_block(acc[i][j]);
      u32x4 w;
      if (INT && raw_int) {
#pragma unroll
        for (int c = 0; c < 4; ++c) w[c] = (uint32_t)b[c];
      } else {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = INT ? (float)(int32_t)b[c] : (float)b[c];
        ops(v, i, j);
#pragma unroll
        for (int c = 0; c < 4; ++c) w[c] = __float_as_uint(v[c]);
      }
      const int soff = __builtin_amdgcn_readfirstlane((int)(((int64_t)16 * i * ldc + 16 * j) * 4));
      __builtin_amdgcn_raw_buffer_store_b128(w, out, (int)lane_off, soff, 2 /* nt */);
    }
}

// `direct`: quad16_direct of the region; `rowcol`: the epilogue is W8A8's, with its vectors already in `rc`.
template <bool INT, typename V16, typename V4>
__device__ __forceinline__ void store_tile16t(const V4 (&acc)[8][8], bool direct, bool rowcol,
                                              const Quad16RowCol& rc, uint32_t* patch, void* C, int64_t ldc,
                                              int64_t row0, int64_t col0, int64_t M, int64_t N, const Epilogue& e,
                                              int lane) {
  if (direct) {
    const bool bf = e.out_kind == BF16;
    if (rowcol) {
      if (bf) store16t_direct<INT, true>(acc, rc, C, ldc, row0, col0, lane);
      else store16t_direct<INT, false>(acc, rc, C, ldc, row0, col0, lane);
    } else {
      Quad16Generic qv;
      quad16_generic(qv, e, row0, col0, lane);
      if (bf) store16t_direct<INT, true>(acc, qv, C, ldc, row0, col0, lane);
      else store16t_direct<INT, false>(acc, qv, C, ldc, row0, col0, lane);
    }
    return;
  }
  if (quad16_direct32(e, C, ldc, row0, col0, M, N)) {
    Quad16Generic qv;
    quad16_generic(qv, e, row0, col0, lane);
    store32t_direct<INT>(acc, qv, e.out_kind == I32, C, ldc, row0, col0, lane);
    return;
  }
  const Epilogue local = e;  // taken by address by the out-of-line store
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // the transposed 32x32 block's quarter (h, k) is the transpose of C's quarter (k, h)
      const V16 blk = join16<V16>(agpr_block(acc[2 * i][2 * j]), agpr_block(acc[2 * i + 1][2 * j]),
                                  agpr_block(acc[2 * i][2 * j + 1]), agpr_block(acc[2 * i + 1][2 * j + 1]));
      patch_put_t<INT>(blk, patch, lane);
      patch_store<INT>(patch, C, ldc, row0 + 32 * i, col0 + 32 * j, M, N, local, lane);
    }
}

// 16 bytes of row `base` starting at byte `kb`, zero past the row's end or for a row outside the matrix. VEC: the
// row is 16-byte aligned and its length a multiple of 16, so one dwordx4 load does it.
template <bool VEC>
__device__ __forceinline__ u32x4 load16(const uint8_t* __restrict__ p, int64_t base, int64_t kb, bool inside,
                                        int64_t kbytes) {
  if constexpr (VEC) {
    return (inside && kb < kbytes) ? *reinterpret_cast<const u32x4*>(p + base + kb) : u32x4{};
  } else {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t v = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int64_t at = kb + i * 4 + b;
        v |= (inside && at < kbytes) ? (uint32_t)p[base + at] << (8 * b) : 0u;
      }
      w[i] = v;
    }
    return u32x4{w[0], w[1], w[2], w[3]};
  }
}

// LDS swizzles. gfx950's LDS serves 16 lanes of a 16-byte read per cycle from 64 banks (256 bytes), so the 16
// rows a read touches must land on 16 different 16-byte positions modulo 256 bytes. With 128-byte rows (8 chunks)
// rows of equal parity share a window half, so chunk c of row r goes to slot c ^ ((r >> 1) & 7); with 64-byte rows
// (4 chunks) rows of equal r & 3 share a quarter, so slot c ^ ((r >> 2) & 3).
__device__ __forceinline__ int swz8(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int swz4(int row) { return (row >> 2) & 3; }

// Tile index of this workgroup. Workgroups are dispatched round-robin over the 8 XCDs, so consecutive ids are
// first regrouped per XCD (each XCD gets one contiguous range of tiles and its own L2 sees a compact panel), then
// ordered in groups of GROUP_M tile rows so neighbours share A rows and B columns.
__device__ __forceinline__ void tile_of(int tiles_m, int tiles_n, int& tm, int& tn) {
#ifndef KRN_GROUP_M
#define KRN_GROUP_M 4
#endif
#ifndef KRN_XCD_REMAP
#define KRN_XCD_REMAP 1
#endif
  constexpr int GROUP_M = KRN_GROUP_M;  // bf16 8192^3, eight-wave ring: 0.5-1.5 % faster than 8 (2: -6 %, 6: -1 %,
                                        // 16: -9 %); fp8 equal; four-wave register-staged 32x32 loop: 8 equal, 2
                                        // -1.5 % (1.5 times the bytes read)
  int nb = tiles_m * tiles_n;
  int bid = blockIdx.x;
  if (KRN_XCD_REMAP && nb % 8 == 0) bid = (bid % 8) * (nb / 8) + bid / 8;
  int per_group = GROUP_M * tiles_n;
  int group = bid / per_group;
  int first = group * GROUP_M;
  int size = min(tiles_m - first, GROUP_M);
  int local = bid % per_group;
  tm = first + local % size;
  tn = local / size;
}

}  // namespace krn
