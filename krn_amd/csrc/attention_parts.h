// What the attention kernels share: the 16-bit formats with their MFMA step, the LDS layouts of K and V tiles, and the
// launch of the key-split kernel.
#pragma once
#include "common.h"

namespace krn {

typedef short v4s __attribute__((ext_vector_type(4)));

template <bool BF>
struct Half;
template <>
struct Half<true> {
  __device__ static uint32_t pack(float lo, float hi) {
    return f2bf2(lo, hi);  // v_cvt_pk_bf16_f32, nearest even
  }
  __device__ static uint16_t from(float x) { return f2bf(x); }
  __device__ static void mma(f32x16& c, u32x4 a, u32x4 b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                0, 0);
  }
};
template <>
struct Half<false> {
  __device__ static uint32_t pack(float lo, float hi) { return (uint32_t)f2h(lo) | ((uint32_t)f2h(hi) << 16); }
  __device__ static uint16_t from(float x) { return f2h(x); }
  __device__ static void mma(f32x16& c, u32x4 a, u32x4 b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                               0);
  }
};

// LDS swizzles of the [key][d] tiles (64 banks serve 256 bytes per cycle). K: the 16-byte reads of 16 consecutive
// keys must hit 16 distinct positions modulo 256 bytes. V: the transposed 8-byte reads cover 4 consecutive keys x
// 64 bytes per 32 lanes. D = 128 (256-byte rows) and D = 64 (128-byte rows) need different XOR patterns.
template <int D>
__device__ __forceinline__ int k_slot(int key, int chunk) {
  return D == 128 ? chunk ^ (key & 15) : chunk ^ ((key >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int v_slot(int key, int chunk) {
  return D == 128 ? chunk ^ ((key & 3) << 2) : chunk ^ (((key >> 1) & 1) << 2);
}

// max(x, x of lane ^ 32): the two lanes that hold one query row (v_permlane32_swap, no LDS round trip). One
// v_max_f32 (written as assembly: as fmaxf the compiler first quiets both operands, two more VALU instructions; the
// instruction quiets a signaling NaN itself, and these operands are arithmetic results or swaps of them).
__device__ __forceinline__ float pair_max(float x) {
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  float y;
  asm("v_max_f32 %0, %1, %2" : "=v"(y) : "v"(__uint_as_float(sw[0])), "v"(__uint_as_float(sw[1])));
  return y;
}

// The key-split kernel (attention_split.hip): workgroups of 32 query rows whose four waves, and `parts` workgroups,
// share the keys. parts > 1 needs `workspace` for the parts' unnormalised rows (split_bytes).
struct AttentionCall {
  const void *q, *k, *v;
  void *o, *workspace;
  int64_t bh, sq, sk;
  float scale;
  int causal, parts;
  hipStream_t stream;
};

inline int64_t attention_split_rows(int64_t sq) { return sq < 32 ? sq : (sq + 31) / 32 * 32; }  // rows kept per head
inline int64_t attention_split_bytes(int64_t bh, int64_t sq, int64_t d, int parts) {
  return parts > 1 ? bh * attention_split_rows(sq) * parts * (d + 2) * 4 : 0;
}

int launch_attention_split(bool bf, int d, const AttentionCall& c);

}  // namespace krn
