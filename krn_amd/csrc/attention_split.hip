// Flash attention forward for launches that would leave most of the chip idle in attention.hip: decoding (one or a few
// queries per head against a long cache) and short prompts of few heads. There a workgroup owns 256 query rows and
// walks all keys: one query per head and 128 heads are 128 workgroups, seven of their eight waves without a row, and
// 4096 keys run one after the other (109 us for 268 MB of K and V).
//
// Here a workgroup owns 32 query rows, and its four waves take a quarter of its keys each; with `parts` > 1 several
// workgroups share the keys of one row block as well. Every wave runs the online softmax of attention.hip on its own
// keys (S^T = K Q^T, O^T += V^T P^T, lazy rescale), the waves' (m, sum, O) meet in LDS, and the parts' in a workspace
// that a second kernel reduces. What bounds it is the stream of K and V: each wave moves 32-key tiles into an LDS ring
// of its own with direct-to-LDS loads of whole lines, the next tile in flight while one multiplies, and no barrier
// runs in the loop. The transposed V reads are one assembly block with their wait: as builtins the compiler waits for
// the tile in flight before them.
#include "attention_parts.h"

namespace krn {

constexpr int SPLIT_WAVES = 4;
constexpr uint32_t OUTSIDE_HEAD = 0x80000000u;  // an offset past every buffer resource (at most 2^31 - 1 bytes)

// the V^T fragments of one 32-wide block of d: [step][part], each four keys of this lane's d column
template <int D>
__device__ __forceinline__ void v_fragments(uint32_t at, u32x4 (&va)[2]) {
  u32x2 w[4];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %4 offset:%5\n\t"
      "ds_read_b64_tr_b16 %2, %4 offset:%6\n\tds_read_b64_tr_b16 %3, %4 offset:%7\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3])
      : "v"(at), "n"(8 * D * 2), "n"(16 * D * 2), "n"(24 * D * 2)
      : "memory");
  va[0] = u32x4{w[0][0], w[0][1], w[1][0], w[1][1]};
  va[1] = u32x4{w[2][0], w[2][1], w[3][0], w[3][1]};
}

template <bool BF, int D, bool ONCE>
__global__ __launch_bounds__(64 * SPLIT_WAVES, 2) void attention_split(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V,
    uint16_t* __restrict__ O, float* __restrict__ planes, int64_t sq, int64_t sk, float scale, int q_tiles, int causal,
    int parts, int heads) {
  constexpr int DCH = D / 8, TILE = 32 * D * 2, ROWS_PER_LOAD = 1024 / (D * 2), LOADS = 32 / ROWS_PER_LOAD;
  constexpr int STAGE = 2 * TILE, RING = 2 * STAGE;  // K and V of 32 keys, two stages per wave
  constexpr int OLD = D + 4;                         // floats per row of a wave's O in LDS
  static_assert(32 * OLD * 4 <= RING, "a wave's O fits its ring");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[SPLIT_WAVES * RING];
  __shared__ float stat[2][SPLIT_WAVES][32];  // m and sum of every wave's rows

  // all blocks of a head on one XCD when heads is a multiple of 8; late query tiles, the long ones under a causal
  // mask, first
  const int head = (int)(blockIdx.x % heads), rest = (int)(blockIdx.x / heads);
  const int part = rest % parts, qt = q_tiles - 1 - rest / parts;
  const int64_t q0 = (int64_t)qt * 32;
  const int t = threadIdx.x, lane = t & 63, half = lane >> 5, r32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint16_t* q = Q + (int64_t)head * sq * D;
  const __amdgpu_buffer_rsrc_t k_rsrc = panel_rsrc(K + (int64_t)head * sk * D, sk * D * 2),
                              v_rsrc = panel_rsrc(V + (int64_t)head * sk * D, sk * D * 2);
  uint8_t* ring = lds + wave * RING;

  const int64_t qrow = q0 + r32;
  u32x4 qf[D / 16];
#pragma unroll
  for (int s = 0; s < D / 16; ++s)
    qf[s] = qrow < sq ? *reinterpret_cast<const u32x4*>(q + qrow * D + s * 16 + half * 8) : u32x4{};

  // this wave's 32-key tiles
  const int64_t kend = causal ? min(sk, q0 + 32) : sk;
  const int tiles = (int)((kend + 31) / 32), units = parts * SPLIT_WAVES, unit = part * SPLIT_WAVES + wave;
  const int first = (int)((int64_t)tiles * unit / units), n = (int)((int64_t)tiles * (unit + 1) / units) - first;

  uint32_t koff[LOADS], voff[LOADS];  // byte offsets within a tile
  const int lrow = lane / DCH, lslot = lane % DCH;
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int row = j * ROWS_PER_LOAD + lrow;
    koff[j] = (uint32_t)(row * D + k_slot<D>(row, lslot) * 8) * 2;
    voff[j] = (uint32_t)(row * D + v_slot<D>(row, lslot) * 8) * 2;
  }
  // tile i of this wave into stage `st`; rows past the last key are zeros
  auto load = [&](int i, uint8_t* st) {
    const int key0 = (first + i) * 32, soff = key0 * D * 2;
    const bool ragged = key0 + 32 > sk;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const bool out = ragged && key0 + j * ROWS_PER_LOAD + lrow >= sk;
      buffer_to_lds16<ONCE>(k_rsrc, st + j * 1024, out ? OUTSIDE_HEAD : koff[j], soff);
      buffer_to_lds16<ONCE>(v_rsrc, st + TILE + j * 1024, out ? OUTSIDE_HEAD : voff[j], soff);
    }
  };

  f32x16 acc[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) acc[i] = f32x16{};
  float m = -1.0e30f, total = 0.0f;
  // V^T fragment addresses: lane group g = lane / 16 reads keys 4 (g / 2) + (lane % 16) / 4 at d columns
  // 16 (g % 2) + 4 (lane % 4) of each 32-wide block
  const int g = lane >> 4, a16 = lane & 15, tr_key = (g >> 1) * 4 + (a16 >> 2), tr_col = (g & 1) * 16 + 4 * (a16 & 3);
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)ring;
  const int64_t row_limit = causal ? qrow : (int64_t)1 << 62;

  if (n > 0) load(0, ring);
  for (int i = 0; i < n; ++i) {
    const int stage = (i & 1) * STAGE;
    if (i + 1 < n) {
      load(i + 1, ring + (STAGE - stage));  // its last reads were waited for by the MFMAs that used them
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const u32x4* kl = reinterpret_cast<const u32x4*>(ring + stage);
    f32x16 s = f32x16{};
#pragma unroll
    for (int j = 0; j < D / 16; ++j) Half<BF>::mma(s, kl[r32 * DCH + k_slot<D>(r32, j * 2 + half)], qf[j]);

    const int64_t c0 = (int64_t)(first + i) * 32;
    const bool masked = c0 + 32 > sk || (causal && c0 + 31 > q0);
    float tmax = -INFINITY;
    if (masked) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t key = c0 + half * 4 + (r >> 2) * 8 + (r & 3);
        float x = s[r] * scale;
        if (key > row_limit) x = -1.0e30f;
        if (key >= sk) x = -INFINITY;  // an invalid lane: no part in maximum, sum or product
        s[r] = x;
        tmax = fmaxf(tmax, x);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[r] * scale);
    }
    tmax = pair_max(tmax);
    if (__builtin_amdgcn_ballot_w64(tmax > m + 8.0f) != 0) {  // the lazy rescale of attention.hip
      const float m_new = fmaxf(m, tmax), corr = __builtin_amdgcn_exp2f(m - m_new);
      total *= corr;
#pragma unroll
      for (int b = 0; b < D / 32; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] *= corr;
      m = m_new;
    }
    const float sc = masked ? 1.0f : scale, neg_m = -m;
    u32x4 pf[2];
    float psum = 0.0f;
#pragma unroll
    for (int step = 0; step < 2; ++step)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[step * 8 + 2 * j], sc, neg_m));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[step * 8 + 2 * j + 1], sc, neg_m));
        psum += p0 + p1;
        pf[step][j] = Half<BF>::pack(p0, p1);
      }
    total += psum;
#pragma unroll
    for (int b = 0; b < D / 32; ++b) {
      const int col = b * 32 + tr_col;
      u32x4 va[2];
      v_fragments<D>(ring_at + stage + TILE + tr_key * (D * 2) + v_slot<D>(tr_key, col >> 3) * 16 + (col & 7) * 2, va);
      Half<BF>::mma(acc[b], va[0], pf[0]);
      Half<BF>::mma(acc[b], va[1], pf[1]);
    }
  }

  // the row sum over both halves of the wave, then the waves' rows meet in LDS
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(total), __float_as_uint(total), false, false);
    total = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  if (half == 0) stat[0][wave][r32] = m, stat[1][wave][r32] = total;
  float* mine = reinterpret_cast<float*>(ring);
#pragma unroll
  for (int b = 0; b < D / 32; ++b)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq)
      *reinterpret_cast<f32x4*>(mine + r32 * OLD + b * 32 + gq * 8 + half * 4) =
          f32x4{acc[b][gq * 4], acc[b][gq * 4 + 1], acc[b][gq * 4 + 2], acc[b][gq * 4 + 3]};
  __syncthreads();
  const int rows = (int)min((int64_t)32, sq - q0);
  const int64_t kept = sq < 32 ? sq : (int64_t)q_tiles * 32;  // rows per head of a plane
  float* plane = planes + ((int64_t)part * heads + head) * kept * (D + 2);
  for (int at = t; at < rows * (D / 4); at += 64 * SPLIT_WAVES) {
    const int row = at / (D / 4), d = at % (D / 4) * 4;
    float top = stat[0][0][row];
#pragma unroll
    for (int w = 1; w < SPLIT_WAVES; ++w) top = fmaxf(top, stat[0][w][row]);
    float sum = 0.0f;
    f32x4 o = f32x4{};
#pragma unroll
    for (int w = 0; w < SPLIT_WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(stat[0][w][row] - top);
      sum += f * stat[1][w][row];
      o += f * *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(lds + w * RING) + row * OLD + d);
    }
    if (parts > 1) {  // unnormalised rows, then their maxima and sums
      *reinterpret_cast<f32x4*>(plane + (q0 + row) * D + d) = o;
      if (d == 0) plane[kept * D + (q0 + row) * 2] = top, plane[kept * D + (q0 + row) * 2 + 1] = sum;
    } else {
      const float inv = 1.0f / sum;
      const u32x2 w = {Half<BF>::pack(o[0] * inv, o[1] * inv), Half<BF>::pack(o[2] * inv, o[3] * inv)};
      *reinterpret_cast<u32x2*>(O + ((int64_t)head * sq + q0 + row) * D + d) = w;
    }
  }
}

// O from the parts' planes, four columns of one row per thread
template <bool BF, int D>
__global__ __launch_bounds__(256) void attention_reduce(const float* __restrict__ planes, uint16_t* __restrict__ O,
                                                        int64_t sq, int64_t kept, int64_t heads, int parts) {
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x, row = at / (D / 4);
  const int d = (int)(at % (D / 4)) * 4;
  if (row >= heads * sq) return;
  const int64_t head = row / sq, r = row % sq, stride = heads * kept * (D + 2);
  const float* plane = planes + head * kept * (D + 2);
  const float *o_at = plane + r * D + d, *s_at = plane + kept * D + r * 2;
  float top = s_at[0];
  for (int p = 1; p < parts; ++p) top = fmaxf(top, s_at[p * stride]);
  float sum = 0.0f;
  f32x4 o = f32x4{};
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const float f = __builtin_amdgcn_exp2f(s_at[p * stride] - top);
    sum += f * s_at[p * stride + 1];
    o += f * *reinterpret_cast<const f32x4*>(o_at + p * stride);
  }
  const float inv = 1.0f / sum;
  const u32x2 w = {Half<BF>::pack(o[0] * inv, o[1] * inv), Half<BF>::pack(o[2] * inv, o[3] * inv)};
  *reinterpret_cast<u32x2*>(O + row * D + d) = w;
}

}  // namespace krn

using namespace krn;

template <bool BF, int D, bool ONCE>
static int launch(const AttentionCall& c) {
  const int q_tiles = (int)((c.sq + 31) / 32);
  const dim3 grid((unsigned)(c.bh * q_tiles * c.parts));
  hipLaunchKernelGGL((attention_split<BF, D, ONCE>), grid, dim3(64 * SPLIT_WAVES), 0, c.stream, (const uint16_t*)c.q,
                     (const uint16_t*)c.k, (const uint16_t*)c.v, (uint16_t*)c.o, (float*)c.workspace, c.sq, c.sk,
                     c.scale, q_tiles, c.causal, c.parts, (int)c.bh);
  if (c.parts > 1) {
    const int64_t threads = c.bh * c.sq * (D / 4);
    hipLaunchKernelGGL((attention_reduce<BF, D>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, c.stream,
                       (const float*)c.workspace, (uint16_t*)c.o, c.sq, attention_split_rows(c.sq), c.bh, c.parts);
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("attention launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

// Up to 32 query rows a head are one row block, whose keys and values are read once. From 128 MiB of them, half of the
// last-level cache, their loads are non-temporal, since little would be found there by a later launch anyway (one query,
// heads x keys, d = 128: bf16 128 x 4096 57.4 -> 52.0 us, 4.7 -> 5.2 TB/s, 128 x 16384 190.9 -> 170.3, 32 x 8192, 128 MiB,
// 34.7 -> 32.0; f16 128 x 4096 56.5 -> 50.8, 32 x 8192 35.0 -> 32.3; d = 64: bf16 128 x 4096, 128 MiB, 31.6 -> 30.1,
// 64 x 16384 63.7 -> 56.7, f16 31.8 -> 29.8 and 64.4 -> 58.6; 32 queries f16 128 x 4096, d = 128, 58.2 -> 53.0). Smaller
// ones keep ordinary loads (64 MiB: bf16 8 x 16384, d = 128, 24.3 us, non-temporally 27.8; f16 25.5 and 28.4; bf16
// 16 x 16384, d = 64, 20.5 and 22.3), and so do longer prompts, whose row blocks share keys in L2 (16 x 1000 x
// 1000, d = 64: 11.9 us, non-temporally 13.2).
int krn::launch_attention_split(bool bf, int d, const AttentionCall& c) {
  const bool once = c.sq <= 32 && c.bh * c.sk * d * 4 >= (int64_t)128 << 20;
#define KRN_SPLIT(BFV, DV) (once ? launch<BFV, DV, true>(c) : launch<BFV, DV, false>(c))
  if (bf) return d == 128 ? KRN_SPLIT(true, 128) : KRN_SPLIT(true, 64);
  return d == 128 ? KRN_SPLIT(false, 128) : KRN_SPLIT(false, 64);
#undef KRN_SPLIT
}
