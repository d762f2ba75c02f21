// Row softmax for gfx950: y[r, c] = exp(x[r, c] - max_r) / sum_r exp(x[r, :] - max_r) over the first `width`
// columns of every row, in float32, rounded once to the element type of y.
//
// This is the lowering of krn's softmax tile programs (reference examples/02_tiles_and_types/01_softmax_rows.py
// :27-40, the long rows in column chunks with a running maximum and sum; tests/helpers/example_softmax.py:12-24,
// one tile per row block, `.softmax(axis=1)` or its spelled-out steps). Both compute the same function: the
// running form and the one-tile form differ only in rounding. Columns past `width` (the one-tile program's lanes
// past its tile) are neither read nor written; a row is a run of valid lanes, so no padding value enters the
// maximum or the sum.
//
// Layout (HBM-bound: one read, one write per element). A row belongs to one wave (four rows per workgroup), four waves,
// eight or sixteen: thread l owns the 16-byte chunks l, l + T, ... of its row. Up to CACHE chunks per thread stay in
// registers as they were read; what a longer row has past them is read again (from L2). A thread keeps a running
// maximum m and sum s of exp(x - m) over its chunks as they arrive (the maximum of all of them first: f16 8192 x 2048
// 12.6 -> 13.1 us), the threads' pairs meet by shuffles and in LDS, and a second pass writes exp(x - m) * (1 / s).
//
// Rows may start at any element: the chunks are loaded and stored 16 bytes at a time at any alignment, and only a chunk
// that crosses the end of its row goes element by element (bf16 1024 x 50001, rows at every alignment, element by
// element before: 145 -> 57 us; the copy of as many bytes takes 31).
#include "common.h"

namespace krn {

constexpr float LOG2E = 1.4426950408889634f;
typedef u32x4 u32x4_any __attribute__((aligned(1)));  // a 16-byte access at any address

template <int KIND>
struct Chunk {  // 16 bytes of a row
  static constexpr int N = KIND == F32 ? 4 : 8;
  static constexpr int BYTES = KIND == F32 ? 4 : 2;
  __device__ static float value(const u32x4& w, int e) {
    if constexpr (KIND == F32) return __uint_as_float(w[e]);
    const uint16_t h = (uint16_t)(w[e >> 1] >> ((e & 1) * 16));
    return KIND == F16 ? h2f(h) : bf2f(h);
  }
  __device__ static void set(u32x4& w, int e, float v) {  // into a zeroed chunk
    if constexpr (KIND == F32) w[e] = __float_as_uint(v);
    else w[e >> 1] |= (uint32_t)(KIND == F16 ? f2h(v) : f2bf(v)) << ((e & 1) * 16);
  }
  static constexpr uint32_t LOWEST = KIND == F32 ? 0xff800000u : KIND == F16 ? 0xfc00fc00u : 0xff80ff80u;  // -infinity
};

// Chunk c of a row; elements at or past `width` are -infinity (they add exp(-inf) = 0 to the sum and never win the
// maximum), and so is a chunk past the row
template <int KIND>
__device__ __forceinline__ u32x4 load_chunk(const uint8_t* row, int64_t c, int64_t width) {
  typedef Chunk<KIND> C;
  const int64_t col = c * C::N;
  if (col + C::N <= width) return *reinterpret_cast<const u32x4_any*>(row + col * C::BYTES);
  u32x4 w = {C::LOWEST, C::LOWEST, C::LOWEST, C::LOWEST};
#pragma unroll
  for (int e = 0; e < C::N; ++e)
    if (col + e < width) {
      if constexpr (KIND == F32) {
        w[e] = reinterpret_cast<const uint32_t*>(row)[col + e];
      } else {
        const uint32_t h = reinterpret_cast<const uint16_t*>(row)[col + e];
        w[e >> 1] = (e & 1) ? (w[e >> 1] & 0xffffu) | h << 16 : (w[e >> 1] & 0xffff0000u) | h;
      }
    }
  return w;
}

// NaN if an element of the chunk is (the maximum passes over NaN), otherwise 0
template <int KIND>
__device__ __forceinline__ float nan_of(const u32x4& w) {
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < Chunk<KIND>::N; ++e) {
    const float x = Chunk<KIND>::value(w, e);
    s = x != x ? x : s;
  }
  return s;
}

// exp(x - m) * inv of a chunk, rounded once, to the output. Chunks at 16-byte addresses are stored non-temporally: the
// output is not read again, and a wave's store covers whole lines (f16 32768 x 4096: 5.0 -> 6.5 TB/s). Unaligned ones
// share their first and last lines with their neighbours and keep ordinary stores, which the L2 joins.
template <int KIND, bool ALIGNED>
__device__ __forceinline__ void store_chunk(uint8_t* row, int64_t c, int64_t width, const u32x4& x, float m, float inv) {
  typedef Chunk<KIND> C;
  const int64_t col = c * C::N;
  u32x4 w = {0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < C::N; ++e) C::set(w, e, __builtin_amdgcn_exp2f((C::value(x, e) - m) * LOG2E) * inv);
  if (col + C::N <= width) {
    if constexpr (ALIGNED) __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(row + col * C::BYTES));
    else *reinterpret_cast<u32x4_any*>(row + col * C::BYTES) = w;
    return;
  }
#pragma unroll
  for (int e = 0; e < C::N; ++e)
    if (col + e < width) {
      if constexpr (KIND == F32) reinterpret_cast<uint32_t*>(row)[col + e] = w[e];
      else reinterpret_cast<uint16_t*>(row)[col + e] = (uint16_t)(w[e >> 1] >> ((e & 1) * 16));
    }
}

// (m, s) and (m2, s2) merged: both sums rescaled to the larger maximum. Without one yet, a sum is 0, or NaN if a NaN was
// read, which must reach both partners: exp(-inf - 0) = 0 keeps both.
__device__ __forceinline__ void combine(float& m, float& s, float m2, float s2) {
  const float m_new = fmaxf(m, m2), top = m_new == -INFINITY ? 0.0f : m_new;
  s = s * __builtin_amdgcn_exp2f((m - top) * LOG2E) + s2 * __builtin_amdgcn_exp2f((m2 - top) * LOG2E);
  m = m_new;
}

// One wave per row fills the chip when rows are many and fit its registers; more waves keep long rows in registers and
// enough loads in flight when rows are few.
template <int KIND, int CACHE, int WAVES, bool ALIGNED>
__global__ __launch_bounds__(WAVES == 1 ? 256 : WAVES * 64) void softmax_rows(const uint8_t* __restrict__ X,
                                                                               uint8_t* __restrict__ Y, int64_t rows,
                                                                               int64_t width, int64_t ldx, int64_t ldy) {
  typedef Chunk<KIND> C;
  constexpr int T = WAVES * 64;
  const int lane = threadIdx.x % T;
  const int64_t row = WAVES == 1 ? (int64_t)blockIdx.x * 4 + threadIdx.x / 64 : blockIdx.x;
  if constexpr (WAVES == 1) {
    if (row >= rows) return;  // a whole wave leaves together; no barrier follows
  }
  const int64_t chunks = (width + C::N - 1) / C::N;
  const uint8_t* x = X + row * ldx * C::BYTES;
  uint8_t* y = Y + row * ldy * C::BYTES;
  u32x4 kept[CACHE];
#pragma unroll
  for (int i = 0; i < CACHE; ++i) kept[i] = load_chunk<KIND>(x, lane + T * i, width);
  float m = -INFINITY, s = 0.0f;
#pragma unroll
  for (int i = 0; i < CACHE; ++i) {
    float top = m;
#pragma unroll
    for (int e = 0; e < C::N; ++e) top = fmaxf(top, C::value(kept[i], e));
    if (top == -INFINITY) {  // nothing valid yet, or NaN
      s += nan_of<KIND>(kept[i]);
      continue;
    }
    float add = 0.0f;
#pragma unroll
    for (int e = 0; e < C::N; ++e) add += __builtin_amdgcn_exp2f((C::value(kept[i], e) - top) * LOG2E);
    s = s * __builtin_amdgcn_exp2f((m - top) * LOG2E) + add;
    m = top;
  }
  for (int64_t c = lane + T * CACHE; c < chunks; c += T) {
    const u32x4 w = load_chunk<KIND>(x, c, width);
    float top = C::value(w, 0), add = 0.0f;
#pragma unroll
    for (int e = 1; e < C::N; ++e) top = fmaxf(top, C::value(w, e));
    if (!(top > -INFINITY)) {
      s += nan_of<KIND>(w);
      continue;
    }
#pragma unroll
    for (int e = 0; e < C::N; ++e) add += __builtin_amdgcn_exp2f((C::value(w, e) - top) * LOG2E);
    combine(m, s, top, add);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) combine(m, s, __shfl_xor(m, off), __shfl_xor(s, off));
  if constexpr (WAVES > 1) {
    __shared__ float part[2][WAVES];
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) part[0][wave] = m, part[1][wave] = s;
    __syncthreads();
    m = part[0][0], s = part[1][0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) combine(m, s, part[0][w], part[1][w]);
  }
  const float inv = 1.0f / s;
  // Before the second pass: the chunks stay as they were read (the compiler would keep 16-bit chunks' float32 values,
  // twice the registers). It pays where it lets another workgroup fit: f16 4096 x 16400 on eight waves 53.1 -> 49.8 us.
  // Elsewhere converting twice costs more: 20000 x 2048 25.2 -> 27.0, 4096 x 8192 20.9 -> 22.3, 1000 x 16384 12.7 ->
  // 13.3, 1000 x 40000 29.2 -> 30.7 (4096 x 12000 on four waves alone would gain, 35.6 -> 34.2).
  if constexpr (CACHE > 4 && CACHE < 8 && WAVES != 4) {
#pragma unroll
    for (int i = 0; i < CACHE; ++i) asm volatile("" : "+v"(kept[i]));
  }
#pragma unroll
  for (int i = 0; i < CACHE; ++i)
    if (lane + T * i < chunks) store_chunk<KIND, ALIGNED>(y, lane + T * i, width, kept[i], m, inv);
  for (int64_t c = lane + T * CACHE; c < chunks; c += T)
    store_chunk<KIND, ALIGNED>(y, c, width, load_chunk<KIND>(x, c, width), m, inv);
}

}  // namespace krn

using namespace krn;

// A workgroup per row takes the rows in runs of 2^21: a launch holds fewer than 2^32 threads, which 2^22 rows of sixteen
// waves reach. A wave per row needs 2^26 rows for that.
template <int KIND, int CACHE, int WAVES>
static void launch_rows(bool aligned, const void* x, void* y, int64_t rows, int64_t width, int64_t ldx, int64_t ldy,
                        hipStream_t stream) {
  constexpr int64_t BYTES = Chunk<KIND>::BYTES;
  const int64_t most = WAVES == 1 ? rows : (int64_t)1 << 21;
  for (int64_t r0 = 0; r0 < rows; r0 += most) {
    const int64_t n = rows - r0 < most ? rows - r0 : most;
    const dim3 grid((unsigned)(WAVES == 1 ? (n + 3) / 4 : n)), block(WAVES == 1 ? 256 : WAVES * 64);
    const uint8_t* xr = (const uint8_t*)x + r0 * ldx * BYTES;
    uint8_t* yr = (uint8_t*)y + r0 * ldy * BYTES;
    if (aligned)
      hipLaunchKernelGGL((softmax_rows<KIND, CACHE, WAVES, true>), grid, block, 0, stream, xr, yr, n, width, ldx, ldy);
    else
      hipLaunchKernelGGL((softmax_rows<KIND, CACHE, WAVES, false>), grid, block, 0, stream, xr, yr, n, width, ldx, ldy);
  }
}

template <int KIND>
static int launch_softmax(const void* x, void* y, int64_t rows, int64_t width, int64_t ldx, int64_t ldy,
                          hipStream_t stream) {
  constexpr int N = Chunk<KIND>::N;
  const bool aligned = (ldy * Chunk<KIND>::BYTES) % 16 == 0 && (uintptr_t)y % 16 == 0;
  const int64_t chunks = (width + N - 1) / N;
#define KRN_ROWS(CACHE, WAVES) launch_rows<KIND, CACHE, WAVES>(aligned, x, y, rows, width, ldx, ldy, stream)
  // No more chunks per thread than the row needs, because a chunk past the row costs what one in it does; no more waves
  // than keep the row in registers, because they wait for each other; and eight waves before sixteen, of which only one
  // workgroup fits a compute unit where two or more of eight do. us, the other choice -> this one:
  //   bf16 20000 x 1000: four chunks 18.4 -> two 14.9; f16 4096 x 3000: two of four waves 12.2 -> six of one 10.5
  //   f16 4096 (1000) x 4096: eight of one wave 12.9 (5.5) -> two of four 13.2 (4.9); 20000 x 4096: 58.3 -> 56.6; f32
  //   4096 (1000) x 2048: 10.3 (4.4) -> 10.9 (4.2); 20000 x 2048: 57.2 -> 54.3
  //   f16 4096 x 8200: eight of four 28 -> five 23.2; x 16384: eight of four 47.7, four of eight 47.3
  //   f16 4096 x 16400: eight of sixteen 151 -> five of eight 49.7, and eight of four with the rest read again 50.1 (at
  //   1000 rows that is the faster by 4 to 9 %); x 20000: 62 -> 58; x 24576: 76 -> 71
  //   f16 4096 x 32768: eight of sixteen 172, four of sixteen 101.7, eight of eight 101.7 to 105; 1000 x 32768:
  //   25.6 -> 23.6
  // Past what eight waves keep, reading up to three more chunks a thread again is still the better one: f32 4096 x 20000
  // 126 (five of sixteen) -> 113, 4096 x 24576 147 -> 142; with fewer rows than compute units it is not: 128 x 57344 f16
  // 12.9 against 11.9 us. Rows of 8192 chunks: 202 -> 193.
  if (chunks <= 64) KRN_ROWS(1, 1);
  else if (chunks <= 128) KRN_ROWS(2, 1);
  else if (chunks <= 256) KRN_ROWS(4, 1);
  else if (chunks <= 320) KRN_ROWS(5, 1);
  else if (chunks <= 384) KRN_ROWS(6, 1);
  else if (chunks <= 512) KRN_ROWS(2, 4);
  else if (chunks <= 768) KRN_ROWS(3, 4);
  else if (chunks <= 1024) KRN_ROWS(4, 4);
  else if (chunks <= 1280) KRN_ROWS(5, 4);
  else if (chunks <= 1536) KRN_ROWS(6, 4);
  else if (chunks <= 1792) KRN_ROWS(7, 4);
  else if (chunks <= 2048) KRN_ROWS(8, 4);
  else if (chunks <= 2560) KRN_ROWS(5, 8);
  else if (chunks <= 3072) KRN_ROWS(6, 8);
  else if (chunks <= 4096 || (chunks <= 7168 && rows > 256)) KRN_ROWS(8, 8);
  else KRN_ROWS(8, 16);
#undef KRN_ROWS
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("softmax launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

extern "C" int krn_softmax_rows(int kind, const void* x, void* y, int64_t rows, int64_t width, int64_t ldx,
                                int64_t ldy, void* stream) {
  if (kind != F32 && kind != F16 && kind != BF16) {
    krn_set_error("softmax: element kind %d; f32, f16 or bf16 only", kind);
    return -1;
  }
  if (rows < 0 || width < 0 || ldx < width || ldy < width) {
    krn_set_error("softmax: %lld rows of %lld columns with row strides %lld and %lld", (long long)rows,
                  (long long)width, (long long)ldx, (long long)ldy);
    return -1;
  }
  if (rows == 0 || width == 0) return 0;
  if ((rows + 3) / 4 > 0x7fffffff) {
    krn_set_error("softmax: %lld rows exceed the grid limit", (long long)rows);
    return -1;
  }
  hipStream_t s = (hipStream_t)stream;
  if (kind == F32) return launch_softmax<F32>(x, y, rows, width, ldx, ldy, s);
  if (kind == F16) return launch_softmax<F16>(x, y, rows, width, ldx, ldy, s);
  return launch_softmax<BF16>(x, y, rows, width, ldx, ldy, s);
}
