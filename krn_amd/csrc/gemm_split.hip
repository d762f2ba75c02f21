// GEMM for the products the whole-tile loops of gemm.hip leave the chip idle on or cannot take: C = epilogue(A B^T)
// (NT, every format) and C = epilogue(A B) with B stored K x N (NN, 16-bit) at any M, N, K and alignment.
//
// What bounds these products is not a rate but how the work is spread: a product of 256 x 4096 x 14336 has 64 tiles of
// 128 x 128 for 256 CUs, each with 224 K slices to run one after the other. So the tiles are smaller where that alone
// fills the chip, and K is split over `parts` workgroups per tile where it does not: each part writes its float32
// (int32) sums to a plane of the caller's workspace, and a second kernel adds the planes in part order and applies the
// epilogue. (One launch with an arrival counter per tile, the last workgroup adding the parts, was slower: the
// release of the partial sums across the XCDs writes back the L2 in every workgroup, 10-15 us per launch.)
//
// Two loaders. `gemm_ring` (16-byte aligned rows): direct-to-LDS loads into a ring of slices, STAGES - 1 of them in
// flight. `gemm_any` (any alignment: the row of an odd K starts anywhere): through registers, two slices ahead, with
// 16-byte loads at any byte address. Chunks past the end of K are zeros in both, so K need not be whole slices; the
// NN form keeps its B slice as [k][n] and reads MFMA fragments with transposed LDS reads, so B needs no transposed copy.
#include "gemm_parts.h"
#include "gemm_split.h"

namespace krn {

// s_barrier for LDS traffic only: loads in flight to registers stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// K part and tile of this workgroup. Workgroups go round-robin over the 8 XCDs; each XCD gets one contiguous range of
// (part, tile) pairs, tiles running first, so that tiles
// of the same rows or columns and K part share its L2 (i8 333 x 5000 x 4096: 24.4 -> 16.5 us; fp8 1673 x 6528 x 1248:
// 32.0 -> 28.9; bf16 256 x 4096 x 14336: 57.4 -> 56.4). With one tile row only A is shared, which is small.
__device__ __forceinline__ int part_tile_of(int tiles_m, int tiles_n, int parts, int& tm, int& tn) {
  const int tiles = tiles_m * tiles_n, total = tiles * parts, id = blockIdx.y * tiles + blockIdx.x;
  const int each = total / 8, more = total % 8, xcd = id % 8;
  const int at = tiles_m > 1 ? xcd * each + min(xcd, more) + id / 8 : id, tile = at % tiles;
  constexpr int GROUP_M = 4;  // tiles of a group of tile rows run column by column
  const int group = tile / (GROUP_M * tiles_n), local = tile % (GROUP_M * tiles_n);
  const int rows = min(tiles_m - group * GROUP_M, GROUP_M);
  // scalar for the compiler too: an index it holds per lane costs a loop at each buffer load (3 us at 12 x 4096 x 1360)
  tm = __builtin_amdgcn_readfirstlane(group * GROUP_M + local % rows);
  tn = __builtin_amdgcn_readfirstlane(local / rows);
  return __builtin_amdgcn_readfirstlane(at / tiles);
}

// a 16-byte piece without its first `drop` bytes (zeros move in at the end; 16 or more: nothing is left)
__device__ __forceinline__ u32x4 drop_bytes(u32x4 v, int drop) {
  uint64_t lo = (uint64_t)v[0] | (uint64_t)v[1] << 32, hi = (uint64_t)v[2] | (uint64_t)v[3] << 32;
  if (drop >= 8) lo = hi, hi = 0;
  const int bits = (drop & 7) * 8;
  if (bits) lo = lo >> bits | hi << (64 - bits), hi >>= bits;
  if (drop >= 16) lo = 0, hi = 0;
  return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// A wave's blocks to C, or to the plane of this K part. One row of blocks at a time goes into patches of its own, and
// one copy of the patch store runs over them: with the out-of-line store the compiler would keep the accumulators in
// AGPRs (a called function may use them) and copy all of them to VGPRs and back around every slice.
template <bool INT, int TM, int TN, typename Acc>
__device__ __forceinline__ void store_blocks(const Acc (&acc)[TM][TN], uint32_t* lds, int wave, void* C,
                                             int part, int64_t ldc, int64_t row0, int64_t col0, int64_t M,
                                             int64_t N, const Epilogue& e, int lane) {
  uint32_t* patch = lds + wave * TN * PATCH_WORDS;
  void* out = static_cast<uint8_t*>(C) + part * (M * ldc * 4);  // part 0 of one: C itself
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) patch_put<INT>(acc[i][j], patch + j * PATCH_WORDS, lane);
#pragma unroll 1
    for (int j = 0; j < TN; ++j)
      patch_store_inline<INT, true, false, true>(patch + j * PATCH_WORDS, out, ldc, row0 + i * 32, col0 + j * 32, M, N, e, lane);
  }
}

// BM x BN tile, WM x WN waves of TM x TN blocks of 32 x 32, 128-byte K slices. `kbytes` = K times the element size,
// rows of A (and of B, NT) `lda` (`ldb`) bytes apart; NN: rows of B are N elements, `ldb` bytes, B has K of them.
template <int FMT, int BM, int BN, int WM, int WN, bool NN>
__global__ __launch_bounds__(256, 2) void gemm_any(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                     void* __restrict__ C, int64_t M, int64_t N, int64_t kbytes,
                                                     int64_t lda, int64_t ldb, int64_t ldc, Epilogue e, int parts) {
  typedef Mfma<FMT> Unit;
  typedef typename Unit::Acc Acc;
  constexpr int BKB = 128, TM = BM / WM / 32, TN = BN / WN / 32, STEP = Unit::kBytes, CH = STEP / 32;
  constexpr int PA = BM / 32, PB = BN / 32;  // 16-byte chunks per thread per slice
  constexpr int STAGE = (BM + BN) * 8;       // 16-byte units
  static_assert(WM * WN == 4 && TM >= 1 && TN >= 1, "four waves");
  static_assert(!NN || FMT == FMT_BF16 || FMT == FMT_F16, "the NN form is 16-bit");
  constexpr int PATCHES = 4 * TN * PATCH_WORDS / 4;  // 16-byte units
  __shared__ __attribute__((aligned(1024))) u32x4 lds[2 * STAGE > PATCHES ? 2 * STAGE : PATCHES];

  int tm, tn;
  const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN);
  const int part = part_tile_of(tiles_m, tiles_n, parts, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN, half = lane >> 5, r32 = lane & 31;

  // this workgroup's K slices; a part that holds the partial last slice takes it first, so that the loop's loads are
  // all whole
  const int slices = (int)((kbytes + BKB - 1) / BKB), whole = (int)(kbytes / BKB);
  const int first = (int)((int64_t)slices * part / parts), n = (int)((int64_t)slices * (part + 1) / parts) - first;
  const bool tail = first + n > whole;
  const int kbase = tail ? first - 1 : first;

  // NT operands: thread t loads chunk t & 7 of rows (t >> 3) + 32 p. NN's B: BN / 8 chunks per k row. A chunk that
  // crosses the end of its row is loaded from the row's last 16 bytes, and the bytes before it are dropped on the way
  // to LDS; rows past the last one read the last (their results are not stored).
  constexpr int NCH = BN / 8, KROWS = 256 / NCH;  // NN: chunks per k row, k rows per load pass
  const int chunk = t & 7, bchunk = NN ? t % NCH : chunk, bk = t / NCH;
  const int64_t b_at = (n0 + bchunk * 8) * 2, b_from = min(b_at, N * 2 - 16);  // NN: this thread's bytes of a row of B
  const bool n_edge = NN && n0 + BN > N;
  const uint8_t* a_base = A + m0 * lda;
  const uint8_t* b_base = NN ? B : B + n0 * ldb;
  uint32_t a_off[PA], b_off[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) a_off[p] = (uint32_t)(min((int64_t)(t >> 3) + 32 * p, M - 1 - m0) * lda);
#pragma unroll
  for (int p = 0; p < PB; ++p)
    b_off[p] = NN ? (uint32_t)((bk + KROWS * p) * ldb + b_from)
                  : (uint32_t)(min((int64_t)(t >> 3) + 32 * p, N - 1 - n0) * ldb);

  u32x4 ra0[PA], rb0[PB], ra1[PA], rb1[PB];
#define KRN_LOAD(s, i)                                                                                                 \
  do {                                                                                                                 \
    const int64_t slice = kbase + min((i), n - 1); /* past the end: the last slice again, never used */                \
    const uint8_t* pa = a_base + slice * BKB + chunk * 16;                                                             \
    _Pragma("unroll") for (int p = 0; p < PA; ++p) ra##s[p] = *reinterpret_cast<const u32x4_any*>(pa + a_off[p]);      \
    const uint8_t* pb = b_base + (NN ? slice * 64 * ldb : slice * BKB + chunk * 16);                                   \
    _Pragma("unroll") for (int p = 0; p < PB; ++p) rb##s[p] = *reinterpret_cast<const u32x4_any*>(pb + b_off[p]);      \
  } while (0)
#define KRN_PUT(s, stage)                                                                                              \
  do {                                                                                                                 \
    u32x4* st = lds + (stage) * STAGE;                                                                                 \
    if (n_edge) {                                                                                                      \
      _Pragma("unroll") for (int p = 0; p < PB; ++p) rb##s[p] = drop_bytes(rb##s[p], (int)min(b_at - b_from, (int64_t)16)); \
    }                                                                                                                  \
    _Pragma("unroll") for (int p = 0; p < PA; ++p) {                                                                   \
      const int row = (t >> 3) + 32 * p;                                                                               \
      st[row * 8 + (chunk ^ swz8(row))] = ra##s[p];                                                                    \
    }                                                                                                                  \
    _Pragma("unroll") for (int p = 0; p < PB; ++p) {                                                                   \
      if constexpr (NN) {                                                                                              \
        const int k = bk + KROWS * p;                                                                                  \
        st[BM * 8 + k * NCH + kn_slot<BN>(k, bchunk)] = rb##s[p];                                                      \
      } else {                                                                                                         \
        const int row = (t >> 3) + 32 * p;                                                                             \
        st[BM * 8 + row * 8 + (chunk ^ swz8(row))] = rb##s[p];                                                         \
      }                                                                                                                \
    }                                                                                                                  \
  } while (0)
  // NN fragments: lane group g = lane / 16 reads k rows 8 (g / 2) + 4 part + (lane % 16) / 4 at columns
  // 16 (g % 2) + 4 (lane % 4) .. + 3 and receives one column's four k
  const int tr_k = half * 8 + ((lane & 15) >> 2), tr_n = ((lane >> 4) & 1) * 16 + 4 * (lane & 3);
#define KRN_COMPUTE(stage)                                                                                             \
  do {                                                                                                                 \
    const u32x4* st = lds + (stage) * STAGE;                                                                           \
    _Pragma("unroll") for (int k = 0; k < BKB / STEP; ++k) {                                                           \
      u32x4 fa[TM][CH], fb[TN][CH];                                                                                    \
      _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int c = 0; c < CH; ++c) {                  \
        const int row = wm * (BM / WM) + i * 32 + r32;                                                                 \
        fa[i][c] = st[row * 8 + (((k * STEP + half * (STEP / 2)) / 16 + c) ^ swz8(row))];                              \
      }                                                                                                                \
      _Pragma("unroll") for (int j = 0; j < TN; ++j) {                                                                 \
        if constexpr (NN) {                                                                                            \
          _Pragma("unroll") for (int q = 0; q < 2; ++q) {                                                              \
            const int kk = k * 16 + tr_k + q * 4, col = wn * (BN / WN) + j * 32 + tr_n;                                \
            const uint8_t* at = reinterpret_cast<const uint8_t*>(st + BM * 8) + kk * (BN * 2) +                        \
                                kn_slot<BN>(kk, col >> 3) * 16 + (col & 7) * 2;                                        \
            const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(                         \
                (__attribute__((address_space(3))) v4s16*)(const_cast<uint8_t*>(at))));                                \
            fb[j][0][2 * q] = w[0], fb[j][0][2 * q + 1] = w[1];                                                        \
          }                                                                                                            \
        } else {                                                                                                       \
          _Pragma("unroll") for (int c = 0; c < CH; ++c) {                                                             \
            const int row = wn * (BN / WN) + j * 32 + r32;                                                             \
            fb[j][c] = st[BM * 8 + row * 8 + (((k * STEP + half * (STEP / 2)) / 16 + c) ^ swz8(row))];                 \
          }                                                                                                            \
        }                                                                                                              \
      }                                                                                                                \
      _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int j = 0; j < TN; ++j)                    \
          Unit::step(acc[i][j], fa[i], fb[j]);                                                                         \
    }                                                                                                                  \
  } while (0)

  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Acc{};
  if (tail) {
    const int64_t kb = (int64_t)whole * BKB + chunk * 16, from = min(kb, kbytes - 16);
    const int drop = (int)min(kb - from, (int64_t)16);
    const int64_t left = kbytes / 2 - (int64_t)whole * 64;  // NN: k rows of B in the partial slice
#pragma unroll
    for (int p = 0; p < PA; ++p) ra0[p] = *reinterpret_cast<const u32x4_any*>(a_base + from + a_off[p]);
#pragma unroll
    for (int p = 0; p < PB; ++p) {
      const uint8_t* at = NN ? B + ((int64_t)whole * 64 + min((int64_t)(bk + KROWS * p), left - 1)) * ldb + b_from
                             : b_base + from + b_off[p];
      rb0[p] = *reinterpret_cast<const u32x4_any*>(at);
    }
#pragma unroll
    for (int p = 0; p < PA; ++p) ra0[p] = drop_bytes(ra0[p], drop);
#pragma unroll
    for (int p = 0; p < PB; ++p) {
      if constexpr (NN) rb0[p] = bk + KROWS * p < left ? rb0[p] : u32x4{};
      else rb0[p] = drop_bytes(rb0[p], drop);
    }
  } else if (n > 0) {
    KRN_LOAD(0, 0);
  }
  if (n > 1) {
    KRN_LOAD(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    KRN_PUT(0, 0);
    KRN_LOAD(0, 2);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    // Two slices per turn, in one block: loads past the last slice repeat it, so that no wait depends on a branch and
    // the compiler cannot sink a load past one (it delayed them to their use); the scheduling barriers keep their place.
    for (int i = 0; i + 1 < n; i += 2) {
      KRN_PUT(1, 1);
      KRN_LOAD(1, i + 3);
      __builtin_amdgcn_sched_barrier(0);
      KRN_COMPUTE(0);
      lds_barrier();
      KRN_PUT(0, 0);
      KRN_LOAD(0, i + 4);
      __builtin_amdgcn_sched_barrier(0);
      KRN_COMPUTE(1);
      lds_barrier();
    }
  } else {
    KRN_PUT(0, 0);
    lds_barrier();
  }
  if (n & 1) KRN_COMPUTE(0);
  lds_barrier();  // every wave is done with the stages before their LDS becomes the store patches
#undef KRN_LOAD
#undef KRN_PUT
#undef KRN_COMPUTE

  store_blocks<FMT == FMT_I8>(acc, reinterpret_cast<uint32_t*>(lds), wave, C, part, ldc, m0 + wm * (BM / WM),
                              n0 + wn * (BN / WN), M, N, e, lane);
}

constexpr uint32_t OUTSIDE = 0x80000000u;  // an offset past every buffer resource (at most 2^31 - 1 bytes)

// One lane's B fragments of a 128-byte slice kept [k][n]: two transposed reads (four k each) per MFMA step, in one
// block with their wait
template <int BN>
__device__ __forceinline__ void tr_read(uint8_t* p, u32x4 (&f)[4]) {
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)p;
  constexpr int Q = 4 * BN * 2, K = 16 * BN * 2;
  u32x2 w[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%9\n\t"
      "ds_read_b64_tr_b16 %2, %8 offset:%10\n\tds_read_b64_tr_b16 %3, %8 offset:%11\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:%12\n\tds_read_b64_tr_b16 %5, %8 offset:%13\n\t"
      "ds_read_b64_tr_b16 %6, %8 offset:%14\n\tds_read_b64_tr_b16 %7, %8 offset:%15\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7])
      : "v"(at), "n"(Q), "n"(K), "n"(K + Q), "n"(2 * K), "n"(2 * K + Q), "n"(3 * K), "n"(3 * K + Q)
      : "memory");
#pragma unroll
  for (int k = 0; k < 4; ++k) f[k] = u32x4{w[2 * k][0], w[2 * k][1], w[2 * k + 1][0], w[2 * k + 1][1]};
}

// The aligned loader: rows of A and B (NN: rows of B) start at 16-byte addresses and are whole 16-byte pieces. A ring of
// STAGES slices filled by direct-to-LDS loads, STAGES - 1 in flight, one barrier per slice; buffer resources sized to the
// operands and an offset past them give zeros for pieces outside. One LDS array: with an array per stage the compiler
// waits for every load in flight before the fragment reads it cannot tell apart (2x slower). The transposed reads of
// the NN form are assembly for the same reason, each block of reads with its wait.
// Two workgroups share a CU where the ring leaves room; the accumulators then live in VGPRs. Where it does not (PIPED:
// one wave per SIMD, nothing else to run while a wave reads its fragments), a slice's fragments are read between the
// MFMAs of the slice before it, whose stage is refilled at once (NT bf16, the plain loop and this one on one box:
// 512 x 8192 x 8192 85.7 -> 81.6 us, 384 x 6144 x 5120 49.8 -> 42.0). The NN form's transposed reads wait in their own block and keep the plain loop.
template <int FMT, int BM, int BN, int WM, int WN, int STAGES, bool PIPED, bool NN>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_ring(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                     void* __restrict__ C, int64_t M, int64_t N, int64_t kbytes,
                                                     int64_t lda, int64_t ldb, int64_t ldc, Epilogue e, int parts) {
  typedef Mfma<FMT> Unit;
  typedef typename Unit::Acc Acc;
  constexpr int BKB = 128, TM = BM / WM / 32, TN = BN / WN / 32, STEP = Unit::kBytes, CH = STEP / 32, KS = BKB / STEP;
  constexpr int CPR = BKB / 16, RPL = 1024 / BKB, WAVES = WM * WN;
  constexpr int NCH = BN / 8, KROWS = BKB / 2, KPL = 64 / NCH;  // NN: chunks per k row, k rows per slice, per load
  constexpr int LA = BM / RPL / WAVES, LB = NN ? KROWS / KPL / WAVES : BN / RPL / WAVES, LOADS = LA + LB;
  static_assert(LA * RPL * WAVES == BM, "whole loads");
  static_assert(NN ? LB * KPL * WAVES == KROWS : LB * RPL * WAVES == BN, "whole loads");
  constexpr int SB = (BM + BN) * BKB;
  constexpr bool PIPE = !NN && PIPED;
  static_assert(STAGES == 4 || (STAGES == 2 && !PIPE), "the loops' stages");
  static_assert((STAGES - 2) * LOADS <= 63, "vmcnt range");
  constexpr int LDS_BYTES = STAGES * SB > WAVES * TN * PATCH_WORDS * 4 ? STAGES * SB : WAVES * TN * PATCH_WORDS * 4;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_BYTES];
  uint8_t *const s0 = lds, *const s1 = lds + SB, *const s2 = lds + 2 * SB, *const s3 = lds + 3 * SB;
  int tm, tn;
  const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN);
  const int part = part_tile_of(tiles_m, tiles_n, parts, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WN, wn = wave % WN, half = lane >> 5, r32 = lane & 31;
  const int slices = (int)((kbytes + BKB - 1) / BKB), whole = (int)(kbytes / BKB);
  const int first = (int)((int64_t)slices * part / parts), n = (int)((int64_t)slices * (part + 1) / parts) - first;
  const bool tail = first + n > whole;  // this part ends with the partial slice: it is taken first
  const int kbase = tail ? first - 1 : first;

  const __amdgpu_buffer_rsrc_t a_rsrc = panel_rsrc(A + m0 * lda, (M - m0) * lda),
                              b_rsrc = NN ? panel_rsrc(B + n0 * 2, kbytes / 2 * ldb - n0 * 2) : panel_rsrc(B + n0 * ldb, (N - n0) * ldb);
  uint32_t a_off[LA], b_off[LB];
  const int lrow = lane / CPR, lslot = lane % CPR;
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int row = (wave * LA + j) * RPL + lrow, c = lslot ^ swz8(row);
    a_off[j] = (uint32_t)(row * lda + c * 16);
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    if constexpr (NN) {
      const int k = (wave * LB + j) * KPL + lane / NCH, c = kn_slot<BN>(k, lane % NCH);
      b_off[j] = n0 + c * 8 < N ? (uint32_t)(k * ldb + c * 16) : OUTSIDE;
    } else {
      const int row = (wave * LB + j) * RPL + lrow, c = lslot ^ swz8(row);
      b_off[j] = (uint32_t)(row * ldb + c * 16);
    }
  }
  const int a_step = BKB, b_step = NN ? (int)(KROWS * ldb) : BKB;
#define KRN_ISSUE(st, i)                                                                                               \
  do {                                                                                                                 \
    const int sl = kbase + (i);                                                                                        \
    _Pragma("unroll") for (int j = 0; j < LA; ++j) buffer_to_lds16(a_rsrc, st + (wave * LA + j) * 1024, a_off[j], sl * a_step); \
    _Pragma("unroll") for (int j = 0; j < LB; ++j) buffer_to_lds16(b_rsrc, st + BM * BKB + (wave * LB + j) * 1024, b_off[j], sl * b_step); \
  } while (0)
#define KRN_ISSUE_TAIL(st)                                                                                             \
  do {                                                                                                                 \
    const int left = (int)(kbytes - (int64_t)whole * BKB);                                                             \
    _Pragma("unroll") for (int j = 0; j < LA; ++j) {                                                                   \
      const int row = (wave * LA + j) * RPL + lrow, c = lslot ^ swz8(row);                                             \
      buffer_to_lds16(a_rsrc, st + (wave * LA + j) * 1024, c * 16 < left ? a_off[j] : OUTSIDE, whole * a_step);        \
    }                                                                                                                  \
    _Pragma("unroll") for (int j = 0; j < LB; ++j) {                                                                   \
      bool in;                                                                                                         \
      if constexpr (NN) in = ((wave * LB + j) * KPL + lane / NCH) * 2 < left;                                          \
      else { const int row = (wave * LB + j) * RPL + lrow; in = (lslot ^ swz8(row)) * 16 < left; }                     \
      buffer_to_lds16(b_rsrc, st + BM * BKB + (wave * LB + j) * 1024, in ? b_off[j] : OUTSIDE, whole * b_step);        \
    }                                                                                                                  \
  } while (0)
  const int tr_k = half * 8 + ((lane & 15) >> 2), tr_n = ((lane >> 4) & 1) * 16 + 4 * (lane & 3);
#define KRN_COMPUTE(stg)                                                                                               \
  do {                                                                                                                 \
    const u32x4* st = reinterpret_cast<const u32x4*>(stg);                                                             \
    u32x4 fa[KS][TM][CH], fb[KS][TN][CH], trd[TN][4];                                                                  \
    _Pragma("unroll") for (int k = 0; k < KS; ++k) {                                                                   \
      _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int c = 0; c < CH; ++c) {                  \
        const int row = wm * (BM / WM) + i * 32 + r32, ch = (k * STEP + half * (STEP / 2)) / 16 + c;                   \
        fa[k][i][c] = st[row * CPR + (ch ^ swz8(row))];                                                                \
      }                                                                                                                \
      _Pragma("unroll") for (int j = 0; j < TN; ++j) {                                                                 \
        if constexpr (NN) {                                                                                            \
          if (k == 0) {                                                                                                \
            const int col = wn * (BN / WN) + j * 32 + tr_n;                                                            \
            tr_read<BN>(stg + BM * BKB + tr_k * (BN * 2) + kn_slot<BN>(tr_k, col >> 3) * 16 + (col & 7) * 2, trd[j]);  \
          }                                                                                                            \
          fb[k][j][0] = trd[j][k];                                                                                     \
        } else _Pragma("unroll") for (int c = 0; c < CH; ++c) {                                                        \
          const int row = wn * (BN / WN) + j * 32 + r32, ch = (k * STEP + half * (STEP / 2)) / 16 + c;                 \
          fb[k][j][c] = st[BM * CPR + row * CPR + (ch ^ swz8(row))];                                                   \
        }                                                                                                              \
      }                                                                                                                \
    }                                                                                                                  \
    _Pragma("unroll") for (int k = 0; k < KS; ++k) _Pragma("unroll") for (int i = 0; i < TM; ++i)                      \
        _Pragma("unroll") for (int j = 0; j < TN; ++j) Unit::step(acc[i][j], fa[k][i], fb[k][j]);                      \
    /* all fragment reads of the slice, then its MFMAs (64 x 64 tiles: 17.9 -> 16.6 us at 256 x 4096 x 4096) */        \
    __builtin_amdgcn_sched_group_barrier(0x100, KS * (TM + (NN ? 0 : TN)) * CH, 0);                                    \
    __builtin_amdgcn_sched_group_barrier(0x008, KS * TM * TN, 0);                                                      \
  } while (0)
#define KRN_VMWAIT(n) __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00 | ((n) & 15) | (((n) >> 4) << 14))
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Acc{};
  if (n > 0) { if (tail) KRN_ISSUE_TAIL(s0); else KRN_ISSUE(s0, 0); }
  if (STAGES == 4 && n > 1) KRN_ISSUE(s1, 1);
  if (STAGES == 4 && n > 2) KRN_ISSUE(s2, 2);
  if constexpr (PIPE) {
    if (n > 3) KRN_ISSUE(s3, 3);
    u32x4 fa0[KS][TM][CH], fb0[KS][TN][CH], fa1[KS][TM][CH], fb1[KS][TN][CH];
#define KRN_READ(stg, set)                                                                                             \
  do {                                                                                                                 \
    const u32x4* st = reinterpret_cast<const u32x4*>(stg);                                                             \
    _Pragma("unroll") for (int k = 0; k < KS; ++k) _Pragma("unroll") for (int c = 0; c < CH; ++c) {                    \
      const int ch = (k * STEP + half * (STEP / 2)) / 16 + c;                                                          \
      _Pragma("unroll") for (int i = 0; i < TM; ++i) {                                                                 \
        const int row = wm * (BM / WM) + i * 32 + r32;                                                                 \
        fa##set[k][i][c] = st[row * CPR + (ch ^ swz8(row))];                                                           \
      }                                                                                                                \
      _Pragma("unroll") for (int j = 0; j < TN; ++j) {                                                                 \
        const int row = wn * (BN / WN) + j * 32 + r32;                                                                 \
        fb##set[k][j][c] = st[BM * CPR + row * CPR + (ch ^ swz8(row))];                                                \
      }                                                                                                                \
    }                                                                                                                  \
  } while (0)
// the reads are used here, so that they stay before this point
#define KRN_HELD(set)                                                                                                  \
  do {                                                                                                                 \
    _Pragma("unroll") for (int k = 0; k < KS; ++k) _Pragma("unroll") for (int c = 0; c < CH; ++c) {                    \
      _Pragma("unroll") for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(fa##set[k][i][c]));                        \
      _Pragma("unroll") for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(fb##set[k][j][c]));                        \
    }                                                                                                                  \
  } while (0)
#define KRN_TURN(d, st, next, set, other)                                                                              \
    if (i + d >= n) break;                                                                                             \
    if (i + d + 3 < n) KRN_VMWAIT(2 * LOADS); else KRN_VMWAIT(0);                                                      \
    __builtin_amdgcn_s_barrier();                                                                                      \
    if (i + d + 4 < n) KRN_ISSUE(st, i + d + 4);                                                                       \
    KRN_READ(next, other);                                                                                             \
    _Pragma("unroll") for (int k = 0; k < KS; ++k) _Pragma("unroll") for (int a = 0; a < TM; ++a)                      \
        _Pragma("unroll") for (int b = 0; b < TN; ++b) Unit::step(acc[a][b], fa##set[k][a], fb##set[k][b]);            \
    _Pragma("unroll") for (int g = 0; g < KS * TM * TN; ++g) {                                                         \
      __builtin_amdgcn_sched_group_barrier(0x100, ((TM + TN) * CH + TM * TN - 1) / (TM * TN), 0);                      \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                               \
    }                                                                                                                  \
    KRN_HELD(other);
    if (n > 3) KRN_VMWAIT(3 * LOADS); else KRN_VMWAIT(0);
    __builtin_amdgcn_s_barrier();
    KRN_READ(s0, 0);
    KRN_HELD(0);
    for (int i = 0;; i += 4) {
      // one workgroup per CU: the accumulators are AGPRs, and stay there around the loop
      _Pragma("unroll") for (int a = 0; a < TM; ++a) _Pragma("unroll") for (int b = 0; b < TN; ++b) asm volatile("" : "+a"(acc[a][b]));
      KRN_TURN(0, s0, s1, 0, 1)
      KRN_TURN(1, s1, s2, 1, 0)
      KRN_TURN(2, s2, s3, 0, 1)
      KRN_TURN(3, s3, s0, 1, 0)
    }
#undef KRN_READ
#undef KRN_HELD
#undef KRN_TURN
  } else {
#define KRN_SLICE(d, st, prev)                                                                                         \
    if (i + d >= n) break;                                                                                             \
    if (i + d + STAGES - 2 < n) KRN_VMWAIT((STAGES - 2) * LOADS); else KRN_VMWAIT(0);                                  \
    __builtin_amdgcn_s_waitcnt(0xc07f); /* lgkmcnt(0): this wave's reads of the stage refilled next */                 \
    __builtin_amdgcn_s_barrier();                                                                                      \
    if (i + d + STAGES - 1 < n) KRN_ISSUE(prev, i + d + STAGES - 1);                                                   \
    KRN_COMPUTE(st);
  for (int i = 0;; i += STAGES) {
    if constexpr (STAGES == 2) { KRN_SLICE(0, s0, s1) KRN_SLICE(1, s1, s0) }
    if constexpr (STAGES == 4) { KRN_SLICE(0, s0, s3) KRN_SLICE(1, s1, s0) KRN_SLICE(2, s2, s1) KRN_SLICE(3, s3, s2) }
  }
  }
#undef KRN_ISSUE
#undef KRN_ISSUE_TAIL
#undef KRN_COMPUTE
#undef KRN_VMWAIT
#undef KRN_SLICE
  __syncthreads();  // every wave is done with the ring before its LDS becomes the store patches
  store_blocks<FMT == FMT_I8>(acc, reinterpret_cast<uint32_t*>(lds), wave, C, part, ldc, m0 + wm * (BM / WM),
                              n0 + wn * (BN / WN), M, N, e, lane);
}

// C = epilogue(sum over the parts' planes), eight columns of a row per thread: bound by reading the planes, which the
// parts have just left in the caches (256 x 4096, four parts: 17 MB).
template <bool INT>
__global__ __launch_bounds__(256) void split_reduce(const uint8_t* __restrict__ planes, void* __restrict__ C, int64_t M,
                                                    int64_t N, int64_t ld, int parts, Epilogue e) {
  const int64_t per_row = ld / 8, at = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t m = at / per_row, n = at % per_row * 8;
  if (m >= M) return;
  typedef std::conditional_t<INT, i32x4, f32x4> V;
  const uint8_t* from = planes + (m * ld + n) * 4;
  V lo = *reinterpret_cast<const V*>(from), hi = *reinterpret_cast<const V*>(from + 16);
#pragma unroll 4
  for (int p = 1; p < parts; ++p) {
    from += M * ld * 4;
    lo += *reinterpret_cast<const V*>(from);
    hi += *reinterpret_cast<const V*>(from + 16);
  }
  const int live = (int)min((int64_t)8, N - n);
  if constexpr (INT) {
    if (e.out_kind == I32) {
      int32_t* out = static_cast<int32_t*>(C) + m * N + n;
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c < live) out[c] = c < 4 ? lo[c & 3] : hi[c & 3];
      return;
    }
  }
  float v[8];
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = (float)lo[c], v[4 + c] = (float)hi[c];
  for (int i = 0; i < e.nops; ++i) {
    const int op = e.op[i] & ((1 << VEC_KIND_SHIFT) - 1), kind = e.op[i] >> VEC_KIND_SHIFT;
    if (op >= RELU) {
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = activation(op, v[c]);
    } else if (op % 3 == 2) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float s = bits_value(kind, vec_bits(e.vec[i], kind, min(n + c, N - 1)));
        v[c] = op < 3 ? __fmul_rn(v[c], s) : __fadd_rn(v[c], s);
      }
    } else {
      const float s = op % 3 == 1 ? bits_value(kind, vec_bits(e.vec[i], kind, m)) : e.scalar[i];
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = op < 3 ? __fmul_rn(v[c], s) : __fadd_rn(v[c], s);
    }
  }
  if (e.out_kind == F32) {
    float* out = static_cast<float*>(C) + m * N + n;
    if (live == 8) {
      *reinterpret_cast<u32x4_any*>(out) = __builtin_bit_cast(u32x4, f32x4{v[0], v[1], v[2], v[3]});
      *reinterpret_cast<u32x4_any*>(out + 4) = __builtin_bit_cast(u32x4, f32x4{v[4], v[5], v[6], v[7]});
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c < live) out[c] = v[c];
    }
    return;
  }
  uint32_t h[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    h[c] = e.out_kind == BF16 ? f2bf2(v[2 * c], v[2 * c + 1])
                              : (uint32_t)f2h(v[2 * c]) | ((uint32_t)f2h(v[2 * c + 1]) << 16);
  uint16_t* out = static_cast<uint16_t*>(C) + m * N + n;
  if (live == 8) {
    *reinterpret_cast<u32x4_any*>(out) = u32x4{h[0], h[1], h[2], h[3]};
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (c < live) out[c] = (uint16_t)(h[c >> 1] >> ((c & 1) * 16));
  }
}

}  // namespace krn

using namespace krn;

static int launched(const char* what) {
  hipError_t err = hipGetLastError();
  if (err == hipSuccess) return 0;
  krn_set_error("%s launch: %s", what, hipGetErrorString(err));
  return (int)err;
}

int krn::launch_reduce(int fmt, int parts, const SplitCall& g) {
  const int64_t ld = split_ld(g.n);
  const dim3 blocks((unsigned)((g.m * (ld / 8) + 255) / 256));
  if (fmt == FMT_I8)
    hipLaunchKernelGGL(split_reduce<true>, blocks, dim3(256), 0, g.stream, (const uint8_t*)g.workspace, g.c, g.m, g.n,
                       ld, parts, g.e);
  else
    hipLaunchKernelGGL(split_reduce<false>, blocks, dim3(256), 0, g.stream, (const uint8_t*)g.workspace, g.c, g.m, g.n,
                       ld, parts, g.e);
  return launched("gemm reduction");
}

template <int FMT, int BM, int BN, int WM, int WN, int STAGES, bool PIPED, bool NN>
static int launch(const SplitCall& g, int parts) {  // STAGES = 0: the loader for any alignment
  const int64_t tiles = ((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN);
  int64_t ldc = g.n;
  Epilogue e = g.e;
  void* c = g.c;
  if (parts > 1) {
    c = g.workspace;
    ldc = split_ld(g.n);
    e = plane_epilogue(FMT);
  }
  const dim3 grid((unsigned)tiles, (unsigned)parts), block(WM * WN * 64);
  if constexpr (STAGES > 0)
    hipLaunchKernelGGL((gemm_ring<FMT, BM, BN, WM, WN, STAGES, PIPED, NN>), grid, block, 0, g.stream, (const uint8_t*)g.a,
                       (const uint8_t*)g.b, c, g.m, g.n, g.kbytes, g.lda, g.ldb, ldc, e, parts);
  else
    hipLaunchKernelGGL((gemm_any<FMT, BM, BN, WM, WN, NN>), grid, block, 0, g.stream, (const uint8_t*)g.a,
                       (const uint8_t*)g.b, c, g.m, g.n, g.kbytes, g.lda, g.ldb, ldc, e, parts);
  const int rc = launched("gemm");
  return rc != 0 || parts == 1 ? rc : launch_reduce(FMT, parts, g);
}

template <int FMT, bool NN>
static int launch_shape(const SplitCall& g, int shape, int parts) {
  switch (shape) {
    case RING_32x64: return launch<FMT, 32, 64, 1, 2, 4, false, NN>(g, parts);
    case RING_64x64: return launch<FMT, 64, 64, 2, 2, 4, false, NN>(g, parts);
    case RING_128x128: return launch<FMT, 128, 128, 2, 2, 2, false, NN>(g, parts);
    case RING_128x128_DEEP: return launch<FMT, 128, 128, 2, 2, 4, true, NN>(g, parts);
    case ANY_32x128: return launch<FMT, 32, 128, 1, 4, 0, false, NN>(g, parts);
    case ANY_64x64: return launch<FMT, 64, 64, 2, 2, 0, false, NN>(g, parts);
    default: return launch<FMT, 128, 128, 2, 2, 0, false, NN>(g, parts);
  }
}

int krn::launch_split(int fmt, bool nn, int shape, int parts, const SplitCall& g) {
  switch (fmt) {
    case FMT_BF16:
      return nn ? launch_shape<FMT_BF16, true>(g, shape, parts)
                : launch_shape<FMT_BF16, false>(g, shape, parts);
    case FMT_F16:
      return nn ? launch_shape<FMT_F16, true>(g, shape, parts)
                : launch_shape<FMT_F16, false>(g, shape, parts);
    case FMT_I8: return launch_shape<FMT_I8, false>(g, shape, parts);
    default: return launch_shape<FMT_FP8, false>(g, shape, parts);
  }
}
