// Tile GEMM for gfx950: C[m, n] = epilogue(sum_k A[m, k] * B[n, k]) with both operands K-contiguous.
//
// This is the lowering of krn's tile contraction `acc += a[rows, ks] @ b[cols, ks].transpose()` followed by
// `c[rows, cols] = f(acc).to(dtype)` (reference compiler/ir.py:309-315 Accumulate, compiler/emit.py:788-821). One
// workgroup owns a BM x BN output tile split among its waves, and every wave keeps its accumulators in registers as
// 32x32 MFMA blocks (`gemm_quad16`: 16x16 blocks of the transposed product). Main loops: `gemm_quad16` (every
// format, also the bf16/f16 NN form, 16x16 MFMAs) for whole 256 x 256 tiles of two K slices or more, `gemm_pipe`
// and `gemm_pp` (fp8) for one slice and, `gemm_pipe`, on 128 x 128 and 128 x 256 tiles for mid-size products,
// `gemm_skinny` for M <= 128 (rings of direct-to-LDS slices per wave); products that leave the chip idle there, unaligned
// rows and most K x N operands run on gemm_split.hip's kernels, and `gemm_tile` (bounds-checked, byte by byte) takes what
// is left: rows shorter than 16 bytes and panels past 31-bit offsets. `plan_of` chooses. All end in `store_tile` (`gemm_quad16`:
// `store_tile16t`): whole blocks straight from the accumulators (the direct epilogue), the rest through an LDS patch.
//
// One byte-oriented main loop serves three operand formats, because each MFMA consumes the same 16 bytes per lane
// per half-wave:
//   bf16 / f16 : v_mfma_f32_32x32x16_{bf16,f16}   16 elements = 32 bytes of K per step
//   int8       : v_mfma_i32_32x32x32_i8           32 elements = 32 bytes of K per step
//   fp8 e4m3   : v_mfma_scale_f32_32x32x64_f8f6f4 64 elements = 64 bytes of K per step (unit E8M0 scales)
// The K order inside one instruction is the hardware's; A and B fragments are read with the same byte layout, so
// every lane pairs A[m, k] with B[n, k] for the same k.
//
// LDS layout: a tile row of a K slice is 64 or 128 bytes (4 or 8 chunks of 16 bytes), swizzled per row so that
// the 16-byte fragment reads of 16 consecutive rows hit distinct banks (swz4 / swz8 below).
#include <mutex>

#include "gemm_split.h"

namespace krn {

// BM x BN tile, WM x WN waves, K sliced 128 bytes at a time. `kbytes` is K times the element size; rows of A and B
// are `lda`/`ldb` bytes apart. VEC: every row is 16-byte aligned and kbytes % 16 == 0, so 16-byte loads are legal.
template <int FMT, int BM, int BN, int WM, int WN, bool VEC>
__global__ __launch_bounds__(256, 1) void gemm_tile(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                    void* __restrict__ C, int64_t M, int64_t N, int64_t kbytes,
                                                    int64_t lda, int64_t ldb, int64_t ldc, Epilogue e) {
  typedef Mfma<FMT> Unit;
  typedef typename Unit::Acc Acc;
  constexpr int BKB = 128;             // bytes of K per slice
  constexpr int TM = BM / WM / 32;     // 32x32 blocks per wave along M
  constexpr int TN = BN / WN / 32;
  constexpr int STEP = Unit::kBytes;   // bytes of K per MFMA
  constexpr int CH = STEP / 32;        // 16-byte chunks per lane per MFMA operand
  constexpr int PA = BM / 32, PB = BN / 32;  // load passes (32 rows of 8 chunks per pass)
  static_assert(WM * WN == 4, "four waves");

  __shared__ u32x4 lds[2][(BM + BN) * 8];

  int tm, tn;
  tile_of((int)((M + BM - 1) / BM), (int)((N + BN - 1) / BN), tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int lrow = t >> 3, lchunk = t & 7;

  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Acc{};

  u32x4 ra[PA], rb[PB];
  const int nk = (int)((kbytes + BKB - 1) / BKB);

  // Global -> registers for K slice `kt`, registers -> LDS stage `s`. Written as macros, not lambdas: a lambda
  // capturing the staging arrays by reference takes their address and sends them to scratch memory.
#define KRN_LOAD(kt)                                                                                            \
  do {                                                                                                          \
    const int64_t kb = (int64_t)(kt) * BKB + lchunk * 16;                                                       \
    _Pragma("unroll") for (int p = 0; p < PA; ++p) {                                                            \
      const int64_t row = m0 + lrow + 32 * p;                                                                   \
      ra[p] = load16<VEC>(A, row * lda, kb, row < M, kbytes);                                                   \
    }                                                                                                           \
    _Pragma("unroll") for (int p = 0; p < PB; ++p) {                                                            \
      const int64_t row = n0 + lrow + 32 * p;                                                                   \
      rb[p] = load16<VEC>(B, row * ldb, kb, row < N, kbytes);                                                   \
    }                                                                                                           \
  } while (0)
#define KRN_STORE(s)                                                                                            \
  do {                                                                                                          \
    _Pragma("unroll") for (int p = 0; p < PA; ++p) {                                                            \
      const int row = lrow + 32 * p;                                                                            \
      lds[s][row * 8 + (lchunk ^ swz8(row))] = ra[p];                                                           \
    }                                                                                                           \
    _Pragma("unroll") for (int p = 0; p < PB; ++p) {                                                            \
      const int row = BM + lrow + 32 * p;                                                                       \
      lds[s][row * 8 + (lchunk ^ swz8(row))] = rb[p];                                                           \
    }                                                                                                           \
  } while (0)

  KRN_LOAD(0);
  KRN_STORE(0);
  __syncthreads();
  const int half = lane >> 5, r32 = lane & 31;
  for (int kt = 0; kt < nk; ++kt) {
    const int s = kt & 1;
    if (kt + 1 < nk) KRN_LOAD(kt + 1);
#pragma unroll
    for (int k = 0; k < BKB / STEP; ++k) {
      u32x4 fa[TM][CH], fb[TN][CH];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * (BM / WM) + i * 32 + r32;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const int chunk = (k * STEP + half * (STEP / 2)) / 16 + c;
          fa[i][c] = lds[s][row * 8 + (chunk ^ swz8(row))];
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = BM + wn * (BN / WN) + j * 32 + r32;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const int chunk = (k * STEP + half * (STEP / 2)) / 16 + c;
          fb[j][c] = lds[s][row * 8 + (chunk ^ swz8(row))];
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) Unit::step(acc[i][j], fa[i], fb[j]);
    }
    if (kt + 1 < nk) KRN_STORE(s ^ 1);
    __syncthreads();
  }

  // C layout of a 32x32 MFMA block: lane holds column (lane & 31) and rows (r/4)*8 + (lane/32)*4 + r%4. Each block
  // goes through a per-wave 32x33-word LDS patch so the global stores run along rows; only the register -> LDS
  // copy is unrolled, which keeps every accumulator index a compile-time constant (a runtime index would send the
  // whole accumulator array to scratch memory).
  uint32_t* patch = reinterpret_cast<uint32_t*>(&lds[0][0]) + wave * PATCH_WORDS;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      store_block<FMT == FMT_I8>(acc[i][j], patch, C, ldc, m0 + wm * (BM / WM) + i * 32,
                                 n0 + wn * (BN / WN) + j * 32, M, N, e, lane);
}

// The pipelined main loop for 256 x 256 tiles (the last row and column of tiles may be ragged; K a multiple of the
// BKB-byte slice, rows 16-byte aligned). Operand slices go straight from global memory into LDS (global_load_lds_dwordx4, no register staging)
// through a ring of STAGES buffers, so the loads of slice k + STAGES - 1 are in flight while slice k multiplies.
// One barrier per slice publishes the landed slice and frees the oldest buffer; it is a bare s_barrier, because the
// workgroup fence of __syncthreads() would wait for every outstanding load and drain the ring. A wave's load
// instruction fills 1 KiB of LDS contiguously (lane i -> slot i), so each lane fetches the global chunk that belongs
// at its swizzled slot. Fragments are double-buffered in registers: the LDS reads of step s + 1 (and, at the end of
// a slice, of the next slice) are issued before the MFMAs of step s, and the scheduler is told to interleave one
// LDS read or one global load with each MFMA, so the memory instructions issue in the shadow of the matrix core.
template <int BKB>
__device__ __forceinline__ int swzk(int row) {
  return BKB == 128 ? swz8(row) : swz4(row);
}

template <int FMT, int BM, int BN, int WM, int WN, int STAGES, int BKB>
__global__ __launch_bounds__(WM * WN * 64, 1) void gemm_pipe(const uint8_t* __restrict__ A,
                                                             const uint8_t* __restrict__ B, void* __restrict__ C,
                                                             int64_t M, int64_t N, int64_t kbytes, int64_t lda,
                                                             int64_t ldb, int64_t ldc, Epilogue e) {
  typedef Mfma<FMT> Unit;
  typedef typename Unit::Acc Acc;
  constexpr int THREADS = WM * WN * 64;
  constexpr int CPR = BKB / 16;              // 16-byte chunks per row
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int STEP = Unit::kBytes;         // bytes of K per MFMA
  constexpr int CH = STEP / 32;              // 16-byte chunks per lane per MFMA operand
  constexpr int KS = BKB / STEP;             // MFMA steps per slice
  constexpr int ROWS_PER_LOAD = 1024 / BKB;  // rows one wave load instruction fills
  constexpr int LOADS_A = BM / ROWS_PER_LOAD / (THREADS / 64), LOADS_B = BN / ROWS_PER_LOAD / (THREADS / 64);
  constexpr int LOADS = LOADS_A + LOADS_B;   // load instructions per wave per slice
  constexpr int STAGE_BYTES = (BM + BN) * BKB;
  constexpr int VMCNT = (STAGES - 2) * LOADS;
  // With three or more stages the A loads of a slice go between the first MFMAs and the B loads between the MFMAs
  // after the barrier, one load every four MFMAs: the workgroup's 32 loads of a slice no longer arrive at the
  // texture unit as one burst (bf16 8192^3 +2.5 %). At the barrier of slice kt the loads younger than slice kt + 1
  // are then slices kt + 2 .. kt + STAGES - 2 and the A loads of slice kt + STAGES - 1.
  constexpr bool SPREAD = STAGES >= 3;
  constexpr int VMCNT_SPLIT = SPREAD ? (STAGES - 3) * LOADS + LOADS_A : VMCNT;
  static_assert(KS % 2 == 0, "an even number of MFMA steps per slice");
  static_assert(LOADS_A * ROWS_PER_LOAD * (THREADS / 64) == BM && LOADS_B * ROWS_PER_LOAD * (THREADS / 64) == BN,
                "the tile splits into whole wave loads");
  static_assert(VMCNT <= 63, "vmcnt range");
  static_assert(STAGES * STAGE_BYTES <= 160 * 1024, "LDS of one CU");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * STAGE_BYTES];

  int tm, tn;
  tile_of((int)((M + BM - 1) / BM), (int)((N + BN - 1) / BN), tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int half = lane >> 5, r32 = lane & 31;

  // this lane's share of each wave load: its row within the 1 KiB block and the global chunk for its slot. Loads go
  // through buffer resources over this tile's A and B panels (base in SGPRs): a lane keeps one 32-bit panel offset
  // per load and the slice offset is an SGPR, so no address arithmetic runs per load (the host routes a tile here
  // only when its panel offsets fit in 31 bits). A panel's resource ends at the operand's last row: rows of a
  // ragged last tile past it load zeros, and their results are never stored.
  const int lrow = lane / CPR, lslot = lane % CPR;
  const __amdgpu_buffer_rsrc_t a_rsrc = panel_rsrc(A + m0 * lda, (M - m0) * lda),
                              b_rsrc = panel_rsrc(B + n0 * ldb, (N - n0) * ldb);
  uint32_t a_off_g[LOADS_A], b_off_g[LOADS_B];
#pragma unroll
  for (int j = 0; j < LOADS_A; ++j) {
    const int row = (wave * LOADS_A + j) * ROWS_PER_LOAD + lrow;
    a_off_g[j] = (uint32_t)(row * lda + (lslot ^ swzk<BKB>(row)) * 16);
  }
#pragma unroll
  for (int j = 0; j < LOADS_B; ++j) {
    const int row = (wave * LOADS_B + j) * ROWS_PER_LOAD + lrow;
    b_off_g[j] = (uint32_t)(row * ldb + (lslot ^ swzk<BKB>(row)) * 16);
  }
  // fragment offsets (16-byte units within a stage) of every MFMA operand this lane reads
  int a_off[TM][KS][CH], b_off[TN][KS][CH];
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int chunk = (k * STEP + half * (STEP / 2)) / 16 + c;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * (BM / WM) + i * 32 + r32;
        a_off[i][k][c] = row * CPR + (chunk ^ swzk<BKB>(row));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn * (BN / WN) + j * 32 + r32;
        b_off[j][k][c] = BM * CPR + row * CPR + (chunk ^ swzk<BKB>(row));
      }
    }
  const int nk = (int)(kbytes / BKB);

#define KRN_ISSUE(slice)                                                                                        \
  do {                                                                                                          \
    uint8_t* stage = lds + ((slice) % STAGES) * STAGE_BYTES;                                                    \
    const int koff = (slice) * BKB;                                                                             \
    _Pragma("unroll") for (int j = 0; j < LOADS_A; ++j)                                                         \
        buffer_to_lds16(a_rsrc, stage + (wave * LOADS_A + j) * 1024, a_off_g[j], koff);                         \
    _Pragma("unroll") for (int j = 0; j < LOADS_B; ++j)                                                         \
        buffer_to_lds16(b_rsrc, stage + BM * BKB + (wave * LOADS_B + j) * 1024, b_off_g[j], koff);              \
  } while (0)
  // vmcnt(n) with lgkmcnt and expcnt left alone (gfx9 s_waitcnt encoding), then every LDS read of this wave done
  // and the workgroup barrier
#define KRN_ISSUE_A(slice)                                                                                      \
  do {                                                                                                          \
    uint8_t* stage = lds + ((slice) % STAGES) * STAGE_BYTES;                                                    \
    const int koff = (slice) * BKB;                                                                             \
    _Pragma("unroll") for (int j = 0; j < LOADS_A; ++j)                                                         \
        buffer_to_lds16(a_rsrc, stage + (wave * LOADS_A + j) * 1024, a_off_g[j], koff);                         \
  } while (0)
#define KRN_ISSUE_B(slice)                                                                                      \
  do {                                                                                                          \
    uint8_t* stage = lds + ((slice) % STAGES) * STAGE_BYTES;                                                    \
    const int koff = (slice) * BKB;                                                                             \
    _Pragma("unroll") for (int j = 0; j < LOADS_B; ++j)                                                         \
        buffer_to_lds16(b_rsrc, stage + BM * BKB + (wave * LOADS_B + j) * 1024, b_off_g[j], koff);              \
  } while (0)
  // scheduling of the spread form: per load, MFMA read MFMA read MFMA load MFMA read (one load every four MFMAs)
#define KRN_SPREAD_A()                                                                                         \
  do {                                                                                                          \
    _Pragma("unroll") for (int q = 0; q < LOADS_A; ++q) {                                                       \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     \
    }                                                                                                           \
  } while (0)
#define KRN_SPREAD_B()                                                                                         \
  do {                                                                                                          \
    _Pragma("unroll") for (int q = 0; q < LOADS_B; ++q) {                                                       \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     \
    }                                                                                                           \
  } while (0)
#define KRN_PUBLISH(n)                                                                                          \
  do {                                                                                                          \
    __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00 | ((n) & 15) | (((n) >> 4) << 14));                              \
    __builtin_amdgcn_s_waitcnt(0xc07f & ~0x0f00);                                                               \
    __builtin_amdgcn_s_barrier();                                                                               \
  } while (0)
#define KRN_FRAGS(dst, slice, k)                                                                                \
  do {                                                                                                          \
    const u32x4* st = reinterpret_cast<const u32x4*>(lds + ((slice) % STAGES) * STAGE_BYTES);                   \
    _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int c = 0; c < CH; ++c)              \
        dst##a[i][c] = st[a_off[i][k][c]];                                                                      \
    _Pragma("unroll") for (int j = 0; j < TN; ++j) _Pragma("unroll") for (int c = 0; c < CH; ++c)              \
        dst##b[j][c] = st[b_off[j][k][c]];                                                                      \
  } while (0)
#define KRN_MMA(src)                                                                                            \
  _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int j = 0; j < TN; ++j)                 \
      Unit::step(acc[i][j], src##a[i], src##b[j])
  // scheduling hints: one LDS read (0x100) or one global load (0x020) between consecutive MFMAs (0x008)
#define KRN_WITH_READS()                                                                                        \
  _Pragma("unroll") for (int q = 0; q < (TM + TN) * CH; ++q) {                                                  \
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                                          \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                          \
  }
#define KRN_WITH_LOADS()                                                                                        \
  _Pragma("unroll") for (int q = 0; q < LOADS; ++q) {                                                           \
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                                                          \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                          \
  }

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) KRN_ISSUE(s);
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Acc{};
  u32x4 f0a[TM][CH], f0b[TN][CH], f1a[TM][CH], f1b[TN][CH];
  if (nk > STAGES - 2) {
    KRN_PUBLISH(VMCNT);
  } else {
    KRN_PUBLISH(0);
  }
  KRN_FRAGS(f0, 0, 0);
  int kt = 0;
  // steady state: every slice refills the ring (branch-free, so the scheduler can interleave)
  for (; kt + STAGES - 1 < nk; ++kt) {
#pragma unroll
    for (int k = 0; k < KS; k += 2) {
      KRN_FRAGS(f1, kt, k + 1);
      if constexpr (SPREAD) {
        if (k == 0) KRN_ISSUE_A(kt + STAGES - 1);
        KRN_MMA(f0);
        KRN_SPREAD_A();
      } else {
        if (k == 0) KRN_ISSUE(kt + STAGES - 1);
        KRN_MMA(f0);
        KRN_WITH_READS();
        if (k == 0) KRN_WITH_LOADS();
      }
      if (k + 2 < KS) {
        KRN_FRAGS(f0, kt, k + 2);
      } else {
        KRN_PUBLISH(VMCNT_SPLIT);
        KRN_FRAGS(f0, kt + 1, 0);
        if constexpr (SPREAD) KRN_ISSUE_B(kt + STAGES - 1);
      }
      KRN_MMA(f1);
      if constexpr (SPREAD) {
        KRN_SPREAD_B();
      } else {
        KRN_WITH_READS();
      }
    }
  }
  // drain: the last STAGES - 1 slices are already in flight
  for (; kt < nk; ++kt) {
#pragma unroll
    for (int k = 0; k < KS; k += 2) {
      KRN_FRAGS(f1, kt, k + 1);
      KRN_MMA(f0);
      KRN_WITH_READS();
      if (k + 2 < KS) {
        KRN_FRAGS(f0, kt, k + 2);
      } else if (kt + 1 < nk) {
        KRN_PUBLISH(0);
        KRN_FRAGS(f0, kt + 1, 0);
      }
      KRN_MMA(f1);
      KRN_WITH_READS();
    }
  }
#undef KRN_ISSUE
#undef KRN_PUBLISH
#undef KRN_FRAGS
#undef KRN_MMA
#undef KRN_WITH_READS
#undef KRN_WITH_LOADS
#undef KRN_ISSUE_A
#undef KRN_ISSUE_B
#undef KRN_SPREAD_A
#undef KRN_SPREAD_B
  __syncthreads();  // every wave is done with the ring before its LDS becomes the store patches

  uint32_t* patch = reinterpret_cast<uint32_t*>(lds) + wave * PATCH_WORDS;
  store_tile<FMT == FMT_I8>(acc, patch, C, ldc, m0 + wm * (BM / WM), n0 + wn * (BN / WN), M, N, e, lane);
}

// The four-wave main loop for whole 256 x 256 tiles with K a multiple of 128 bytes (bf16/f16 NT and NN, fp8, int8),
// on the 16x16 MFMA forms. Each wave owns a 128 x 128 quarter (wave w: rows 128 (w >> 1), columns 128 (w & 1)) as
// 8 x 8 accumulator blocks of 16 x 16 in AGPRs, each computed transposed (B A^T: the B fragment is the MFMA's first
// operand), so that a lane holds four columns of one row for the store (`store_tile16t`). 128-byte K slices go straight from global memory into LDS stages,
// two for A and three for B (5 x 32 KiB fill the 160 KiB), each stage a separate array so that the compiler can tell
// every fragment read from the loads in flight into the other stages; wave w loads rows 64 w .. 64 w + 63 of A and
// of B, 8 rows (1 KiB) per load, chunk c of row r at slot c ^ ((r >> 1) & 7).
//
// bf16/f16/int8: a slice is two steps of 64 bytes of K; fp8: one step of 128 (16x16x128). One set of fragments (A
// blocks 0-3 and B blocks 0-3 of 32 rows, each two 16-row halves) is refilled in place: steps alternate between
// running their 16 blocks of 32 x 32 row by row (block (I, J) is group 4 I + J of four MFMAs) and column by column,
// so a block's fragments are dead after its last group of the step and take the next step's at once (row order
// frees A block I after group 4 I + 3 and B block J after 12 + J; column order frees B block J after 4 J + 3 and A
// block I after 12 + I). The one barrier per slice sits after group 3 of its last step: by then this wave has read
// all of slice kt and its loads of slice kt + 1 have landed. B's slice kt + 2 is loaded during the slice, before
// and after the barrier (into the stage slice kt - 1 left, free since the last barrier), one load every other group;
// A's slice kt + 2 after the barrier, one load per group, into the stage slice kt leaves. Loads issued in a burst
// (the 16 of a slice in 8 groups) ask the vector memory path for twice what it delivers and stall the MFMA issue
// behind them (bf16 8192^3: 1452 TFLOP/s spread against 1392, MFMA busy 0.79 against 0.71; 0.84 with no loads).
//
// Measured against the 32x32 forms: MFMA-only loops on random operands sustain 16 % (bf16) and 25 % (int8) more
// on 16x16 at the same power limit; bf16 8192^3 on the register-staged 32x32 loop 1335 TFLOP/s, W8A8 M = 4096 on
// the eight-wave 32x32 loop 0.275 ms against 0.269; fp8 8192^3 equal (0.442 ms), the 16x16 form at a higher clock
// with proportionally less MFMA time.
template <int FMT, bool NN = false>
__global__ __launch_bounds__(256, 1) void gemm_quad16(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                     void* __restrict__ C, int64_t M, int64_t N, int64_t kbytes,
                                                     int64_t lda, int64_t ldb, int64_t ldc, Epilogue e) {
  constexpr int NA = 2, NB = 3;  // LDS stages of A and B
  typedef Mfma16<FMT> Unit;
  typedef typename Unit::Acc Acc;
  typedef typename Mfma<FMT>::Acc Acc32;
  // fp8: one 16x16x128 step per slice, 32 bytes of K per lane and operand; otherwise two steps of 16 bytes
  constexpr bool F8 = FMT == FMT_FP8;
  constexpr int NSTEP = F8 ? 1 : 2;
  typedef typename std::conditional<F8, i32x8, u32x4>::type Frag;
  static_assert(!NN || FMT == FMT_BF16 || FMT == FMT_F16, "NN: 16-bit operands");
  constexpr int BM = 256, BN = 256, BKB = 128;
  constexpr int HALF = BM * BKB;  // 32 KiB: one operand's rows of one slice
  constexpr int UNROLL = 6;  // slices per loop iteration: every stage index a constant
  __shared__ __attribute__((aligned(1024))) uint8_t la0[HALF];
  __shared__ __attribute__((aligned(1024))) uint8_t la1[HALF];
  __shared__ __attribute__((aligned(1024))) uint8_t lb0[HALF];
  __shared__ __attribute__((aligned(1024))) uint8_t lb1[HALF];
  __shared__ __attribute__((aligned(1024))) uint8_t lb2[HALF];
  int tm, tn;
  tile_of((int)((M + BM - 1) / BM), (int)((N + BN - 1) / BN), tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  auto uniform = [](const void* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const void*)(((uint64_t)hi << 32) | lo);
  };
  const int64_t a_bytes = __builtin_amdgcn_readfirstlane((int)min((M - m0) * lda, (int64_t)0x7fffffff));
  // NN: the panel is columns n0 .. n0 + 255 of every row of B (the host checks that it is addressable)
  const int64_t b_bytes = __builtin_amdgcn_readfirstlane(
      NN ? (int)((kbytes / 2 - 1) * ldb + BN * 2) : (int)min((N - n0) * ldb, (int64_t)0x7fffffff));
  const __amdgpu_buffer_rsrc_t a_rsrc = panel_rsrc(uniform(A + m0 * lda), a_bytes),
                              b_rsrc = panel_rsrc(uniform(B + (NN ? n0 * 2 : n0 * ldb)), b_bytes);
  // load item j of an operand: rows 64 wave + 8 j .. + 7; lane i takes row i / 8 and the global chunk that belongs at
  // slot i % 8. The swizzle of row 8 j + i / 8 depends on j only through j & 1.
  const int lrow = lane >> 3, lslot = lane & 7;
  uint32_t ga[2], gb[4];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int row = wave * 64 + p * 8 + lrow;
    ga[p] = (uint32_t)(row * lda + ((lslot ^ swz8(row)) * 16));
    gb[p] = (uint32_t)(row * ldb + ((lslot ^ swz8(row)) * 16));
  }
  // NN: a slice of B is 64 k rows of 512 bytes ([k][n]); wave w loads k rows 16 w .. 16 w + 15, two per load (item
  // j: rows 16 w + 2 j + i / 32, lane i at slot i % 32). Chunk c of row k sits at slot c ^ nn_swz(k), which puts the
  // 8 rows a transposed fragment read serves per pass on 8 distinct 32-byte bank groups. The lane offsets depend on
  // j through j & 1 and j >> 2; the rest is the scalar offset 2 j ldb.
  auto nn_swz = [](int k) { return 2 * ((k & 3) | (((k >> 3) & 1) << 2)); };
  if constexpr (NN) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = (q >> 1) * 4 + (q & 1);
      const int krow = wave * 16 + 2 * j + (lane >> 5), slot = lane & 31;
      gb[q] = (uint32_t)((wave * 16 + (lane >> 5)) * ldb + ((slot ^ nn_swz(krow)) * 16));
    }
  }
  // NN fragment reads (ds_read_b64_tr_b16): lane L = 16 g + a reads k row 8 g + 4 p + a / 4 (part p) of the step's
  // 32 and columns 4 (a % 4) .. + 3 of its 16, and receives column a of the 16 at the four k of the part
  const int tg = lane >> 4, ta = lane & 15;
  const int tr_row = (8 * tg + (ta >> 2)) * 512, tr_swz = nn_swz(8 * tg + (ta >> 2));
  const int tr_col = wn * 128 + 4 * (ta & 3);
  const int wbase = wave * 8192;
  // fragment bases: lane L reads row L & 15 of a 16-row half, 16-byte chunk 4 x + (L >> 4) (step x), or for fp8
  // chunks 2 (L >> 4) + x (x = 0, 1: the lane's 32 bytes)
  int ra[2], rb[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int chunk = F8 ? 2 * (lane >> 4) + x : 4 * x + (lane >> 4);
    const int part = (lane & 15) * 128 + ((chunk ^ (((lane & 15) >> 1) & 7)) * 16);
    ra[x] = part + wm * 128 * 128;
    rb[x] = part + wn * 128 * 128;
  }
  const int one = 127;  // fp8: the unit E8M0 scale
  const int nk = (int)(kbytes / BKB);  // >= 2 (host)

  Frag F[16];  // A block I half R at 2 I + R, B block J half Q at 8 + 2 J + Q
  Acc acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = Acc{};

#define KD_A(p) ((p) == 0 ? la0 : la1)
#define KD_B(p) ((p) == 0 ? lb0 : (p) == 1 ? lb1 : lb2)
#define KD_LOADA(j, sl, pa)                                                                                    \
  buffer_to_lds16(a_rsrc, KD_A(pa) + wbase + (j) * 1024, ga[(j) & 1], (int)((sl) * BKB + ((j) & 6) * 8 * lda))
#define KD_LOADB(j, sl, pb)                                                                                    \
  do {                                                                                                         \
    if constexpr (NN)                                                                                          \
      buffer_to_lds16(b_rsrc, KD_B(pb) + wbase + (j) * 1024, gb[((j) >> 2) * 2 + ((j) & 1)],                   \
                      (int)(((sl) * 64 + 2 * (j)) * ldb));                                                     \
    else                                                                                                       \
      buffer_to_lds16(b_rsrc, KD_B(pb) + wbase + (j) * 1024, gb[(j) & 1],                                      \
                      (int)((sl) * BKB + ((j) & 6) * 8 * ldb));                                                \
  } while (0)
#define KD_TR(pb, s, p, col)                                                                                   \
  __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s16*)( \
                                KD_B(pb) + tr_row + ((s) * 32 + (p) * 4) * 512 +                               \
                                ((((col) >> 3) ^ tr_swz) * 16) + ((col) & 7) * 2)))
#define KD_READ(r, c, pa, pb, s)                                                                               \
  do {                                                                                                         \
    if constexpr (F8) {                                                                                        \
      const uint8_t* p8 = ((r) < 4 ? KD_A(pa) : KD_B(pb)) + (((r) & 3) * 32 + (c) * 16) * 128;                 \
      const u32x4 lo = *reinterpret_cast<const u32x4*>(p8 + ((r) < 4 ? ra[0] : rb[0]));                        \
      const u32x4 hi = *reinterpret_cast<const u32x4*>(p8 + ((r) < 4 ? ra[1] : rb[1]));                        \
      F[(r) * 2 + (c)] = Frag{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],                                   \
                              (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};                                 \
    } else {                                                                                                   \
      if (NN && (r) >= 4) {                                                                                    \
        const int col = tr_col + ((r) - 4) * 32 + (c) * 16;                                                    \
        const u32x2 lo = KD_TR(pb, s, 0, col), hi = KD_TR(pb, s, 1, col);                                      \
        F[(r) * 2 + (c)] = u32x4{lo[0], lo[1], hi[0], hi[1]};                                                  \
      } else {                                                                                                 \
        F[(r) * 2 + (c)] = *reinterpret_cast<const u32x4*>(                                                    \
            ((r) < 4 ? KD_A(pa) + ra[s] : KD_B(pb) + rb[s]) + (((r) & 3) * 32 + (c) * 16) * 128);              \
      }                                                                                                        \
    }                                                                                                          \
  } while (0)
#define KD_FENCE() __builtin_amdgcn_sched_barrier(0)
#define KD_MMA(I, J)                                                                                           \
  _Pragma("unroll") for (int R = 0; R < 2; ++R) _Pragma("unroll") for (int Q = 0; Q < 2; ++Q) {               \
    if constexpr (F8)                                                                                          \
      Unit::step_agpr(acc[(I) * 2 + R][(J) * 2 + Q], F[8 + (J) * 2 + Q], F[(I) * 2 + R], one);                \
    else                                                                                                       \
      Unit::step_agpr(acc[(I) * 2 + R][(J) * 2 + Q], F[8 + (J) * 2 + Q], F[(I) * 2 + R]);                     \
  }
  // One step of slice kt (A stage PA, B stage PB). ORD 0: its 16 blocks row by row (group g = 4 I + J), 1: column
  // by column (g = 4 J + I); either way A block I is dead after its group with J = 3 and B block J after its group
  // with I = 3, and the next step's fragments of that block are read at once (ORD 0 reads A first, 1 reads B first).
  // The next step is step s + 1 of this slice, or (LAST) step 0 of slice kt + 1. In the last step, after group 3,
  // the barrier (this wave's loads of slice kt + 1 landed: only the loads of a three-stage operand's slice kt + 2,
  // issued last, may still be in flight), then the loads into the stages slice kt leaves, two-stage operands first
  // (past the end: the last slice again, into a stage nothing reads any more).
#define KD_STEP(PA, PB, ORD, LAST, kt, s)                                                                      \
  do {                                                                                                         \
    const int NA_ = (LAST) ? ((PA) + 1) % NA : (PA), NB_ = (LAST) ? ((PB) + 1) % NB : (PB);                    \
    const int NS_ = (LAST) ? 0 : (s) + 1;                                                                      \
    _Pragma("unroll") for (int g = 0; g < 16; ++g) {                                                           \
      const int I = (ORD) ? (g & 3) : (g >> 2), J = (ORD) ? (g >> 2) : (g & 3);                                \
      KD_MMA(I, J);                                                                                            \
      KD_FENCE();                                                                                              \
      if ((LAST) && g == 3) {                                                                                  \
        /* still in flight may be only B's slice kt + 2: its loads of step 0 (eight), or of this step's groups 0  \
           and 2 (fp8) */                                                                                      \
        if constexpr (NSTEP == 1)                                                                              \
          __builtin_amdgcn_s_waitcnt(0x0070 | 2); /* vmcnt(2) lgkmcnt(0) */                                     \
        else                                                                                                   \
          __builtin_amdgcn_s_waitcnt(0x0070 | 8); /* vmcnt(8) lgkmcnt(0) */                                     \
        __builtin_amdgcn_s_barrier();                                                                          \
        KD_FENCE();                                                                                            \
      }                                                                                                        \
      if ((NSTEP == 1 || !(LAST)) && (NSTEP == 1 ? (g & 1) == 0 : (g & 1))) {                                  \
        KD_LOADB(g >> 1, min((kt) + 2, nk - 1), ((PB) + 2) % NB);                                              \
        KD_FENCE();                                                                                            \
      }                                                                                                        \
      if ((LAST) && g >= 3 && g < 11) { /* (spread over groups 3-15 instead: 0.4 % slower) */                  \
        KD_LOADA(g - 3, min((kt) + 2, nk - 1), PA);                                                            \
        KD_FENCE();                                                                                            \
      }                                                                                                        \
      _Pragma("unroll") for (int o = 0; o < 2; ++o) {                                                          \
        if ((o == 0) == ((ORD) == 0) && J == 3) {                                                              \
          KD_READ(I, 0, NA_, NB_, NS_);                                                                        \
          KD_READ(I, 1, NA_, NB_, NS_);                                                                        \
          KD_FENCE();                                                                                          \
        }                                                                                                      \
        if ((o == 0) == ((ORD) == 1) && I == 3) {                                                              \
          KD_READ(4 + J, 0, NA_, NB_, NS_);                                                                    \
          KD_READ(4 + J, 1, NA_, NB_, NS_);                                                                    \
          KD_FENCE();                                                                                          \
        }                                                                                                      \
      }                                                                                                        \
    }                                                                                                          \
  } while (0)
  // slice u of an unrolled run (u even at the start of a run, so that the order alternates from step to step):
  // step 0 row by row, step 1 column by column; fp8's one step per slice alternates from slice to slice
#define KD_SLICE(u, kt)                                                                                        \
  do {                                                                                                         \
    if constexpr (NSTEP == 2) {                                                                                \
      KD_STEP((u) % NA, (u) % NB, 0, false, kt, 0);                                                            \
      KD_STEP((u) % NA, (u) % NB, 1, true, kt, 1);                                                             \
    } else {                                                                                                   \
      KD_STEP((u) % NA, (u) % NB, (u) & 1, true, kt, 0);                                                       \
    }                                                                                                          \
  } while (0)

  // the prologue: slices 0 and 1 of A and B (B's slice 2 loads during slice 0, as in the loop); once slice 0 has
  // landed everywhere, its step-0 fragments
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) {
#pragma unroll
    for (int j = 0; j < 8; ++j) KD_LOADA(j, min(sl, nk - 1), sl);
#pragma unroll
    for (int j = 0; j < 8; ++j) KD_LOADB(j, min(sl, nk - 1), sl);
  }
#define KD_VMWAIT(n) __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00 | ((n) & 15) | (((n) >> 4) << 14))
  KD_VMWAIT(16);  // slice 0's 16 loads came first
  __builtin_amdgcn_s_barrier();
  KD_FENCE();
  // in the order step 1 reads them (B0 B1 B2 A0 A1 A2 B3 A3), so that the loop's first MFMAs wait on the same
  // partial LDS count whether they follow this or the loop's last step
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const int r = x < 3 ? 4 + x : x < 6 ? x - 3 : x == 6 ? 7 : 3;
    KD_READ(r, 0, 0, 0, 0);
    KD_READ(r, 1, 0, 0, 0);
    KD_FENCE();
  }
  int kt = 0;
  for (; kt + UNROLL <= nk; kt += UNROLL) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) KD_SLICE(u, kt + u);
  }
  // W8A8's scale vectors go out before the last (up to five) slices, so that their latency runs under MFMAs
  const int64_t row0 = m0 + wm * 128, col0 = n0 + wn * 128;
  const bool direct = quad16_direct(e, C, ldc, row0, col0, M, N), rowcol = direct && quad16_is_rowcol(e);
  Quad16RowCol rc;
  if (rowcol) quad16_rowcol(rc, e, row0, col0, lane);
#pragma unroll
  for (int u = 0; u < UNROLL - 1; ++u)
    if (kt + u < nk) KD_SLICE(u, kt + u);
#undef KD_A
#undef KD_B
#undef KD_LOADA
#undef KD_LOADB
#undef KD_READ
#undef KD_FENCE
#undef KD_MMA
#undef KD_STEP
#undef KD_SLICE
#undef KD_TR
#undef KD_VMWAIT
  __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00);  // vmcnt(0): no load still writes the stages
  // the MFMAs are assembly, so the compiler inserts no wait states between the last of them and the first read of
  // their results: 24 cycles cover the longest 16x16 form
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  __syncthreads();  // every wave is done with the stages before their LDS becomes the store patches
  uint32_t* patch = reinterpret_cast<uint32_t*>(la0) + wave * PATCH_WORDS;
  store_tile16t<FMT == FMT_I8, Acc32>(acc, direct, rowcol, rc, patch, C, ldc, row0, col0, M, N, e, lane);
}

// Ping-pong main loop for whole 256 x 256 tiles with 64-byte K slices (bf16/f16: two 32x32x16 steps, int8: two
// 32x32x32 steps, fp8: one 32x32x64 step per slice -- 512 MFMA cycles per wave in every format). Eight waves form two
// groups of four: group g owns rows [128 g, 128 g + 128) of the tile, and within a group wave q owns the 64 x 128
// block (q >> 1, q & 1). Waves w and w + 4 run on the same SIMD, and group 1 starts one barrier late, so on every
// SIMD one wave issues its 16 MFMAs while the other reads its next fragments from LDS and issues direct-to-LDS loads:
// the matrix core is fed from one wave while the other's LDS and memory waits are hidden behind it.
//
// Every slot ends in a workgroup barrier. Per slice j a wave runs a memory phase (issue its part of the loads of
// slice j + STAGES - 1, read the fragments of slice j, wait for them and for its own loads of slice j + 1) and then
// a compute phase (the MFMAs of slice j). Group 0 loads the A rows of every slice, group 1 the B rows. Slice j is
// read by group 0 in slot 2j and by group 1 in slot 2j + 1, so its stage is free from slot 2j + 2 on, which is when
// the loads of slice j + STAGES (same stage) are issued at the earliest.
template <int FMT, int STAGES>
__global__ __launch_bounds__(512, 1) void gemm_pp(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                  void* __restrict__ C, int64_t M, int64_t N, int64_t kbytes,
                                                  int64_t lda, int64_t ldb, int64_t ldc, Epilogue e) {
  typedef Mfma<FMT> Unit;
  typedef typename Unit::Acc Acc;
  constexpr int BM = 256, BN = 256, BKB = 64, CPR = 4;  // 64-byte slice rows of four 16-byte chunks
  constexpr int TM = 2, TN = 4;                          // 32x32 blocks per wave
  constexpr int STEP = Unit::kBytes, CH = STEP / 32, KS = BKB / STEP;
  constexpr int PART = BM * BKB;                         // bytes of one operand's rows in a stage (16 KiB)
  constexpr int STAGE_BYTES = 2 * PART;
  constexpr int LOADS = PART / 1024 / 4;                 // 1 KiB wave loads per wave per slice (4)
  constexpr int VMWAIT = (STAGES - 2) * LOADS;
  static_assert(STAGES >= 3 && STAGES * STAGE_BYTES <= 160 * 1024, "LDS of one CU");
  static_assert(VMWAIT <= 63, "vmcnt range");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * STAGE_BYTES];

  int tm, tn;
  tile_of((int)((M + BM - 1) / BM), (int)((N + BN - 1) / BN), tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave >> 2, q = wave & 3;
  const int half = lane >> 5, r32 = lane & 31;

  // loads: group 0 fills the A part of a stage, group 1 the B part; wave q the rows [64 q, 64 q + 64)
  const int lrow = lane / CPR, lslot = lane % CPR;
  // through a buffer resource over the group's panel, as in gemm_pipe
  const __amdgpu_buffer_rsrc_t rsrc = g ? panel_rsrc(B + n0 * ldb, (N - n0) * ldb) : panel_rsrc(A + m0 * lda, (M - m0) * lda);
  uint32_t src_off[LOADS];
  {
    const int64_t ld = g ? ldb : lda;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int row = (q * LOADS + j) * 16 + lrow;
      src_off[j] = (uint32_t)(row * ld + (lslot ^ swz4(row)) * 16);
    }
  }
  const int dst0 = g * PART + q * LOADS * 1024;
  // fragment offsets (16-byte units within a stage)
  const int wr = g * 128 + (q >> 1) * 64, wc = (q & 1) * 128;
  int a_off[TM][KS][CH], b_off[TN][KS][CH];
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int chunk = (k * STEP + half * (STEP / 2)) / 16 + c;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wr + i * 32 + r32;
        a_off[i][k][c] = row * CPR + (chunk ^ swz4(row));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wc + j * 32 + r32;
        b_off[j][k][c] = BM * CPR + row * CPR + (chunk ^ swz4(row));
      }
    }
  const int nk = (int)(kbytes / BKB);

#define KRN_ISSUE(slice)                                                                                        \
  do {                                                                                                          \
    uint8_t* stage = lds + ((slice) % STAGES) * STAGE_BYTES + dst0;                                             \
    const int koff = (slice) * BKB;                                                                             \
    _Pragma("unroll") for (int j = 0; j < LOADS; ++j) buffer_to_lds16(rsrc, stage + j * 1024, src_off[j], koff); \
  } while (0)
#define KRN_VMWAIT(n) __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00 | ((n) & 15) | (((n) >> 4) << 14))
#define KRN_LGKWAIT() __builtin_amdgcn_s_waitcnt(0xc07f & ~0x0f00)

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) KRN_ISSUE(s);
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = Acc{};
  if (nk > STAGES - 2) {
    KRN_VMWAIT(VMWAIT);
  } else {
    KRN_VMWAIT(0);
  }
  __builtin_amdgcn_s_barrier();
  if (g == 1) __builtin_amdgcn_s_barrier();
  u32x4 fa[KS][TM][CH], fb[KS][TN][CH];
  for (int kt = 0; kt < nk; ++kt) {
    // memory phase
    const bool refill = kt + STAGES - 1 < nk;
    if (refill) KRN_ISSUE(kt + STAGES - 1);
    {
      const u32x4* st = reinterpret_cast<const u32x4*>(lds + (kt % STAGES) * STAGE_BYTES);
#pragma unroll
      for (int k = 0; k < KS; ++k) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int c = 0; c < CH; ++c) fa[k][i][c] = st[a_off[i][k][c]];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int c = 0; c < CH; ++c) fb[k][j][c] = st[b_off[j][k][c]];
      }
    }
    KRN_LGKWAIT();
    if (refill) {
      KRN_VMWAIT(VMWAIT);
    } else {
      KRN_VMWAIT(0);
    }
    __builtin_amdgcn_s_barrier();
    // compute phase
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) Unit::step(acc[i][j], fa[k][i], fb[k][j]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
  }
  if (g == 0) __builtin_amdgcn_s_barrier();
#undef KRN_ISSUE
#undef KRN_VMWAIT
#undef KRN_LGKWAIT
  __syncthreads();  // every wave is done with the ring before its LDS becomes the store patches

  uint32_t* patch = reinterpret_cast<uint32_t*>(lds) + wave * PATCH_WORDS;
  store_tile<FMT == FMT_I8>(acc, patch, C, ldc, m0 + wr, n0 + wc, M, N, e, lane);
}

// Skinny products (M <= 128), the HBM-bound shapes: B (N x K) is streamed from HBM once and A (M x K) is read by
// every workgroup from L2. A workgroup owns 32 output columns and all M rows (MT blocks of 32); its WAVES waves split
// K, wave w taking one contiguous run of 128-byte K slices (runs far apart in a row keep each wave's HBM requests on
// few DRAM pages). Each wave moves its slices of A and B into its own LDS ring with direct-to-LDS loads that cover 8
// whole 128-byte rows per instruction, then reads the MFMA operands from LDS: loads with one lane per row (32 rows x
// 16 bytes per instruction) would fetch every line four times. Row R of a staged slice holds its 16-byte chunk c at
// position c ^ ((R >> 1) & 7), so a ds_read_b128 of one chunk from 16 consecutive rows touches all 64 banks once.
// Lane (r32, half) takes chunks half * 4 + q of its row for A and for B alike, and MFMA step s the s-th 16 bytes of
// them (32 bytes for fp8): both operands see the same K permutation, so the dot products are unchanged. The ring has
// STAGES stages per wave, STAGES - 1 slices in flight while one is multiplied. The partial sums meet in LDS, and
// waves 0..MT-1 each store one 32 x 32 block through the common epilogue.
template <int FMT, int MT, int WAVES, int STAGES, bool ACT, int AL = MT * 4>
__global__ __launch_bounds__(WAVES * 64, 1) void gemm_skinny(const uint8_t* __restrict__ A,
                                                              const uint8_t* __restrict__ B, void* __restrict__ C,
                                                              int64_t M, int64_t N, int64_t kbytes, int64_t lda,
                                                              int64_t ldb, int64_t ldc, Epilogue e, int parts) {
  typedef Mfma<FMT> Unit;
  typedef typename Unit::Acc Acc;
  typedef std::conditional_t<FMT == FMT_I8, int, float> Elem;
  constexpr int CH = Unit::kBytes / 32;       // 16-byte registers per lane per MFMA step
  constexpr int STEPS = 4 / CH;               // MFMA steps per 128-byte slice
  constexpr int STAGE = (MT + 1) * 4096;      // one slice: MT * 32 rows of A, then 32 rows of B, 128 bytes each
  constexpr int LOADS = AL + 4;               // DMA instructions per slice: AL of A's rows (8 each), 4 of B's
  static_assert(AL >= 1 && AL <= MT * 4, "A loads cover at most the ring's A rows");
  constexpr int AHEAD = (STAGES - 1) * LOADS; // loads still in flight when the oldest slice is waited for
  constexpr int RING_WORDS = WAVES * STAGES * STAGE / 4;
  constexpr int RED_WORDS = WAVES * MT * 16 * 64;
  constexpr int W1 = RING_WORDS > RED_WORDS ? RING_WORDS : RED_WORDS;
  constexpr int LDS_WORDS = W1 > WAVES * PATCH_WORDS ? W1 : WAVES * PATCH_WORDS;
  static_assert(LDS_WORDS * 4 <= 160 * 1024, "the ring exceeds the LDS of a CU");
  __shared__ __attribute__((aligned(16))) uint32_t lds[LDS_WORDS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, r32 = lane & 31;
  const int64_t n0 = (int64_t)blockIdx.x * 32;
  // DMA instruction j fills rows 8 j .. 8 j + 7 of the stage (A's rows first, then B's); lane L lands at position
  // L & 7 of row 8 j + (L >> 3) and so fetches the chunk that the swizzle puts there. Rows past the end of A or B
  // read the last row: their results are never stored.
  // Only the first AL eight-row groups of A are loaded: the ring rows past them hold whatever the LDS held, and
  // their results (rows >= 8 AL >= M) are never stored.
  const uint8_t* src[LOADS];
  int dst[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int g = j < AL ? j : MT * 4 + (j - AL);  // eight-row group of the stage
    const int chunk = (lane & 7) ^ (((g & 3) * 4 + (lane >> 4)) & 7);
    const int64_t row = g * 8 + (lane >> 3);  // row of the stage
    src[j] = j < AL ? A + min(row, M - 1) * lda + chunk * 16 : B + min(n0 + row - MT * 32, N - 1) * ldb + chunk * 16;
    dst[j] = g * 1024;
  }
  uint8_t* ring = reinterpret_cast<uint8_t*>(lds) + wave * STAGES * STAGE;
  int rd[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) rd[q] = r32 * 128 + (((half * 4 + q) ^ ((r32 >> 1) & 7)) * 16);
  const int slices = (int)(kbytes / 128), part = blockIdx.y;
  int from = 0, nk = slices;  // this workgroup's slices
  if (parts > 1) {
    from = slices * part / parts;
    nk = slices * (part + 1) / parts - from;
    C = static_cast<uint8_t*>(C) + part * (M * ldc * 4);
  }
  const int per = nk / WAVES, rem = nk % WAVES;
  const int begin = from + wave * per + min(wave, rem), cnt = per + (wave < rem ? 1 : 0);
  // the storing waves fetch the epilogue's vector operands now: loads issued at the very end of a workgroup would
  // wait behind the other workgroups' streams
  EpiPre pre;
  if (e.nops > 0) epi_prefetch(pre, e, A, (int64_t)wave * 32, n0, M, N, lane);
  Acc acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = Acc{};
  auto issue = [&](int slice, int stage) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads of the stage are done before it is refilled
    const int64_t off = (int64_t)slice * 128;
#pragma unroll
    for (int j = 0; j < AL; ++j)
      __builtin_amdgcn_global_load_lds((const void*)(src[j] + off),
                                       (__attribute__((address_space(3))) void*)(ring + stage * STAGE + dst[j]), 16,
                                       0, 0);
    // B (the weights, read once) streams non-temporally when M <= 32: fp8 M = 1 13.4 -> 11.8 us, M = 16 13.4 ->
    // 12.5 us, W8A8 M = 16 12.6 -> 12.0 us. With four row blocks (M = 128) it was 22 % slower, so A-heavy shapes
    // keep the default policy.
#pragma unroll
    for (int j = AL; j < LOADS; ++j)
      __builtin_amdgcn_global_load_lds((const void*)(src[j] + off),
                                       (__attribute__((address_space(3))) void*)(ring + stage * STAGE + dst[j]), 16,
                                       0, MT == 1 ? 2 : 0);
  };
  auto consume = [&](int stage) {
    const uint8_t* base = ring + stage * STAGE;
    u32x4 ra[MT][4], rb[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) rb[q] = *reinterpret_cast<const u32x4*>(base + MT * 4096 + rd[q]);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) ra[t][q] = *reinterpret_cast<const u32x4*>(base + t * 4096 + rd[q]);
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int t = 0; t < MT; ++t) Unit::step(acc[t], &ra[t][s * CH], &rb[s * CH]);
  };
#pragma unroll
  for (int p = 0; p < STAGES - 1; ++p)
    if (p < cnt) issue(begin + p, p);
  // steady state: STAGES slices per iteration, so every stage index is a constant and there are no branches (the
  // waits stay exact); vmcnt(AHEAD) = all but the newest STAGES - 1 slices have landed (gfx9 s_waitcnt encoding,
  // other counters left free)
  int i = 0;
  for (; i + 2 * STAGES - 2 < cnt; i += STAGES) {
#pragma unroll
    for (int j = 0; j < STAGES; ++j) {
      issue(begin + i + j + STAGES - 1, (j + STAGES - 1) % STAGES);
      __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00 | (AHEAD & 15) | ((AHEAD >> 4) << 14));
      consume(j);
    }
  }
  // at most 2 * STAGES - 2 slices are left, and i is a multiple of STAGES
#pragma unroll
  for (int j = 0; j < 2 * STAGES - 2; ++j) {
    if (i + j < cnt) {
      if (i + j + STAGES - 1 < cnt) issue(begin + i + j + STAGES - 1, (j + STAGES - 1) % STAGES);
      __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00);  // vmcnt(0)
      consume(j % STAGES);
    }
  }
  __syncthreads();  // the partial sums overwrite other waves' rings
  Elem* partial = reinterpret_cast<Elem*>(lds);
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) partial[((wave * MT + t) * 16 + r) * 64 + lane] = acc[t][r];
  __syncthreads();
  Acc sum = Acc{};
  if (wave < MT) {
    for (int v = 0; v < WAVES; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[r] += partial[((v * MT + wave) * 16 + r) * 64 + lane];
  }
  __syncthreads();
  if (wave < MT) {
    patch_put<FMT == FMT_I8>(sum, lds + wave * PATCH_WORDS, lane);
    patch_store_inline<FMT == FMT_I8, ACT, true>(lds + wave * PATCH_WORDS, C, ldc, (int64_t)wave * 32, n0, M, N, e,
                                                 lane, &pre);
  }
}

}  // namespace krn

using namespace krn;

template <int FMT, int BM, int BN, int WM, int WN>
static int launch_gemm(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                       int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  const int64_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  if (tiles == 0) return 0;
  if (tiles > 0x7fffffff) {
    krn_set_error("gemm: %lld tiles exceed the grid limit", (long long)tiles);
    return -1;
  }
  const bool vec = kbytes % 16 == 0 && lda % 16 == 0 && ldb % 16 == 0 && (uintptr_t)a % 16 == 0 &&
                   (uintptr_t)b % 16 == 0;
  dim3 grid((unsigned)tiles), block(256);
  if (vec) {
    hipLaunchKernelGGL((gemm_tile<FMT, BM, BN, WM, WN, true>), grid, block, 0, stream, (const uint8_t*)a,
                       (const uint8_t*)b, c, m, n, kbytes, lda, ldb, ldc, e);
  } else {
    hipLaunchKernelGGL((gemm_tile<FMT, BM, BN, WM, WN, false>), grid, block, 0, stream, (const uint8_t*)a,
                       (const uint8_t*)b, c, m, n, kbytes, lda, ldb, ldc, e);
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("gemm launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

template <int FMT, int BM, int BN, int WM, int WN, int STAGES, int BKB>
static int launch_pipe(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                       int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  const int64_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  if (tiles > 0x7fffffff) {
    krn_set_error("gemm: %lld tiles exceed the grid limit", (long long)tiles);
    return -1;
  }
  hipLaunchKernelGGL((gemm_pipe<FMT, BM, BN, WM, WN, STAGES, BKB>), dim3((unsigned)tiles), dim3(WM * WN * 64), 0, stream,
                     (const uint8_t*)a, (const uint8_t*)b, c, m, n, kbytes, lda, ldb, ldc, e);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("gemm launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

template <int FMT>
static int launch_quad16(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                         int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  const int64_t tiles = ((m + 255) / 256) * ((n + 255) / 256);
  if (tiles > 0x7fffffff) {
    krn_set_error("gemm: %lld tiles exceed the grid limit", (long long)tiles);
    return -1;
  }
  hipLaunchKernelGGL((gemm_quad16<FMT>), dim3((unsigned)tiles), dim3(256), 0, stream, (const uint8_t*)a,
                     (const uint8_t*)b, c, m, n, kbytes, lda, ldb, ldc, e);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("gemm launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

template <int FMT, int STAGES>
static int launch_pp(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                     int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  const int64_t tiles = ((m + 255) / 256) * ((n + 255) / 256);
  if (tiles > 0x7fffffff) {
    krn_set_error("gemm: %lld tiles exceed the grid limit", (long long)tiles);
    return -1;
  }
  hipLaunchKernelGGL((gemm_pp<FMT, STAGES>), dim3((unsigned)tiles), dim3(512), 0, stream, (const uint8_t*)a,
                     (const uint8_t*)b, c, m, n, kbytes, lda, ldb, ldc, e);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("gemm launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

template <int FMT, int MT, int STAGES>
static int launch_skinny_mt(const SplitCall& g, int parts) {
  int64_t ldc = g.n;
  Epilogue e = g.e;
  void* c = g.c;
  if (parts > 1) {
    ldc = split_ld(g.n);
    e = plane_epilogue(FMT);
    c = g.workspace;
  }
  // an epilogue without activations gets a kernel without their code (a quarter of the size, and no instruction
  // cache misses in the epilogue)
  bool act = false;
  for (int i = 0; i < e.nops; ++i) act |= (e.op[i] & ((1 << VEC_KIND_SHIFT) - 1)) >= RELU;
  const dim3 grid((unsigned)((g.n + 31) / 32), (unsigned)parts), block(4 * 64);
  // one row block: only the eight-row groups of A that hold rows < M are loaded
#define KRN_SKINNY(AL)                                                                                           \
  do {                                                                                                           \
    if (act)                                                                                                     \
      hipLaunchKernelGGL((gemm_skinny<FMT, MT, 4, STAGES, true, AL>), grid, block, 0, g.stream,                  \
                         (const uint8_t*)g.a, (const uint8_t*)g.b, c, g.m, g.n, g.kbytes, g.lda, g.ldb, ldc, e, parts); \
    else                                                                                                         \
      hipLaunchKernelGGL((gemm_skinny<FMT, MT, 4, STAGES, false, AL>), grid, block, 0, g.stream,                 \
                         (const uint8_t*)g.a, (const uint8_t*)g.b, c, g.m, g.n, g.kbytes, g.lda, g.ldb, ldc, e, parts); \
  } while (0)
  if constexpr (MT == 1) {
    if (g.m <= 8) KRN_SKINNY(1);
    else if (g.m <= 16) KRN_SKINNY(2);
    else if (g.m <= 24) KRN_SKINNY(3);
    else KRN_SKINNY(4);
  } else {
    KRN_SKINNY(MT * 4);
  }
#undef KRN_SKINNY
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("gemm launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return parts > 1 ? launch_reduce(FMT, parts, g) : 0;
}

// M <= 128 rows with 16-byte aligned rows of a multiple of 128 bytes: one workgroup per 32 output columns, four
// waves (one per SIMD, all issuing MFMAs: fewer leave bf16 compute-bound at 128 rows). One row block and at most one
// workgroup per CU (N <= 8192): a four-stage ring per wave (128 KiB; fp8 M = 1 11.5 -> 11.2 us against two stages);
// more workgroups than CUs: two stages (64 KiB), so that two workgroups share a CU and one's reduction and epilogue
// overlap the other's stream (W8A8 M = 16, N = 14336: 15.4 us, against 18.7 us with four stages); more row blocks:
// two stages, 96 to 160 KiB.
template <int FMT>
static int launch_skinny(const SplitCall& g, int parts) {
  switch ((g.m + 31) / 32) {
    case 1:
      return (g.n + 31) / 32 * parts <= 256 ? launch_skinny_mt<FMT, 1, 4>(g, parts)
                                            : launch_skinny_mt<FMT, 1, 2>(g, parts);
    case 2: return launch_skinny_mt<FMT, 2, 2>(g, parts);
    case 3: return launch_skinny_mt<FMT, 3, 2>(g, parts);
    case 4: return launch_skinny_mt<FMT, 4, 2>(g, parts);
  }
  krn_set_error("gemm: %lld rows are too many for the skinny kernel", (long long)g.m);
  return -1;
}

// 256 x 256 tiles (ragged at the edges).
template <int FMT>
static int launch_whole(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                        int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  // Two slices or more: the four-wave loop on 16x16 MFMAs (gemm_quad16). One slice (K = 128 bytes): fp8 the
  // eight-wave ping-pong, int8 and bf16/f16 the eight-wave direct-to-LDS ring.
  if (kbytes >= 256) return launch_quad16<FMT>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
  if constexpr (FMT == FMT_FP8)
    return launch_pp<FMT, 4>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
  else if constexpr (FMT == FMT_I8)
    return launch_pipe<FMT, 256, 256, 4, 2, 2, 128>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
  else
    return launch_pipe<FMT, 256, 256, 4, 2, 4, 64>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
}

// Up to one wave of 128 x 128 tiles (at most 256 tiles): the pipelined loop on 128 x 128 tiles with four waves, a
// 64 KiB ring (measured 20-40 % faster than the register-staged tiles at 1024^3 and 2048^3 for every format)
template <int FMT>
static int launch_mid(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                      int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  if constexpr (FMT == FMT_BF16 || FMT == FMT_F16)
    return launch_pipe<FMT, 128, 128, 2, 2, 4, 64>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
  else
    return launch_pipe<FMT, 128, 128, 2, 2, 2, 128>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
}

// 128 x 256 tiles, eight waves (64 x 64 each), for the products between one wave of 128 x 128 tiles and 128 tiles
// of 256 x 256 (bf16/f16 and int8; int8 with three 128-byte stages, 144 KiB: the W8A8 4096 x 14336 x 4096 column
// tail 49.9 -> 45.2 us against two)
template <int FMT>
static int launch_band(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t kbytes, int64_t lda,
                       int64_t ldb, int64_t ldc, const Epilogue& e, hipStream_t stream) {
  if constexpr (FMT == FMT_BF16 || FMT == FMT_F16)
    return launch_pipe<FMT, 128, 256, 2, 4, 4, 64>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
  else
    return launch_pipe<FMT, 128, 256, 2, 4, 3, 128>(a, b, c, m, n, kbytes, lda, ldb, ldc, e, stream);
}

// How a product runs: the kernel family, for RING and ANY the tile and loader, the K parts, and the workspace bytes.
enum Route : int { SKINNY, WHOLE, MID, BAND, TILE, SPLIT, NN_WHOLE, NN_TRANSPOSED };
struct Plan {
  Route route;
  int shape, parts;
  int64_t workspace;
};

// The NN products gemm_quad16 takes with B read K-major from LDS (no transposed copy): at least 128 tiles
// of 256 x 256, N a multiple of 256, K of 64 (whole 128-byte slices, at least two), 16-byte aligned operands, and
// panels addressable by 31-bit buffer offsets.
static bool nn_direct(const void* a, const void* b, int64_t m, int64_t n, int64_t k) {
  const int64_t t256 = ((m + 255) / 256) * (n / 256);
  return m > 0 && n > 0 && n % 256 == 0 && k % 64 == 0 && k >= 128 && t256 >= 128 && t256 <= 0x7fffffff &&
         (uintptr_t)a % 16 == 0 &&
         (uintptr_t)b % 16 == 0 && 256 * k * 2 <= 0x7fffffff && (k - 1) * n * 2 + 512 <= 0x7fffffff;
}

// The products of nn_direct
static int launch_nn_whole(bool bf, const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
                           const Epilogue& e, hipStream_t stream) {
  const dim3 tiles((unsigned)(((m + 255) / 256) * (n / 256)));
  if (bf)
    hipLaunchKernelGGL((gemm_quad16<FMT_BF16, true>), tiles, dim3(256), 0, stream, (const uint8_t*)a, (const uint8_t*)b, c,
                       m, n, k * 2, k * 2, n * 2, n, e);
  else
    hipLaunchKernelGGL((gemm_quad16<FMT_F16, true>), tiles, dim3(256), 0, stream, (const uint8_t*)a, (const uint8_t*)b, c,
                       m, n, k * 2, k * 2, n * 2, n, e);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("gemm_nn launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}

// Estimated microseconds of a split-kernel launch beyond its fixed cost, from sweeps of each tile over 10 to 1500
// workgroups (bf16 unless noted): a 128-byte K slice takes a CU `slice` us, with `more` us for every workgroup the
// busiest CU holds once that is larger. 256 x 4096 x 4096 on 64 x 64 tiles 16.5 us (one workgroup per CU), 512 rows
// 27.5 us (two); 128 x 128 tiles, operands from HBM: two workgroups per CU 57.9 us at 256 x 4096 x 14336 in eight parts,
// one with four stages 52.9 in four; 512 x 8192 x 8192 four stages 82-83, two stages 110; unaligned 1024 x 4096 x 4097
// 60 us on 128 x 128.
static const struct { int bm, bn; double slice, more, more_nn; } SPLIT_TILES[] = {
    {32, 64, 0.23, 0.15, 0.17},   {64, 64, 0.28, 0.22, 0.25},   {128, 128, 0.80, 0.60, 0.52}, {128, 128, 0.62, 0.62, 0.82},
    {32, 128, 0.70, 0.75, 0.75},  {64, 64, 0.43, 0.35, 0.38},   {128, 128, 0.92, 0.92, 0.95}};
static int64_t split_tiles(int shape, int64_t m, int64_t n) {
  const auto& t = SPLIT_TILES[shape];
  return ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
}
static double split_cost(int shape, bool nn, int64_t m, int64_t n, int64_t slices, int parts) {
  const auto& t = SPLIT_TILES[shape];
  const int64_t wgs = split_tiles(shape, m, n) * parts;
  const double per_cu = (double)((wgs + 255) / 256);
  double us = (double)((slices + parts - 1) / parts) * fmax(t.slice, (nn ? t.more_nn : t.more) * per_cu);
  if (parts > 1) us += 8.0 + (double)parts * (double)split_plane(m, n) / 5e6;  // the second launch reads the planes
  return us;
}

// Whether the four-wave loop (MID) is the faster of the two 128 x 128 loops that run one tile per CU, the other being the
// ring's four stages (RING_128x128_DEEP, one part). The ring reads whole lines and takes the same time per slice whatever
// K is, but costs 2 us more where MID stores whole blocks straight from its accumulators; MID's blocks that a ragged N
// cuts go out element by element. Measured on 129 to 256 tiles, MID against the ring, us:
//   16-bit, up to 32 slices: 2048 x 2048 x 512 8.5 / 10.8, x 2048 21.2 / 23.3, 1500 x 2000 x 1024 14.0 / 15.7; from 33 on
//   x 3072 32.9 / 31.3, except on rows of 8 and 16 KiB whose operands the last-level cache holds (2048 x 2048 x 4096
//   38.5 / 40.4, x 8192 70.6 / 72.5; from HBM 512 x 8192 x 8192 93.4 / 79.1). N not a multiple of 16: 400 x 7000 x 512
//   12.4 / 11.0.
//   int8, up to 18 slices: 2048 x 2048 x 1024 15.3 / 17.3, x 2304 22.9 / 23.4, x 2560 25.6 / 24.9; 1500 x 2000 20.5 / 17.1.
//   fp8, up to 8 slices: 2048 x 2048 x 1024 11.6 / 11.9, x 1280 13.5 / 12.9; ragged M, 1181 x 1792 x 512 9.0 / 9.1, x 640
//   10.1 / 9.6; 1500 x 2000 x 512 11.2 / 10.1.
static bool four_wave_wins(int fmt, int64_t m, int64_t n, int64_t slices) {
  if (fmt == FMT_I8) return n % 64 == 0 && slices <= 18;
  if (fmt == FMT_FP8) return n % 64 == 0 && slices <= (m % 64 == 0 ? 8 : 4);
  if (n % 16 != 0) return false;
  return slices <= 32 || ((slices == 64 || slices == 128) && (m + n) * slices * 128 <= (int64_t)80 << 20);
}

// Workgroups of a launch: of 256 threads, and a launch's threads along an axis stay below 2^32 (a launch past that runs
// nothing: 2^30 rows of 64 x 64 tiles left C unwritten)
constexpr int64_t MOST_TILES = ((int64_t)1 << 24) - 1;

// Kernel choice on 256 CUs. Products that fill the chip with 256 x 256 tiles (at least 128 of them, ragged edges
// included, K in whole 128-byte slices, 16-byte aligned rows) and those with at most 128 rows keep their kernels; what
// is left is a choice between tiles by estimated time: the eight- and four-wave loops on 128 x 256 and 128 x 128
// tiles (NT, whole slices), and the split kernels on smaller tiles, over K, or with unaligned rows. `workspace` bounds
// the planes of K parts. `in_place`: C shares memory with A or B. The parts then write to planes whatever the shape, and C
// is written once all of them have read; without a workspace for two planes, no tile is smaller than 128 x 128 (a
// product of one such tile column reads its rows before it writes them).
static Plan plan_of(int fmt, bool nn, const void* a, const void* b, int64_t m, int64_t n, int64_t k, int64_t elem,
                    int64_t workspace, bool in_place = false) {
  const int64_t kbytes = k * elem, slices = (kbytes + 127) / 128;
  const bool aligned = kbytes % 16 == 0 && (uintptr_t)a % 16 == 0 && (uintptr_t)b % 16 == 0 && (!nn || n % 8 == 0);
  const int64_t t256 = ((m + 255) / 256) * ((n + 255) / 256), t128 = ((m + 127) / 128) * ((n + 127) / 128);
  const bool piped = !nn && aligned && kbytes % 128 == 0 && kbytes > 0 && m > 0 && n > 0;
  // the split kernels' 128-row panels (NN: all of B) are addressed by 31-bit offsets, rows hold a whole 16-byte load
  const bool split = kbytes >= 16 && m > 0 && n > 0 && 128 * kbytes <= 0x7fffffff &&
                     (!nn || (n >= 8 && kbytes / 2 * n * 2 <= 0x7fffffff));
  if (in_place && split && 2 * split_plane(m, n) <= workspace)
    return {SPLIT, aligned ? RING_128x128 : ANY_128x128, 2, 2 * split_plane(m, n)};
  if (nn && nn_direct(a, b, m, n, k)) return {NN_WHOLE, 0, 1, 0};
  if (piped && t256 >= 128 && m > 128 && 256 * kbytes <= 0x7fffffff) return {WHOLE, 0, 1, 0};
  Plan best{TILE, 0, 1, 0};
  double least = 1e30;
  if (piped && m <= 128) {
    // One workgroup per 32 columns; with few columns K is split as well. A slice takes a workgroup RATE, with one block
    // of 32 rows to four, beyond the launch's fixed cost (1 x 4096 x 4096 bf16, 64 slices: 9.2 us on 128 workgroups;
    // 16 x 1024 x 14336, 224 slices: 28.2 on 32, split 11.4); the second launch of a split costs 8, most of it on the
    // host (3 x 768 x 4992 f16: 7.8 us, split 11.6). Parts of whole 16 KiB start on the same memory channels, which costs
    // 6 us or more once B is too large for the last-level cache to help: 4096 x 16384 in 16 bits, whole and in two parts,
    // 1 row 30.1 and 35.5 us, 8 rows 32.7 and 36.0; 16 rows, where a slice takes longer, 36.3 and 34.3, 32 rows 43.9 and
    // 34.3. Not so at 96 MiB (3072 x 16384, 1 row: 26.2 and 23.6) and for other parts (4096 x 28672: 46.4 and 38.6).
    static const double RATE[] = {0.12, 0.14, 0.24, 0.35};
    const int64_t groups = (n + 31) / 32;
    const double rate = m <= 12 ? 0.10 : RATE[(m - 1) / 32];
    const double whole_k = (double)slices * rate * (double)((groups + 255) / 256);
    best = {SKINNY, 0, 1, 0}, least = whole_k;
    for (int parts = 2; parts <= 16 && groups * parts <= 256 && slices / parts >= 8; ++parts) {
      const int64_t need = parts * split_plane(m, n);
      const bool same_channels = slices % (parts * 128) == 0 && n * kbytes >= (int64_t)112 << 20;
      const double us = whole_k / parts + (same_channels ? 14.0 : 8.0) + (double)need / 5e6;
      if (need <= workspace && us < least) best = {SKINNY, 0, parts, need}, least = us;
    }
    // 65 to 128 rows of 16-bit operands: four row blocks per wave make the skinny loop slower than 128 x 128 tiles
    // with K split (128 x 8192 x 8192 bf16 48.5 -> 41 us; fp8 the other way, 19 against 30 us)
    if (m <= 64 || elem == 1) return best;
    least -= 2.0;  // near ties stay (89 x 1536 x 2560 f16: 11.0 us, 32 x 64 tiles 11.7)
  } else if (piped && 128 * kbytes <= 0x7fffffff) {
    // the four-wave loop: 0.66 us a slice from the caches, 0.74 from HBM (95 us at 512 x 8192 x 8192)
    if (t128 <= 256) best = {MID, 0, 1, 0}, least = 0.66 * (double)slices;
    else if (fmt != FMT_FP8 && 256 * kbytes <= 0x7fffffff)
      best = {BAND, 0, 1, 0},
      least = 0.95 * (double)slices * (double)((((m + 127) / 128) * ((n + 255) / 256) + 255) / 256);
  } else if (nn && aligned && kbytes % 128 == 0 && t256 >= 128 && n * k * 2 <= workspace) {
    // a transposed copy of B, then the whole-tile loop
    best = {NN_TRANSPOSED, 0, 1, n * k * 2};
    least = 6.0 + (double)(n * k * 4) / 4.5e6 + 1.41 * (double)slices * (double)((t256 + 255) / 256);
  }
  if (!split) return nn && n * k * 2 <= workspace ? Plan{NN_TRANSPOSED, 0, 1, n * k * 2} : best;
  for (int shape = aligned ? RING_32x64 : ANY_32x128; shape <= (aligned ? RING_128x128_DEEP : ANY_128x128); ++shape)
    for (int parts = 1; parts <= 16 && (parts == 1 || slices / parts >= 8); ++parts) {
      const int64_t need = parts > 1 ? parts * split_plane(m, n) : 0;
      if (need > workspace || split_tiles(shape, m, n) > MOST_TILES) break;
      if (shape == RING_128x128_DEEP && parts == 1 && best.route == MID && four_wave_wins(fmt, m, n, slices)) continue;
      if (in_place && shape != RING_128x128 && shape != RING_128x128_DEEP && shape != ANY_128x128) break;
      const double us = split_cost(shape, nn, m, n, slices, parts);
      if (us < least) best = {SPLIT, shape, parts, need}, least = us;
    }
  return best;
}

template <int FMT>
static int launch_planned(const Plan& p, bool nn, const SplitCall& g) {
  switch (p.route) {
    case SKINNY: return launch_skinny<FMT>(g, p.parts);
    case SPLIT: return launch_split(FMT, nn, p.shape, p.parts, g);
    case MID: return launch_mid<FMT>(g.a, g.b, g.c, g.m, g.n, g.kbytes, g.lda, g.ldb, g.n, g.e, g.stream);
    case BAND:  // never fp8
      if constexpr (FMT != FMT_FP8)
        return launch_band<FMT>(g.a, g.b, g.c, g.m, g.n, g.kbytes, g.lda, g.ldb, g.n, g.e, g.stream);
      break;
    case WHOLE: break;
    default:
      return launch_gemm<FMT, 128, 128, 2, 2>(g.a, g.b, g.c, g.m, g.n, g.kbytes, g.lda, g.ldb, g.n, g.e, g.stream);
  }
  // A last wave of 256 x 256 tiles at most half full (W8A8 4096 x 14336: 896 tiles, 3.5 waves on 256 CUs) would
  // leave half the chip idle for a whole tile time. When the full waves cover whole columns of tiles, those
  // columns run as 256 x 256 tiles and the remaining columns as a second launch of 128 x 256 tiles (twice as many,
  // half the work each), which fills the last wave. The two launches write disjoint columns of C.
  const int64_t t256 = ((g.m + 255) / 256) * ((g.n + 255) / 256);
  const int64_t full_tiles = (t256 / 256) * 256, tile_rows = (g.m + 255) / 256;
  if constexpr (FMT != FMT_FP8) {
    if (t256 % 256 != 0 && t256 % 256 <= 128 && full_tiles > 0 && full_tiles % tile_rows == 0) {
      const int64_t n_split = full_tiles / tile_rows * 256;
      Epilogue tail = g.e;  // the epilogue of the columns from n_split on: column vectors start at that column
      for (int i = 0; i < g.e.nops; ++i) {
        const int op = g.e.op[i] & ((1 << VEC_KIND_SHIFT) - 1), kind = g.e.op[i] >> VEC_KIND_SHIFT;
        if (op == MUL_COL || op == ADD_COL)
          tail.vec[i] = static_cast<const uint8_t*>(g.e.vec[i]) + n_split * (kind == 0 ? 4 : 2);
      }
      const int out_bytes = (g.e.out_kind == F32 || g.e.out_kind == I32) ? 4 : 2;
      const int rc = launch_whole<FMT>(g.a, g.b, g.c, g.m, n_split, g.kbytes, g.lda, g.ldb, g.n, g.e, g.stream);
      if (rc != 0) return rc;
      return launch_band<FMT>(g.a, static_cast<const uint8_t*>(g.b) + n_split * g.ldb,
                              static_cast<uint8_t*>(g.c) + n_split * out_bytes, g.m, g.n - n_split, g.kbytes, g.lda,
                              g.ldb, g.n, tail, g.stream);
    }
  }
  return launch_whole<FMT>(g.a, g.b, g.c, g.m, g.n, g.kbytes, g.lda, g.ldb, g.n, g.e, g.stream);
}

extern "C" int krn_transpose16(const void* in, void* out, int64_t rows, int64_t cols, void* stream);

static int gemm_dispatch(int fmt, bool nn, const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
                         int64_t elem, const Epilogue& e, void* workspace, int64_t workspace_bytes,
                         hipStream_t stream) {
  if (m == 0 || n == 0) return 0;
  const int64_t c_bytes = m * n * (e.out_kind == F32 || e.out_kind == I32 ? 4 : 2);
  const bool in_place = share_memory(c, c_bytes, a, m * k * elem) || share_memory(c, c_bytes, b, n * k * elem);
  // more rows than a launch of 128-row tiles holds (M of 2^31 and more): in runs of 2^30
  constexpr int64_t RUN = (int64_t)1 << 30;
  if (!in_place && m > RUN && (m + 127) / 128 * ((n + 127) / 128) > MOST_TILES) {
    for (int64_t r0 = 0; r0 < m; r0 += RUN) {
      Epilogue run = e;  // row vectors start at the run's first row
      for (int i = 0; i < e.nops; ++i) {
        const int op = e.op[i] & ((1 << VEC_KIND_SHIFT) - 1), kind = e.op[i] >> VEC_KIND_SHIFT;
        if (op == MUL_ROW || op == ADD_ROW) run.vec[i] = static_cast<const uint8_t*>(e.vec[i]) + r0 * (kind == 0 ? 4 : 2);
      }
      const int rc = gemm_dispatch(fmt, nn, static_cast<const uint8_t*>(a) + r0 * k * elem, b,
                                   static_cast<uint8_t*>(c) + c_bytes / m * r0, m - r0 < RUN ? m - r0 : RUN, n, k, elem,
                                   run, workspace, workspace_bytes, stream);
      if (rc != 0) return rc;
    }
    return 0;
  }
  const Plan p = plan_of(fmt, nn, a, b, m, n, k, elem, workspace ? workspace_bytes : 0, in_place);
  const SplitCall g{a, b, c, m, n, k * elem, k * elem, nn ? n * 2 : k * elem, e, workspace, stream};
  if (p.route == NN_WHOLE) return launch_nn_whole(fmt == FMT_BF16, a, b, c, m, n, k, e, stream);
  if (nn && p.route != SPLIT) {
    if (n * k * 2 > (workspace ? workspace_bytes : 0) && k > 0) {
      krn_set_error("gemm: this product needs a workspace of %lld bytes for the transposed operand",
                    (long long)(n * k * 2));
      return -1;
    }
    if (k > 0) {
      const int rc = krn_transpose16(b, workspace, k, n, stream);
      if (rc) return rc;
    }
    return gemm_dispatch(fmt, false, a, workspace, c, m, n, k, elem, e, nullptr, 0, stream);
  }
  switch (fmt) {
    case FMT_BF16: return launch_planned<FMT_BF16>(p, nn, g);
    case FMT_F16: return launch_planned<FMT_F16>(p, nn, g);
    case FMT_I8: return launch_planned<FMT_I8>(p, nn, g);
    case FMT_FP8: return launch_planned<FMT_FP8>(p, nn, g);
  }
  krn_set_error("gemm: unknown operand format %d", fmt);
  return -1;
}

// The epilogue chain of a launch, checked: at most four known operations, a vector for every per-row or per-column
// one. `who` prefixes the error message.
static bool epilogue_of(Epilogue& e, int out_kind, int nops, const int* ops, const float* scalars,
                        const void* const* vectors, const char* who) {
  e.out_kind = out_kind;
  if (nops < 0 || nops > 4) {
    krn_set_error("%s: %d epilogue operations, at most 4", who, nops);
    return false;
  }
  e.nops = nops;
  for (int i = 0; i < nops; ++i) {
    e.op[i] = ops[i];
    e.scalar[i] = scalars ? scalars[i] : 0.0f;
    e.vec[i] = vectors ? vectors[i] : nullptr;
    const int op = ops[i] & ((1 << VEC_KIND_SHIFT) - 1), kind = ops[i] >> VEC_KIND_SHIFT;
    if (ops[i] < 0 || op > SILU || kind > 2 || (kind != 0 && (op >= RELU || op % 3 == 0))) {
      krn_set_error("%s: unknown epilogue operation %d", who, ops[i]);
      return false;
    }
    if (op < RELU && op % 3 != 0 && e.vec[i] == nullptr) {
      krn_set_error("%s: epilogue operation %d needs a vector", who, i);
      return false;
    }
  }
  return true;
}

// The arguments of an entry point, checked; the format and element size of the operands.
static bool gemm_arguments(Epilogue& e, int& fmt, int64_t& elem, int in_kind, int out_kind, int64_t m, int64_t n,
                           int64_t k, int nops, const int* ops, const float* scalars, const void* const* vectors) {
  if (!epilogue_of(e, out_kind, nops, ops, scalars, vectors, "gemm")) return false;
  if (m < 0 || n < 0 || k < 0) {
    krn_set_error("gemm: negative extent");
    return false;
  }
  switch (in_kind) {
    case BF16: fmt = FMT_BF16; elem = 2; break;
    case F16: fmt = FMT_F16; elem = 2; break;
    case I8: fmt = FMT_I8; elem = 1; break;
    case F8E4M3: fmt = FMT_FP8; elem = 1; break;
    default: krn_set_error("gemm: operand kind %d has no matrix unit product", in_kind); return false;
  }
  if (out_kind == I32 && (fmt != FMT_I8 || nops != 0)) {
    krn_set_error("gemm: an int32 result needs int8 operands and no epilogue operations");
    return false;
  }
  if (out_kind != F32 && out_kind != F16 && out_kind != BF16 && out_kind != I32) {
    krn_set_error("gemm: output kind %d is not stored by the tile GEMM", out_kind);
    return false;
  }
  return true;
}

extern "C" {

int krn_gemm(int b_kn, int in_kind, const void* a, const void* b, void* c, int out_kind, int64_t m, int64_t n,
             int64_t k, int nops, const int* ops, const float* scalars, const void* const* vectors, void* workspace,
             int64_t workspace_bytes, void* stream);

// See include/krn_amd.h for the contract of each entry point.
int krn_gemm_nt(int in_kind, const void* a, const void* b, void* c, int out_kind, int64_t m, int64_t n, int64_t k,
                int nops, const int* ops, const float* scalars, const void* const* vectors, void* stream) {
  return krn_gemm(0, in_kind, a, b, c, out_kind, m, n, k, nops, ops, scalars, vectors, nullptr, 0, stream);
}

int krn_gemm(int b_kn, int in_kind, const void* a, const void* b, void* c, int out_kind, int64_t m, int64_t n,
             int64_t k, int nops, const int* ops, const float* scalars, const void* const* vectors, void* workspace,
             int64_t workspace_bytes, void* stream) {
  Epilogue e{};
  int fmt;
  int64_t elem;
  if (!gemm_arguments(e, fmt, elem, in_kind, out_kind, m, n, k, nops, ops, scalars, vectors)) return -1;
  if (b_kn && elem != 2) {
    krn_set_error("gemm: operand kind %d; the NN product takes bf16 or f16 operands", in_kind);
    return -1;
  }
  return gemm_dispatch(fmt, b_kn != 0, a, b, c, m, n, k, elem, e, workspace, workspace_bytes, (hipStream_t)stream);
}

int64_t krn_gemm_workspace(int b_kn, int in_kind, const void* a, const void* b, int64_t m, int64_t n, int64_t k) {
  const int fmt = in_kind == BF16 ? FMT_BF16 : in_kind == F16 ? FMT_F16 : in_kind == I8 ? FMT_I8 : FMT_FP8;
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  return plan_of(fmt, b_kn != 0, a, b, m, n, k, fmt == FMT_BF16 || fmt == FMT_F16 ? 2 : 1, INT64_MAX).workspace;
}

int64_t krn_gemm_workspace_in_place(int64_t m, int64_t n) { return m <= 0 || n <= 0 ? 0 : 2 * split_plane(m, n); }

}  // extern "C"

// out[c, r] = in[r, c] for 16-bit elements, through a 64x65-word LDS tile: the B operand of a `b[ks, cols]`
// product is turned K-contiguous before the NT main loop reads it.
__global__ __launch_bounds__(256) void transpose16(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                   int64_t rows, int64_t cols) {
  __shared__ uint16_t tile[64][65];
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    const int64_t r = r0 + i, c = c0 + tx;
    tile[i][tx] = (r < rows && c < cols) ? in[r * cols + c] : 0;
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    const int64_t c = c0 + i, r = r0 + tx;
    if (c < cols && r < rows) out[c * rows + r] = tile[tx][i];
  }
}

// The NN product `a[rows, ks] @ b[ks, cols]` with B stored K x N: read as it lies where gemm_quad16 takes it, otherwise
// transposed into `bt` (N x K, n * k 16-bit elements) for the NT kernels. Both launches go on `stream`, in that order.
static int gemm_nn_through(int in_kind, const void* a, const void* b, void* c, int out_kind, int64_t m, int64_t n,
                           int64_t k, int nops, const int* ops, const float* scalars, const void* const* vectors,
                           void* bt, void* stream) {
  if (in_kind != BF16 && in_kind != F16) {
    krn_set_error("gemm_nn: operand kind %d; the NN product takes bf16 or f16 operands", in_kind);
    return -1;
  }
  if (m < 0 || n < 0 || k < 0) {
    krn_set_error("gemm_nn: negative extent");
    return -1;
  }
  if (nn_direct(a, b, m, n, k)) {
    Epilogue e{};
    if (!epilogue_of(e, out_kind, nops, ops, scalars, vectors, "gemm_nn")) return -1;
    if (out_kind != F32 && out_kind != F16 && out_kind != BF16) {
      krn_set_error("gemm_nn: output kind %d is not stored by the tile GEMM", out_kind);
      return -1;
    }
    return launch_nn_whole(in_kind == BF16, a, b, c, m, n, k, e, (hipStream_t)stream);
  }
  if (bt == nullptr && n > 0 && k > 0) {
    krn_set_error("gemm_nn: this product needs the transposed operand's workspace");
    return -1;
  }
  if (n > 0 && k > 0) {
    const int rc = krn_transpose16(b, bt, k, n, stream);
    if (rc) return rc;
  }
  return krn_gemm_nt(in_kind, a, bt, c, out_kind, m, n, k, nops, ops, scalars, vectors, stream);
}

extern "C" int64_t krn_gemm_nn_workspace(int64_t n, int64_t k) { return n < 0 || k < 0 ? 0 : n * k * 2; }

extern "C" int64_t krn_gemm_nn_workspace_for(const void* a, const void* b, int64_t m, int64_t n, int64_t k) {
  return nn_direct(a, b, m, n, k) ? 0 : krn_gemm_nn_workspace(n, k);
}

extern "C" int krn_gemm_nn(int in_kind, const void* a, const void* b, void* c, int out_kind, int64_t m, int64_t n,
                           int64_t k, int nops, const int* ops, const float* scalars, const void* const* vectors,
                           void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = nn_direct(a, b, m, n, k) ? 0 : krn_gemm_nn_workspace(n, k);
  if (need > 0 && (workspace == nullptr || workspace_bytes < need)) {
    krn_set_error("gemm_nn: the workspace holds %lld bytes, the transposed operand needs %lld",
                  (long long)workspace_bytes, (long long)need);
    return -1;
  }
  return gemm_nn_through(in_kind, a, b, c, out_kind, m, n, k, nops, ops, scalars, vectors, workspace, stream);
}

// The scratch of krn_gemm_nn_noalloc: the transposed B operand lives in this file-scope device array instead of a
// caller's workspace or an allocation. Every GPU the library runs on holds its own copy until the process ends. In
// host code `scratch` names a host-side stand-in, not the device memory: the device address comes from
// hipGetSymbolAddress, once per device, and only that address is handed to kernels.
constexpr int64_t KRN_NN_SCRATCH_BYTES = (int64_t)64 << 20;
static __device__ __align__(256) uint8_t scratch[KRN_NN_SCRATCH_BYTES];
constexpr int KRN_MAX_DEVICES = 64;

// Per device: the array's address, and an event recorded after the last eager call that used it. Every call first
// makes its stream wait (hipStreamWaitEvent, on the device) for that event, so two streams never hold the array at
// once (on the previous call's own stream the wait is already satisfied by stream order; it is kept unconditional so
// a stream handle reused after a destroy cannot skip it). The lock covers the look-up, that wait, the enqueue and the new record, so
// host threads are ordered too. A stream under graph capture neither waits nor records (an event of the eager world
// cannot order graph replays): a captured call is ordered only by the graph's and the caller's own dependencies.
struct ScratchUse {
  void* ptr = nullptr;
  hipEvent_t done = nullptr;  // recorded after the last eager call that used the array
  bool used = false;
};
static std::mutex scratch_lock;
static ScratchUse scratch_use[KRN_MAX_DEVICES];

// The device the call runs on: the stream's own device, which must be the current one (the address comes from
// the current device's array). The null stream runs on the current device.
static int scratch_device(hipStream_t stream) {
  int device = -1;
  hipError_t rc = hipGetDevice(&device);
  if (rc != hipSuccess || device < 0 || device >= KRN_MAX_DEVICES) {
    krn_set_error("gemm_nn_noalloc: no usable current device (%s, ordinal %d)", hipGetErrorString(rc), device);
    return -1;
  }
  if (stream != nullptr) {
    int of_stream = -1;
    rc = hipStreamGetDevice(stream, &of_stream);
    if (rc != hipSuccess) {
      krn_set_error("gemm_nn_noalloc: hipStreamGetDevice failed: %s", hipGetErrorString(rc));
      return -1;
    }
    if (of_stream != device) {
      krn_set_error("gemm_nn_noalloc: the stream belongs to device %d but device %d is current; make the stream's "
                    "device current", of_stream, device);
      return -1;
    }
  }
  return device;
}

// Set-up of one device, on its first call, with the lock held: the array's address and the ordering event.
static bool scratch_setup(int device) {
  ScratchUse& use = scratch_use[device];
  if (use.ptr != nullptr) return true;
  void* ptr = nullptr;
  hipError_t rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (rc != hipSuccess || ptr == nullptr) {
    krn_set_error("gemm_nn_noalloc: hipGetSymbolAddress of the scratch array failed: %s", hipGetErrorString(rc));
    return false;
  }
  rc = hipEventCreateWithFlags(&use.done, hipEventDisableTiming);
  if (rc != hipSuccess) {
    krn_set_error("gemm_nn_noalloc: hipEventCreateWithFlags failed: %s", hipGetErrorString(rc));
    return false;
  }
  use.ptr = ptr;
  return true;
}

extern "C" int64_t krn_gemm_nn_noalloc_limit(void) { return KRN_NN_SCRATCH_BYTES; }

extern "C" int krn_gemm_nn_noalloc(int in_kind, const void* a, const void* b, void* c, int out_kind, int64_t m,
                                   int64_t n, int64_t k, int nops, const int* ops, const float* scalars,
                                   const void* const* vectors, void* stream) {
  const int64_t need = nn_direct(a, b, m, n, k) ? 0 : krn_gemm_nn_workspace(n, k);
  if (need > KRN_NN_SCRATCH_BYTES) {
    krn_set_error("gemm_nn_noalloc: B of %lld x %lld needs %lld bytes of scratch; the library holds %lld "
                  "(use krn_gemm_nn with a workspace)", (long long)k, (long long)n, (long long)need,
                  (long long)KRN_NN_SCRATCH_BYTES);
    return -1;
  }
  if (need == 0) return gemm_nn_through(in_kind, a, b, c, out_kind, m, n, k, nops, ops, scalars, vectors, nullptr,
                                        stream);
  hipStream_t s = (hipStream_t)stream;
  const int device = scratch_device(s);
  if (device < 0) return -1;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  hipError_t rc = hipStreamIsCapturing(s, &capture);
  if (rc != hipSuccess) {
    krn_set_error("gemm_nn_noalloc: hipStreamIsCapturing failed: %s", hipGetErrorString(rc));
    return -1;
  }
  const bool eager = capture == hipStreamCaptureStatusNone;
  std::lock_guard<std::mutex> hold(scratch_lock);
  if (!scratch_setup(device)) return -1;
  ScratchUse& use = scratch_use[device];
  if (eager && use.used && (rc = hipStreamWaitEvent(s, use.done, 0)) != hipSuccess) {
    krn_set_error("gemm_nn_noalloc: hipStreamWaitEvent failed: %s", hipGetErrorString(rc));
    return -1;
  }
  const int status = gemm_nn_through(in_kind, a, b, c, out_kind, m, n, k, nops, ops, scalars, vectors, use.ptr, s);
  if (status != 0 || !eager) return status;
  if ((rc = hipEventRecord(use.done, s)) != hipSuccess) {
    krn_set_error("gemm_nn_noalloc: hipEventRecord failed: %s", hipGetErrorString(rc));
    return -1;
  }
  use.used = true;
  return 0;
}

// Whole 128 x 128 tiles (rows and cols multiples of 128, 16-byte aligned): rows land in LDS with 16-byte loads (256
// contiguous bytes per 16 lanes); each thread then reads one 8 x 8 block with eight 16-byte LDS reads, transposes it
// in registers (v_perm_b32 pairs the 16-bit halves of two rows) and writes eight 16-byte pieces of output rows, 256
// contiguous bytes per 16 lanes (8192^2: 70 -> 56 us).
__global__ __launch_bounds__(256) void transpose16_tiles(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                         int64_t rows, int64_t cols) {
  constexpr int P = 128 + 8;  // LDS row pitch in elements: 16 bytes of padding keep the block reads off one bank
  __shared__ __attribute__((aligned(16))) uint16_t tile[128 * P];
  const int t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * 128, c0 = (int64_t)blockIdx.x * 128;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int row = p * 16 + (t >> 4), cb = (t & 15) * 8;
    *reinterpret_cast<u32x4*>(tile + row * P + cb) =
        __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(in + (r0 + row) * cols + c0 + cb));
  }
  __syncthreads();
  const int bi = t & 15, bj = t >> 4;
  u32x4 r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = *reinterpret_cast<const u32x4*>(tile + (bi * 8 + i) * P + bj * 8);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;  // the high or the low halves of two words
    u32x4 o;
#pragma unroll
    for (int w = 0; w < 4; ++w) o[w] = __builtin_amdgcn_perm(r[2 * w + 1][j >> 1], r[2 * w][j >> 1], sel);
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(out + (c0 + bj * 8 + j) * rows + r0 + bi * 8));
  }
}

extern "C" int krn_transpose16(const void* in, void* out, int64_t rows, int64_t cols, void* stream) {
  if (rows < 0 || cols < 0) {
    krn_set_error("transpose: negative extent");
    return -1;
  }
  if (rows == 0 || cols == 0) return 0;
  if (rows % 128 == 0 && cols % 128 == 0 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0 &&
      cols / 128 <= 0x7fffffff && rows / 128 <= 65535) {
    hipLaunchKernelGGL(transpose16_tiles, dim3((unsigned)(cols / 128), (unsigned)(rows / 128)), dim3(256), 0,
                       (hipStream_t)stream, (const uint16_t*)in, (uint16_t*)out, rows, cols);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
      krn_set_error("transpose launch: %s", hipGetErrorString(err));
      return (int)err;
    }
    return 0;
  }
  const int64_t gx = (cols + 63) / 64, gy = (rows + 63) / 64;
  if (gx > 0x7fffffff || gy > 65535) {
    krn_set_error("transpose: %lld x %lld exceeds the grid limit", (long long)rows, (long long)cols);
    return -1;
  }
  hipLaunchKernelGGL(transpose16, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)in, (uint16_t*)out, rows, cols);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    krn_set_error("transpose launch: %s", hipGetErrorString(err));
    return (int)err;
  }
  return 0;
}
