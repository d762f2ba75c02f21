// Splitting K over workgroups: what the kernels of gemm_split.hip take, and their entry.
#pragma once
#include "gemm_parts.h"

namespace krn {

// K in `parts` runs of slices, one workgroup per tile and run. With more than one part each writes its sums, without
// an epilogue, to a plane of its own (M rows of split_ld(N) four-byte elements); a second kernel adds the planes.

// NN: where chunk c (8 columns) of k row k lies in its LDS row: the four k rows of a transposed read, 64 bytes each,
// on distinct banks
template <int BN>
__device__ __forceinline__ int kn_slot(int k, int c) {
  return BN == 128 ? c ^ ((k & 3) << 2) : c ^ (((k >> 1) & 1) << 2);
}

// Tile and loader: the ring of direct-to-LDS slices needs 16-byte aligned rows, the other takes any alignment. DEEP:
// four stages instead of two, for one workgroup per CU (NT: fragments read a slice ahead).
enum SplitShape : int {
  RING_32x64, RING_64x64, RING_128x128, RING_128x128_DEEP, ANY_32x128, ANY_64x64, ANY_128x128
};

struct SplitCall {
  const void *a, *b;
  void* c;
  int64_t m, n, kbytes, lda, ldb;
  Epilogue e;
  void* workspace;  // the parts' planes (more than one part)
  hipStream_t stream;
};

// the planes' row length in elements: whole 32-byte pieces, so that every row is aligned for 16-byte accesses; the
// kernels get it as ldc, and find plane p at p * M * ldc elements
inline int64_t split_ld(int64_t n) { return (n + 7) / 8 * 8; }
inline int64_t split_plane(int64_t m, int64_t n) { return m * split_ld(n) * 4; }

// what a part stores: its sums as they are
inline Epilogue plane_epilogue(int fmt) {
  Epilogue e{};
  e.out_kind = fmt == FMT_I8 ? I32 : F32;
  return e;
}

int launch_split(int fmt, bool nn, int shape, int parts, const SplitCall& g);
int launch_reduce(int fmt, int parts, const SplitCall& g);

}  // namespace krn
