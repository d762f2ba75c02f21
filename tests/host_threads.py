"""The generic lowering's kernels on the CPU: the emitted HIP source compiled for the host, every GPU thread a fiber
that runs until it meets a barrier or another lane, the lowest thread first or the highest first. A missing barrier that
the order of the threads can show is shown by one of the two; lanes of a wave get no order that the source does not ask
for. The shuffles and the 16 x 16 float products of the emitted code are lane exchanges here."""

import ctypes
import hashlib
import os
import subprocess

import numpy as np

from krn_amd.compiler import hipgen, ir
from krn_amd.compiler.space import geometry, runtime_args
from oracle.cbackend import CACHE, CLANG

SHIM = r"""
#include <math.h>
#include <string.h>
#include <ucontext.h>
#include <array>
#include <functional>
#include <map>
#include <vector>
#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(n)
struct Dim { unsigned x, y, z; };
static Dim threadIdx, blockIdx, gridDim;
struct Fiber {
  ucontext_t context;
  std::vector<char> stack;
  std::map<int, std::vector<std::array<char, 64>>> said;  // what this lane gave at each exchange of the source, in order
  bool done, waiting;
};
static std::vector<Fiber> fibers;
static ucontext_t scheduler;
static unsigned current;
static unsigned long events;  // anything a waiting fiber may wait for
static std::function<void()> kernel_body;
static void yield() { unsigned me = current; swapcontext(&fibers[me].context, &scheduler); threadIdx.x = current = me; }
static void __syncthreads() {
  Fiber& f = fibers[current];
  f.waiting = true, ++events;
  while (f.waiting) yield();
}
template <typename V> static size_t say(int site, const V& v) {
  auto& said = fibers[current].said[site];
  said.emplace_back();
  static_assert(sizeof(V) <= 64, "an exchange holds 64 bytes");
  memcpy(said.back().data(), &v, sizeof(V)), ++events;
  return said.size() - 1;
}
template <typename V> static V hear(int site, unsigned lane, size_t at) {
  while (fibers[lane].said[site].size() <= at) yield();
  V v;
  memcpy(&v, fibers[lane].said[site][at].data(), sizeof(V));
  return v;
}
template <typename V> static V shuffle(int site, V v, int mask) {
  return hear<V>(site, current ^ (unsigned)mask, say(site, v));
}
#define __shfl_xor(v, mask) shuffle(__COUNTER__, v, mask)
static inline unsigned __float_as_uint(float x) { unsigned u; memcpy(&u, &x, 4); return u; }
static inline float __uint_as_float(unsigned u) { float x; memcpy(&x, &u, 4); return x; }
static inline float widened(_Float16 x) { return (float)x; }
static inline float widened(__bf16 x) { unsigned short w; memcpy(&w, &x, 2); return __uint_as_float((unsigned)w << 16); }
template <typename E, int PER, typename V, typename C> static C product16(int site, const V& a, const V& b, C c) {
  struct Pair { V a, b; } mine = {a, b};
  const unsigned wave = current & ~63u, lane = current & 63u;
  const size_t at = say(site, mine);
  for (int i = 0; i < 4; ++i)
    for (unsigned part = 0; part < 4; ++part) {
      const Pair row = hear<Pair>(site, wave + part * 16 + lane / 16 * 4 + i, at), col = hear<Pair>(site, wave + part * 16 + lane % 16, at);
      E x[PER], y[PER];
      memcpy(x, &row.a, sizeof x), memcpy(y, &col.b, sizeof y);
      for (int k = 0; k < PER; ++k) c[i] = fmaf(widened(x[k]), widened(y[k]), c[i]);
    }
  return c;
}
#define __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, x, y, z) product16<_Float16, 8>(__COUNTER__, a, b, c)
#define __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, x, y, z) product16<_Float16, 4>(__COUNTER__, a, b, c)
#define __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, x, y, z) product16<__bf16, 8>(__COUNTER__, a, b, c)
#define __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, x, y, z) product16<__bf16, 4>(__COUNTER__, a, b, c)
static void fiber_main() {
  kernel_body();
  fibers[current].done = true, ++events;
  swapcontext(&fibers[current].context, &scheduler);
}
static int run_grid(Dim grid, unsigned threads, int last_first) {
  gridDim = grid;
  for (unsigned b = 0; b < grid.x * grid.y * grid.z; ++b) {
    blockIdx = Dim{b % grid.x, b / grid.x % grid.y, b / grid.x / grid.y};
    fibers.clear(), fibers.resize(threads);
    for (Fiber& f : fibers) {
      f.stack.resize(32768), f.done = f.waiting = false;
      getcontext(&f.context);
      f.context.uc_stack.ss_sp = f.stack.data(), f.context.uc_stack.ss_size = f.stack.size(), f.context.uc_link = nullptr;
      makecontext(&f.context, fiber_main, 0);
    }
    for (;;) {
      const unsigned long before = events;
      unsigned left = 0, waiting = 0;
      for (unsigned i = 0; i < threads; ++i) {
        const unsigned t = last_first ? threads - 1 - i : i;
        if (!fibers[t].done && !fibers[t].waiting) {
          threadIdx.x = current = t;
          swapcontext(&scheduler, &fibers[t].context);
        }
        left += !fibers[t].done, waiting += !fibers[t].done && fibers[t].waiting;
      }
      if (left == 0) break;
      if (waiting == left) for (Fiber& f : fibers) f.waiting = false;
      else if (events == before) return 1;  // lanes that wait for one that never comes
    }
  }
  return 0;
}
"""


def compiled(kernel: ir.Kernel, **options) -> tuple[ctypes.CDLL, int]:
    entry = f"krn_{kernel.name}"
    source, scratch = hipgen.emit(kernel, entry, **options)
    slots = [slot for name, kind in kernel.params for slot in ir.slots(name, kind)]
    kinds = [f"{hipgen.storage(d)}*" if role == "ptr" else hipgen.ctype(d) for _, d, role in slots]
    params = [f"{kind} p{i}" for i, kind in enumerate(kinds)]
    call = [f"p{i}" for i in range(len(kinds))] + (["scratch"] if scratch else [])
    text = (f"{SHIM}\n{source}\nextern \"C\" int run({', '.join([*params, 'char* scratch'])}, unsigned gx, unsigned gy, "
            f"unsigned gz, unsigned threads, int last_first) {{\n"
            f"  kernel_body = [=] {{ {entry}({', '.join(call)}); }};\n"
            "  return run_grid(Dim{gx, gy, gz}, threads, last_first);\n}\n")
    CACHE.mkdir(parents=True, exist_ok=True)
    library = CACHE / f"threads_{kernel.name}_{hashlib.sha256(text.encode()).hexdigest()[:24]}.so"
    if not library.exists():
        cpp, temporary = library.with_suffix(".cpp"), library.with_suffix(f".{os.getpid()}.tmp")
        cpp.write_text(text)
        result = subprocess.run([CLANG, "-O1", "-march=native", "-std=c++17", "-ffp-contract=off", "-fwrapv", "-w", "-shared",
                                 "-fPIC", "-x", "c++", str(cpp), "-o", str(temporary), "-lstdc++", "-lm"],
                                capture_output=True, text=True)
        if result.returncode:
            raise RuntimeError(f"the emitted source does not compile for the host:\n{result.stderr}\n{source}")
        temporary.replace(library)
    return ctypes.CDLL(str(library)), scratch


def run(kernel: ir.Kernel, args, launch=None, last_first: bool = False, **options) -> None:
    """One launch of `kernel` on numpy arrays (bf16 as uint16 words) and scalars; the same array twice is the same
    memory twice."""
    library, scratch = compiled(kernel, **options)
    values = runtime_args(kernel, args)
    grid = launch if launch is not None else geometry(kernel, values)
    native: list = []
    for (_, kind), value in zip(kernel.params, values):
        if isinstance(kind, ir.TensorType):
            assert value.flags.c_contiguous and value.ndim == kind.rank
            native += [ctypes.c_void_p(value.ctypes.data), *(ctypes.c_longlong(n) for n in value.shape)]
        elif kind.is_float:
            native.append(ctypes.c_double(value) if kind.bits == 64 else ctypes.c_float(value))
        else:
            native.append(ctypes.c_longlong(int(value)) if kind.bits == 64 else ctypes.c_int(int(value)))
    memory = np.zeros(scratch * grid.x * grid.y * grid.z + 1, np.uint8)
    dims = (ctypes.c_uint(n) for n in (grid.x, grid.y, grid.z, hipgen.threads(kernel)))
    assert library.run(*native, ctypes.c_void_p(memory.ctypes.data), *dims, ctypes.c_int(last_first)) == 0, "deadlock"
