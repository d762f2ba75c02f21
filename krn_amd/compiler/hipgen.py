"""Generic lowering of any captured tile program to HIP C++ for gfx950, compiled at run time with hiprtc.

This is the path for tile programs that are not one of the contraction shapes the hand-written MFMA kernels serve
(`cdna4.lower` decides). One workgroup of 256 or 1024 threads (`threads`) runs one block; tile variables live in LDS
with a validity byte per lane; a tile statement is one loop over its elements, strided over the workgroup. Its
arithmetic is the tile semantics of krn's C-family lowering (reference src/krn/compiler/emit.py): a product stages both
operands as float32 (invalid lanes zero) and runs one fused multiply-add per k in k order for each output element
(emit.py:788-796), a reduction takes the valid lanes of its axis from the first one (emit.py:997-1034; float32 sums in
up to 64 interleaved parts), stores skip invalid lanes and elements outside the tensor. The kernel ABI is krn's
generated-kernel ABI (reference src/krn/compiler/cuda.py:319 and ir.py:441-452): `extern "C" __global__`, a tensor is a
pointer plus one `long long` extent per axis, scalars by value.
"""

import math
from dataclasses import dataclass

from krn_amd.compiler import ir
from krn_amd.dtypes import BF16, BOOL, F8E4M3, F16, F32, F64, I8, I32, I64, PY_FLOAT, PY_INT, Dtype, Kind

LDS_LIMIT = 160 * 1024


class LoweringError(ValueError):
    """A tile program the generic gfx950 lowering does not cover."""


def ctype(dtype: Dtype) -> str:
    if dtype.is_narrow:
        return "unsigned char"
    named = {
        BOOL: "unsigned char", F16: "_Float16", BF16: "float", F32: "float", F64: "double", PY_INT: "long long",
        PY_FLOAT: "double", I8: "signed char", I32: "int", I64: "long long",
    }  # fmt: skip
    if dtype in named:
        return named[dtype]
    if dtype.kind is Kind.UINT:
        return {8: "unsigned char", 16: "unsigned short", 32: "unsigned", 64: "unsigned long long"}[dtype.bits]
    return {8: "signed char", 16: "short", 32: "int", 64: "long long"}[dtype.bits]


def storage(dtype: Dtype) -> str:
    return "unsigned short" if dtype == BF16 else ctype(dtype)


SIZES = {"unsigned char": 1, "signed char": 1, "_Float16": 2, "short": 2, "unsigned short": 2, "float": 4, "int": 4,
         "unsigned": 4, "double": 8, "long long": 8, "unsigned long long": 8}

PRELUDE = r"""
typedef unsigned int u32;
typedef _Float16 _k_half4 __attribute__((ext_vector_type(4)));
typedef short _k_short4 __attribute__((ext_vector_type(4)));
typedef _Float16 _k_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 _k_bf16x8 __attribute__((ext_vector_type(8)));
typedef float _k_float4 __attribute__((ext_vector_type(4)));
typedef int _k_int4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float kb16(float x) {
  u32 u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) u = (u | 0x400000u) & 0xffff0000u;
  else u = (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
  return __uint_as_float(u);
}
__device__ __forceinline__ float kb16_load(unsigned short w) { return __uint_as_float((u32)w << 16); }
__device__ __forceinline__ unsigned short kb16_word(float x) { return (unsigned short)(__float_as_uint(kb16(x)) >> 16); }
__device__ __forceinline__ float k8dec(unsigned char c) {
  int m = c & 7, e = (c >> 3) & 15;
  if ((c & 0x7f) == 0x7f) return __builtin_nanf("");
  float v = e ? ldexpf(1.0f + m * 0.125f, e - 7) : ldexpf(m * 0.125f, -6);
  return (c & 0x80) ? -v : v;
}
__device__ __forceinline__ unsigned char k8enc(float x) {
  if (x != x) return 0x7f;
  unsigned char sign = signbit(x) ? 0x80 : 0;
  float a = fabsf(x);
  if (a > 448.0f) a = 448.0f;
  int best = 0; float bd = __builtin_inff();
  for (int c = 0; c < 0x7f; ++c) {
    float d = fabsf(k8dec((unsigned char)c) - a);
    if (d < bd || (d == bd && (c & 1) == 0)) { bd = d; best = c; }
  }
  return sign | (unsigned char)best;
}
__device__ __forceinline__ float kmax(float a, float b) { return a != a ? a : b != b ? b : a > b ? a : b; }
__device__ __forceinline__ float kmin(float a, float b) { return a != a ? a : b != b ? b : a < b ? a : b; }
// activations as krn states them (reference compiler/emit.py:112-114)
__device__ __forceinline__ float krelu(float x) { return x < 0.0f ? 0.0f : x; }
__device__ __forceinline__ float kgelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.7071067811865476f)); }
__device__ __forceinline__ float ksilu(float x) { return x / (1.0f + expf(-x)); }
"""

MATH = {
    ir.Fn.EXP: "expf({0})", ir.Fn.EXP2: "exp2f({0})", ir.Fn.LOG: "logf({0})", ir.Fn.LOG2: "log2f({0})",
    ir.Fn.SQRT: "sqrtf({0})", ir.Fn.RSQRT: "(1.0f / sqrtf({0}))", ir.Fn.ABS: "fabsf({0})", ir.Fn.TANH: "tanhf({0})",
    ir.Fn.RELU: "krelu({0})", ir.Fn.GELU: "kgelu({0})", ir.Fn.SILU: "ksilu({0})",
    ir.Fn.SIGMOID: "(1.0f / (1.0f + expf(-({0}))))", ir.Fn.ERF: "erff({0})",
    ir.Fn.MAXIMUM: "kmax({0}, {1})", ir.Fn.MINIMUM: "kmin({0}, {1})",
}  # fmt: skip


@dataclass(frozen=True)
class MfmaForm:
    """A 16 x 16 x K_STEP matrix-core instruction the generic lowering uses for a product."""

    name: str
    builtin: str
    k_step: int
    element: str  # the staged operand element
    operand_vec: str  # one lane's operand of one instruction
    acc_vec: str
    integer: bool = False


# per operand type, the forms in order of preference: gfx950's 16x16x32 f16/bf16 instructions consume twice the K of
# the 16x16x16 ones (kept for products whose K is a multiple of 16 only); fp8 e4m3 (the OCP format on gfx950) and
# int8 consume 32 bytes of K per instruction
MFMA_FORMS = {
    F16: (MfmaForm("f16", "__builtin_amdgcn_mfma_f32_16x16x32_f16", 32, "unsigned short", "_k_half8", "_k_float4"),
          MfmaForm("f16", "__builtin_amdgcn_mfma_f32_16x16x16f16", 16, "unsigned short", "_k_half4", "_k_float4")),
    BF16: (MfmaForm("bf16", "__builtin_amdgcn_mfma_f32_16x16x32_bf16", 32, "unsigned short", "_k_bf16x8",
                    "_k_float4"),
           MfmaForm("bf16", "__builtin_amdgcn_mfma_f32_16x16x16bf16_1k", 16, "unsigned short", "_k_short4",
                    "_k_float4")),
    F8E4M3: (MfmaForm("fp8", "__builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8", 32, "unsigned char", "long",
                      "_k_float4"),),
    I8: (MfmaForm("i8", "__builtin_amdgcn_mfma_i32_16x16x32_i8", 32, "signed char", "long", "_k_int4", True),),
}


def mfma_form(s: ir.Accumulate) -> MfmaForm | None:
    """The matrix-core instruction for a product, when its operand types have one and the tile extents are whole
    instructions (m and n multiples of 16, k of the instruction's K); None keeps the scalar fused multiply-adds.
    f16/bf16/fp8 products accumulate in float32, int8 ones in int32 (exact, so any order gives the same result)."""
    (m, k), n = s.lhs.shape, s.rhs.shape[1]
    if s.lhs.dtype != s.rhs.dtype or s.lhs.dtype not in MFMA_FORMS or m % 16 or n % 16:
        return None
    for form in MFMA_FORMS[s.lhs.dtype]:
        if (s.acc.dtype == I32) != form.integer or (not form.integer and s.acc.dtype != F32):
            continue
        if k % form.k_step == 0:
            return form
    return None


MANY_BLOCKS = 1 << 22  # along x, of 1024 threads: 2^32


def threads(kernel: ir.Kernel, blocks: int = 1) -> int:
    """Threads of one block: 256, and 1024 for programs whose tiles have 4096 elements and more and whose products, if
    any, run on the matrix cores. Their LDS leaves room for one or two blocks on a CU, and 256 threads would be one
    wave per SIMD with nothing to cover its LDS latency (flash attention, 64 x 64 tiles, d = 32, 16 x 512:
    100 us with 256 threads, 51 with 1024). A scalar product keeps 256: fewer outputs per thread are more LDS reads per
    multiply-add. A launch's threads along an axis stay below 2^32, so MANY_BLOCKS take 256 as well."""
    large = max((math.prod(v.shape) for v in kernel.tiles), default=1) >= 4096
    scalar = any(isinstance(s, ir.Accumulate) and mfma_form(s) is None for s in ir.walk(kernel.body))
    return 1024 if large and not scalar and blocks < MANY_BLOCKS else 256


def products(kernel: ir.Kernel) -> list[str]:
    """How the generic lowering runs each product of `kernel`: "mfma 16x16x<K> <type>" or "scalar fma"."""
    found: list[str] = []

    def walk(statements) -> None:
        for s in statements:
            if isinstance(s, ir.Accumulate):
                form = mfma_form(s)
                found.append(f"mfma 16x16x{form.k_step} {form.name}" if form else "scalar fma")
            for field_name in ("body", "then", "orelse"):
                walk(getattr(s, field_name, ()) or ())

    walk(kernel.body)
    return found


# A program's own names in the source: prefixed, so that neither a parameter nor a name that capture gives a loop variable
# (`_i1` for the first `i`) can be one of the emitter's (`_i1` is a loop's column index), of the prelude's or of HIP's


def user(name: str) -> str:
    return f"u_{name}"


def dim(tensor: str, axis: int) -> str:
    """`tensor.shape[axis]`; no parameter can have this name (`user` begins with u, and no local with n)."""
    return f"n{axis}_{tensor}"


Access = tuple[tuple, str]  # a resource (("lds", first byte, end byte) or ("tensor", name)) and how it is indexed


class Emitter:
    """The source of one kernel. A statement's elementwise operations run fused, in one loop over its elements, each
    operation one rounded line; tile variables live in LDS, and so do the intermediate tiles that other threads read
    (reductions, staged product operands, transposed loads), in memory that the next statement reuses: a program's
    footprint is its variables and the largest statement, not every operation (flash attention with 64 x 64 tiles and
    d = 32: 321 KiB, in global scratch, before; 16 heads of 512 took 1270 us).

    Loops over the same elements need no barrier between them when each reads only what its own thread wrote: `sync`
    keeps what has been read and written since the last barrier and puts one only before a conflict. Tensors are told
    apart by their parameters' names, unless `overlapping`: then any two of them may share memory, and a statement's
    loads are complete before it, or a later one, stores."""

    def __init__(self, kernel: ir.Kernel, entry: str, overlapping: bool = False, blocks: int = 1) -> None:
        self.kernel, self.entry, self.overlapping = kernel, entry, overlapping
        self.threads = threads(kernel, blocks)
        self.mfma_products = 0
        self.lines: list[str] = []
        self.depth = 1
        self.count = 0
        self.names: dict[str, tuple[str, int, int]] = {}  # buffer -> element type, offset, bytes
        self.order: list[str] = []  # buffers in the order of their declaration
        self.top = self.peak = 0  # the statement's end of used memory, and the most any statement uses
        self.tile_vars: dict[str, tuple[str, str]] = {}
        self.node: dict[int, object] = {}  # what a statement has prepared for its expressions, by identity
        self.memo: dict[tuple, tuple[str, str]] = {}
        self.reads: list[Access] = []
        self.writes: list[Access] = []
        self.pending: list[tuple[Access, bool]] = []  # since the last barrier: access, whether it wrote
        self.open: tuple[tuple[int, ...], int, int] | None = None  # the last `elements` loop: shape, first and last line

    def put(self, text: str) -> None:
        self.lines.append("  " * self.depth + text)

    def fresh(self, stem: str) -> str:
        self.count += 1
        return f"_{stem}{self.count}"

    # ---- memory

    def reserve(self, name: str, element: str, size: int) -> str:
        nbytes = (SIZES[element] * max(size, 1) + 15) // 16 * 16
        self.names[name] = (element, self.top, nbytes)
        self.order.append(name)
        self.top += nbytes
        self.peak = max(self.peak, self.top)
        return name

    def buffer(self, dtype: Dtype, shape: tuple[int, ...], stem: str = "t") -> tuple[str, str]:
        self.count += 1
        size = math.prod(shape) if shape else 1
        return (self.reserve(f"{stem}{self.count}", ctype(dtype), size),
                self.reserve(f"{stem}{self.count}_v", "unsigned char", size))

    def access(self, name: str, pattern: str, write: bool = False) -> None:
        """Note that the loop being emitted touches buffer `name` at `pattern`: "e<size>" is the element of the
        thread's own index in a loop over <size> elements, "any" everything else."""
        _, start, nbytes = self.names[name]
        (self.writes if write else self.reads).append((("lds", start, start + nbytes), pattern))

    def conflict(self, a: Access, b: Access) -> bool:
        (ra, pa), (rb, pb) = a, b
        if ra[0] != rb[0] or (ra[0] == "tensor" and ra[1] != rb[1] and not self.overlapping):
            return False
        if ra[0] == "lds" and (ra[2] <= rb[1] or rb[2] <= ra[1]):
            return False
        return pa == "any" or pa != pb or ra != rb

    def sync(self, reads: list[Access], writes: list[Access]) -> None:
        """A barrier if these accesses meet one since the last barrier that another thread may have made."""
        if any(self.conflict(w, old) for w in writes for old, _ in self.pending) or any(
                self.conflict(r, old) for r in reads for old, wrote in self.pending if wrote):
            self.barrier()
        self.pending += [(r, False) for r in reads] + [(w, True) for w in writes]

    def barrier(self) -> None:
        self.put("__syncthreads();")
        self.pending = []

    def region(self, emit) -> None:
        """The lines `emit` puts, after the barrier their accesses need."""
        outer, reads, writes = self.lines, self.reads, self.writes
        self.lines, self.reads, self.writes, self.memo = [], [], [], {}
        emit()
        inner, self.lines = self.lines, outer
        self.sync(self.reads, self.writes)
        self.lines += inner
        self.reads, self.writes, self.memo = reads, writes, {}

    def loop(self, shape: tuple[int, ...], body) -> None:
        """`body(index names)` for every element of `shape`, strided over the workgroup."""
        def emit() -> None:
            self.put(f"for (int _e = threadIdx.x; _e < {math.prod(shape)}; _e += {self.threads}) {{")
            self.depth += 1
            names = []
            for a in range(len(shape)):
                self.put(f"const int _i{a} = _e / {math.prod(shape[a + 1:])} % {shape[a]};")
                names.append(f"_i{a}")
            body(names)
            self.depth -= 1
            self.put("}")

        self.region(emit)

    @staticmethod
    def aligned(idx: list[str], of: tuple[int, ...]) -> list[str]:
        """The indices of a tile of shape `of` broadcast numpy-style (aligned from the right) to the loop `idx`."""
        skip = len(idx) - len(of)
        return ["0" if extent == 1 else idx[a + skip] for a, extent in enumerate(of)]

    @staticmethod
    def linear(idx: list[str], of: tuple[int, ...]) -> str:
        return " + ".join(f"{i} * {math.prod(of[a + 1:])}" for a, i in enumerate(idx) if i != "0") or "0"

    # ---- the kernel

    def emit(self) -> tuple[str, int]:
        for var in self.kernel.tiles:
            self.tile_vars[var.name] = self.buffer(var.dtype, var.shape, stem=f"v_{var.name.strip('_')}_")
        self.fixed = self.top  # bytes of the variables; the statements' temporaries follow
        self.body(self.kernel.body)
        params = []
        for name, kind in self.kernel.params:
            if isinstance(kind, ir.TensorType):
                alone = "" if self.overlapping else "__restrict__ "
                params.append(f"{storage(kind.dtype)}* {alone}{user(name)}")
                params += [f"long long {dim(name, a)}" for a in range(kind.rank)]
            else:
                params.append(f"{ctype(kind if kind != I64 else PY_INT)} {user(name)}")
        total = self.peak
        scratch = total > LDS_LIMIT  # tiles beyond one CU's LDS live in a per-block slice of global scratch
        if scratch:
            params.append("char* __restrict__ _scratch")
        head = [PRELUDE, f'extern "C" __global__ __launch_bounds__({self.threads}) void {self.entry}({", ".join(params)}) {{']
        if scratch:
            head.append(f"  char* _block = _scratch + ((long long)blockIdx.x + (long long)blockIdx.y * gridDim.x + "
                        f"(long long)blockIdx.z * gridDim.x * gridDim.y) * {total}LL;")
        else:
            head.append(f"  __shared__ __attribute__((aligned(16))) char _block[{max(total - self.fixed, 16)}];")
        for name in self.order:
            element, offset, nbytes = self.names[name]
            if offset < self.fixed and not scratch:
                # a variable is an array of its own, which the compiler can tell from the others
                head.append(f"  __shared__ __attribute__((aligned(16))) {element} {name}[{nbytes // SIZES[element]}];")
            else:
                head.append(f"  {element}* {name} = ({element}*)(_block + {offset - (0 if scratch else self.fixed)});")
        self.scratch_bytes = total if scratch else 0
        head += ["  const long long bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;",
                 "  (void)bx; (void)by; (void)bz;"]
        return "\n".join([*head, *self.lines, "}", ""]), self.scratch_bytes

    def body(self, statements) -> None:
        self.open = None
        for s, following in zip(statements, [*statements[1:], None]):
            # `acc = zeros` right before `acc += a @ b`: the product starts from zero itself
            self.fresh_acc = isinstance(s, ir.Accumulate) and self.skipped is s.acc
            self.skipped = None
            if (isinstance(s, ir.TileAssign) and isinstance(s.value, ir.Zeros) and isinstance(following, ir.Accumulate)
                    and following.acc == s.var and not self.reads_var(following, s.var)):
                self.skipped = following.acc
                continue
            mark, self.node = self.top, {}
            getattr(self, f"stmt_{type(s).__name__}")(s)
            self.top = mark  # the statement's temporaries are dead
        self.open = None

    fresh_acc = False
    skipped: ir.Var | None = None

    @staticmethod
    def reads_var(s: ir.Accumulate, var: ir.Var) -> bool:
        def within(e: ir.Expr) -> bool:
            return (isinstance(e, ir.Var) and e.name == var.name) or any(within(child) for child in ir.children(e))

        return within(s.lhs) or within(s.rhs)

    # ---- expressions: `prepare` before the loop, `value` inside it

    def prepare(self, e: ir.Expr, product: bool = False) -> None:
        """What an expression's elements need before a loop can compute them: the starts of its loads, the results of
        its reductions, a transposed load turned through LDS (in a product the staging loop turns it)."""
        if id(e) in self.node or not e.shape or isinstance(e, ir.Var):
            return
        match e:
            case ir.TileLoad(slices=slices):
                starts = [self.fresh("s") for _ in slices]
                for name, sl in zip(starts, slices):
                    self.put(f"const long long {name} = {self.scalar(sl.start)};")
                self.node[id(e)] = starts
            case ir.Arange(start=start):
                name = self.fresh("s")
                self.put(f"const long long {name} = {self.scalar(start)};")
                self.node[id(e)] = name
            case ir.Reduce():
                self.prepare(e.operand)
                self.node[id(e)] = self.reduce(e)
            case ir.Transpose(operand=o) if not product and self.loads(o):
                self.prepare(o)
                self.node[id(e)] = self.materialise(o)
            case _:
                for child in ir.children(e):
                    self.prepare(child, product)
                self.node.setdefault(id(e), None)

    @staticmethod
    def loads(e: ir.Expr, tensor: str | None = None) -> bool:
        """Whether evaluating `e` loads from a tensor (from `tensor`)."""
        if isinstance(e, ir.TileLoad):
            return tensor is None or e.tensor.name == tensor
        return any(Emitter.loads(child, tensor) for child in ir.children(e))

    def materialise(self, e: ir.Expr) -> tuple[str, str]:
        value, valid = self.buffer(e.dtype, e.shape)

        def body(idx):
            x, ok = self.value(e, idx)
            self.store(value, valid, "_e", x, ok, f"e{math.prod(e.shape)}")

        self.loop(e.shape, body)
        return value, valid

    def store(self, value: str, valid: str, at: str, x: str, ok: str, pattern: str) -> None:
        self.put(f"{value}[{at}] = {x}; {valid}[{at}] = {ok};")
        self.access(value, pattern, write=True)
        self.access(valid, pattern, write=True)

    def fetch(self, buffers: tuple[str, str], idx: list[str], shape: tuple[int, ...], own: bool) -> tuple[str, str]:
        """An element of a tile in LDS; `own`: it is the loop's own element."""
        at = "_e" if own else self.linear(idx, shape)
        for name in buffers:
            self.access(name, f"e{math.prod(shape)}" if own else "any")
        return f"{buffers[0]}[{at}]", f"{buffers[1]}[{at}]"

    def line(self, dtype: Dtype, text: str) -> str:
        name = self.fresh("x")
        self.put(f"const {ctype(dtype)} {name} = {text};")
        return name

    @staticmethod
    def both(checks: list[str]) -> str:
        kept = list(dict.fromkeys(c for c in checks if c != "1"))
        return " & ".join(kept) or "1"

    def value(self, e: ir.Expr, idx: list[str]) -> tuple[str, str]:
        """The element of `e` at `idx` (its value and its validity), computed in the current loop."""
        if not e.shape:
            return f"(({ctype(e.dtype)}){self.scalar(e)})", "1"  # of its own type: C adds narrow integers as int
        idx = self.aligned(idx, e.shape)
        key = (id(e), *idx)
        if key not in self.memo:
            self.memo[key] = self.compute(e, idx)
        return self.memo[key]

    def own(self, idx: list[str], shape: tuple[int, ...]) -> bool:
        """Whether `idx` is the element of the surrounding `loop`, whose shape is `shape`."""
        return self.loop_shape == shape and idx == self.aligned([f"_i{a}" for a in range(len(shape))], shape)

    loop_shape: tuple[int, ...] | None = None

    def compute(self, e: ir.Expr, idx: list[str]) -> tuple[str, str]:
        match e:
            case ir.Var(name=n):
                return self.fetch(self.tile_vars[n], idx, e.shape, self.own(idx, e.shape))
            case ir.Reduce():
                return self.fetch(self.node[id(e)], idx, e.shape, False)
            case ir.Zeros():
                return f"(({ctype(e.dtype)})0)", "1"
            case ir.Arange():
                return self.line(e.dtype, f"({ctype(e.dtype)})({self.node[id(e)]} + {idx[e.axis]})"), "1"
            case ir.Transpose(operand=o):
                if self.node.get(id(e)):
                    return self.fetch(self.node[id(e)], [idx[1], idx[0]], o.shape, False)
                return self.value(o, [idx[1], idx[0]])
            case ir.TileLoad():
                return self.load(e, idx)
        operands = [self.value(child, idx) for child in ir.children(e)]
        texts, valid = [v for v, _ in operands], self.both([ok for _, ok in operands])
        match e:
            case ir.Cast(operand=o):
                text = self.cast(texts[0], o.dtype, e.dtype)
            case ir.Unary():
                text = self.rounded(f"-{texts[0]}", e.dtype)
            case ir.Binary():
                text = self.binary(e, texts)
            case ir.Math(fn=fn):
                template = MATH[fn]
                if e.dtype == F64:
                    template = template.replace("f(", "(")
                text = self.rounded(template.format(*texts), e.dtype)
            case ir.Select():
                text = f"({texts[0]} ? {texts[1]} : {texts[2]})"
            case _:
                raise LoweringError(f"tile {type(e).__name__} is not lowered")
        if valid.count("&") > 2:
            valid = self.line(BOOL, valid)
        return self.line(e.dtype, text), valid

    def cells(self, starts: list[str], slices, tensor: str, idx: list[str]) -> tuple[str, str]:
        """The linear index of a tile element in its tensor, and whether it lies inside."""
        axes = iter(idx)
        cells = [st if sl.squeeze else f"({st} + {next(axes)})" for st, sl in zip(starts, slices)]
        inside = " && ".join(f"{c} >= 0 && {c} < {dim(tensor, a)}" for a, c in enumerate(cells))
        linear = " + ".join(c + "".join(f" * {dim(tensor, b)}" for b in range(a + 1, len(cells)))
                            for a, c in enumerate(cells))
        return linear, inside

    def load(self, e: ir.TileLoad, idx: list[str]) -> tuple[str, str]:
        tensor = e.tensor.name
        # a tile axis of extent 1 that the loop broadcasts is element 0 of its slice
        linear, inside = self.cells(self.node[id(e)], e.slices, tensor, idx)
        ok = self.line(BOOL, inside)
        element = f"{user(tensor)}[{linear}]"
        if e.dtype == BF16:
            element = f"kb16_load({element})"
        self.reads.append((("tensor", tensor), "any"))
        return self.line(e.dtype, f"{ok} ? {element} : ({ctype(e.dtype)})0"), ok

    def binary(self, e: ir.Binary, t: list[str]) -> str:
        op = {ir.Op.AND: "&", ir.Op.OR: "|"}.get(e.op, e.op.value)
        if e.op is ir.Op.MOD and e.lhs.dtype.is_float:
            return f"fmodf({t[0]}, {t[1]})"
        if e.op in ir.COMPARISONS:
            return f"({t[0]} {op} {t[1]})"
        if e.op is ir.Op.DIV and e.lhs.dtype.is_int:
            return f"({t[1]} ? {t[0]} / {t[1]} : 0)"
        return self.rounded(f"{t[0]} {op} {t[1]}", e.dtype)

    def reduce(self, e: ir.Reduce) -> tuple[str, str]:
        """A reduction over one axis, valid lanes only. float32 and integer ones share an output among up to 64
        neighbouring threads, each from its first valid lane, joined by shuffles; the 16-bit types, which round after
        every step, keep one thread and the order of the axis."""
        value, valid = self.buffer(e.dtype, e.shape)
        shape, axis = e.operand.shape, e.axis
        outputs, extent = math.prod(shape) // shape[axis], shape[axis]
        join = {
            ir.Reduction.MAX: "_acc = (_y > _acc || _y != _y) ? _y : _acc;",
            ir.Reduction.MIN: "_acc = (_y < _acc || _y != _y) ? _y : _acc;",
            ir.Reduction.SUM: "_acc = _acc + _y;",
        }[e.op]
        if e.dtype == BF16:
            join = join.replace("_acc + _y", "kb16(_acc + _y)")
        group = 1
        if e.dtype in (F32, I32) or (e.op is not ir.Reduction.SUM and e.dtype == BF16):
            while group < 64 and 2 * group <= extent and outputs * group < self.threads:
                group *= 2
        kept = [s for a, s in enumerate(shape) if a != axis]
        acc = ctype(e.dtype)

        def emit() -> None:
            self.put(f"for (int _t = threadIdx.x; _t < {outputs * group}; _t += {self.threads}) {{")
            self.depth += 1
            self.put(f"const int _o = _t / {group};")
            idx, position = [], 0
            for a in range(len(shape)):
                if a == axis:
                    idx.append("_r")
                else:
                    idx.append(f"(_o / {math.prod(kept[position + 1:])} % {kept[position]})")
                    position += 1
            self.put(f"{acc} _acc = 0; unsigned char _seen = 0;")
            self.put(f"for (int _r = _t % {group}; _r < {extent}; _r += {group}) {{")
            self.depth += 1
            x, ok = self.value(e.operand, idx)
            take = f"{acc} _y = {x}; if (_seen) {{ {join} }} else {{ _acc = _y; _seen = 1; }}"
            self.put(f"{{ {take} }}" if ok == "1" else f"if ({ok}) {{ {take} }}")
            self.depth -= 1
            self.put("}")
            if group > 1:
                self.put(f"for (int _g = {group // 2}; _g; _g >>= 1) {{")
                self.put(f"  const {acc} _y = __shfl_xor(_acc, _g); const int _other = __shfl_xor((int)_seen, _g);")
                self.put(f"  if (_other) {{ if (_seen) {{ {join} }} else _acc = _y; _seen = 1; }}")
                self.put("}")
            self.put(f"if (_t % {group} == 0) {{ {value}[_o] = _acc; {valid}[_o] = _seen; }}")
            self.depth -= 1
            self.put("}")
            for name in (value, valid):
                self.access(name, "any", write=True)

        self.region(emit)
        return value, valid

    # ---- statements

    def stmt_TileAssign(self, s: ir.TileAssign) -> None:
        if s.value == s.var:
            return
        self.prepare(s.value)
        target = self.tile_vars[s.var.name]
        if self.reads_elsewhere(s.value, s.var, s.var.shape):
            temporary = self.materialise(s.value)  # other threads' elements of the variable: computed before it changes
            shape = s.value.shape
            self.loop(s.var.shape, lambda idx: self.store(
                *target, "_e", *self.fetch(temporary, self.aligned(idx, shape), shape, False),
                f"e{math.prod(s.var.shape)}"))
            return

        def body(idx):
            x, ok = self.value(s.value, idx)
            self.store(*target, "_e", x, ok, f"e{math.prod(s.var.shape)}")

        self.elements(s.var.shape, body)

    def elements(self, shape: tuple[int, ...], body) -> None:
        """`loop` whose index is the thread's own element of every tile of this shape. It joins the loop just before it
        when that one runs over the same elements and nothing but the starts of slices stands between them."""
        before = len(self.lines)
        self.loop_shape = shape
        self.loop(shape, body)
        self.loop_shape = None
        added = self.lines[before:]
        if self.open is not None and self.open[0] == shape and "__syncthreads();" not in added[0]:
            _, first, last = self.open
            between = self.lines[last + 1:before]
            if all(line.lstrip().startswith("const long long _s") for line in between):
                inner = added[1 + len(shape):-1]  # without the loop's head, index names and end
                self.lines[first:] = [*between, *self.lines[first:last], *inner, self.lines[last]]
                self.open = (shape, first + len(between), len(self.lines) - 1)
                return
        start = before + (1 if "__syncthreads();" in added[0] else 0)
        self.open = (shape, start, len(self.lines) - 1)

    @staticmethod
    def reads_elsewhere(e: ir.Expr, var: ir.Var, shape: tuple[int, ...] | None) -> bool:
        """Whether computing `e` at an element reads `var` at another one (through a transpose or a broadcast)."""
        if isinstance(e, ir.Var):
            return e.name == var.name and e.shape != shape
        if isinstance(e, ir.Reduce):
            return False  # computed before the loop
        inner = None if isinstance(e, ir.Transpose) else shape
        return any(Emitter.reads_elsewhere(child, var, inner) for child in ir.children(e))

    def stmt_TileStore(self, s: ir.TileStore) -> None:
        self.prepare(s.value)
        tensor, starts = s.tensor.name, [self.fresh("s") for _ in s.slices]
        for name, sl in zip(starts, s.slices):
            self.put(f"const long long {name} = {self.scalar(sl.start)};")
        # a value loaded from the memory it is stored to is complete before any of it is stored
        shared = None if self.overlapping else tensor
        temporary = self.materialise(s.value) if self.loads(s.value, shared) else None

        def store(idx):
            linear, inside = self.cells(starts, s.slices, tensor, idx)
            if temporary is not None:
                x, ok = self.fetch(temporary, idx, s.value.shape, False)
            else:
                x, ok = self.value(s.value, idx)
            element = f"kb16_word({x})" if s.tensor.type.dtype == BF16 else x
            self.put(f"if ({'' if ok == '1' else f'({ok}) && '}{inside}) {user(tensor)}[{linear}] = {element};")
            self.writes.append((("tensor", tensor), "any"))

        self.elements(s.value.shape, store)

    def stmt_Accumulate(self, s: ir.Accumulate) -> None:
        self.prepare(s.lhs, product=True)
        self.prepare(s.rhs, product=True)
        form = mfma_form(s)
        if form is not None:
            self.mfma_product(s, form)
        else:
            self.scalar_product(s)
        self.product_validity(s)

    def product_validity(self, s: ir.Accumulate) -> None:
        """An accumulator element stays valid when its row of lhs and its column of rhs have a valid lane each."""
        (m, k), n = s.lhs.shape, s.rhs.shape[1]
        flags = [self.any_valid(s.lhs, m, k, False), self.any_valid(s.rhs, n, k, True)]
        valid, zero = self.tile_vars[s.acc.name][1], self.fresh_acc

        def body(idx):
            checks = [flag[0] if isinstance(flag, tuple) else f"{flag}[{i}]" for flag, i in zip(flags, idx)]
            for flag in flags:
                if isinstance(flag, str):
                    self.access(flag, "any")
            checks = [self.line(BOOL, flag[1](i)) if isinstance(flag, tuple) else c
                      for flag, i, c in zip(flags, idx, checks)]
            if not zero:
                self.access(valid, f"e{m * n}")
                checks = [f"{valid}[_e]", *checks]
            self.access(valid, f"e{m * n}", write=True)
            self.put(f"{valid}[_e] = {self.both(checks)};")

        self.elements((m, n), body)

    def any_valid(self, e: ir.Expr, rows: int, k: int, transposed: bool):
        """Whether row i of an operand (column i of a (k, n) one) has a valid lane: the name of a flag per row, or, for
        a load, whose lanes are valid in a block, ("load", the condition as a function of i)."""
        turned = isinstance(e, ir.Transpose)
        load = e.operand if turned else e
        if isinstance(load, ir.TileLoad):
            starts, tensor = self.node[id(load)], load.tensor.name
            kept = [a for a, sl in enumerate(load.slices) if not sl.squeeze]
            row_axis, k_axis = (kept[1], kept[0]) if transposed != turned else (kept[0], kept[1])

            def condition(i: str) -> str:
                checks = [f"{st} >= 0 && {st} < {dim(tensor, a)}" for a, (st, sl) in enumerate(zip(starts, load.slices))
                          if sl.squeeze]
                checks.append(f"{starts[k_axis]} < {dim(tensor, k_axis)} && {starts[k_axis]} + {k} > 0")
                checks.append(f"{starts[row_axis]} + {i} >= 0 && {starts[row_axis]} + {i} < {dim(tensor, row_axis)}")
                return " && ".join(checks)

            return ("load", condition)
        flag = self.reserve(self.fresh("any"), "unsigned char", rows)

        def emit() -> None:
            self.put(f"for (int _t = threadIdx.x; _t < {rows}; _t += {self.threads}) {{")
            self.depth += 1
            self.put("unsigned char _any = 0;")
            self.put(f"for (int _k = 0; _k < {k}; ++_k) {{")
            self.depth += 1
            self.put(f"_any |= {self.value(e, ['_k', '_t'] if transposed else ['_t', '_k'])[1]};")
            self.depth -= 1
            self.put("}")
            self.put(f"{flag}[_t] = _any;")
            self.access(flag, "any", write=True)
            self.depth -= 1
            self.put("}")

        self.region(emit)
        return flag

    def scalar_product(self, s: ir.Accumulate) -> None:
        """One fused multiply-add per k in k order for each output. Both operands are staged k-major, and a thread keeps
        a block of outputs in registers over the whole k: of 4 x 4 two 16-byte LDS reads per 16 multiply-adds (one
        output at a time, two reads each, 256^3 took 38 us)."""
        (m, k), n = s.lhs.shape, s.rhs.shape[1]
        acc = self.tile_vars[s.acc.name][0]
        integer = s.acc.dtype == I32
        stage = "int" if integer else "float"
        zero = self.fresh_acc
        a, b = self.staged(stage, s.lhs, m, k, False), self.staged(stage, s.rhs, n, k, True)
        rm, rn = next((r for r in ((4, 4), (2, 4), (1, 4), (2, 2), (1, 2), (1, 1))
                       if m % r[0] == 0 and n % r[1] == 0 and (m // r[0]) * (n // r[1]) >= min(self.threads, m * n)), (1, 1))

        def emit() -> None:
            self.put(f"for (int _t = threadIdx.x; _t < {(m // rm) * (n // rn)}; _t += {self.threads}) {{")
            self.depth += 1
            self.put(f"const int _i = _t / {n // rn} * {rm}, _j = _t % {n // rn} * {rn};")
            kind = "unsigned" if integer else "float"
            self.put(f"{kind} _s[{rm}][{rn}];")
            start = "0" if zero else f"({kind}){acc}[(_i + _y) * {n} + _j + _x]"
            each = f"for (int _y = 0; _y < {rm}; ++_y) for (int _x = 0; _x < {rn}; ++_x)"
            self.put(f"_Pragma(\"unroll\") {each} _s[_y][_x] = {start};")
            self.put(f"_Pragma(\"unroll 4\") for (int _k = 0; _k < {k}; ++_k) {{")
            self.put(f"  {stage} _p[{rm}], _q[{rn}];")
            self.put(f"  for (int _y = 0; _y < {rm}; ++_y) _p[_y] = {a}[_k * {m + 4} + _i + _y];")
            self.put(f"  for (int _x = 0; _x < {rn}; ++_x) _q[_x] = {b}[_k * {n + 4} + _j + _x];")
            step = ("_s[_y][_x] += (unsigned)(_p[_y] * _q[_x]);" if integer
                    else "_s[_y][_x] = fmaf(_p[_y], _q[_x], _s[_y][_x]);")
            self.put(f"  _Pragma(\"unroll\") {each} {step}")
            self.put("}")
            self.put(f"_Pragma(\"unroll\") {each} {acc}[(_i + _y) * {n} + _j + _x] = ({stage})_s[_y][_x];")
            self.depth -= 1
            self.put("}")
            for name in (a, b, *(() if zero else (acc,))):
                self.access(name, "any")
            self.access(acc, "any", write=True)

        self.region(emit)

    def staged(self, stage: str, e: ir.Expr, rows: int, k: int, transposed: bool) -> str:
        """An operand of a scalar product in LDS as `k` rows of `rows` elements (and four more, so that a column of
        them is not in one bank), invalid lanes zero; `transposed` reads
        a (k, rows) tile. The loop runs along the operand's own rows, so that loads from a tensor are contiguous."""
        name = self.reserve(self.fresh("st"), stage, (rows + 4) * k)
        along_rows = transposed != isinstance(e, ir.Transpose)

        def body(idx):
            kk, rr = (idx[0], idx[1]) if along_rows else (idx[1], idx[0])
            x, ok = self.value(e, [kk, rr] if transposed else [rr, kk])
            element = f"k8dec({x})" if e.dtype.is_narrow else f"({stage}){x}"
            self.put(f"{name}[{kk} * {rows + 4} + {rr}] = {element if ok == '1' else f'({ok}) ? {element} : ({stage})0'};")
            self.access(name, "any", write=True)

        self.loop((k, rows) if along_rows else (rows, k), body)
        return name

    def mfma_product(self, s: ir.Accumulate, form: "MfmaForm") -> None:
        """acc[m, n] += lhs[m, k] @ rhs[k, n] on the matrix cores: both operands staged into LDS K-contiguous as the
        instruction's operand type (invalid lanes 0, so they add nothing), then each wave takes 16 x 16 output blocks
        in turn, loads the block's accumulators, runs k / K_STEP MFMAs and writes them back. Lane l of
        a 16x16xK MFMA holds operand row (or column) l % 16 and K_STEP / 4 consecutive k from (l / 16) * K_STEP / 4,
        and accumulators rows 4 (l / 16) + i, column l % 16 (reference compiler/hip.py:70-97 `AMDMFMA.product`,
        compiler/emit.py:924-955 `matrix_stage`). Staged rows are 16 bytes longer than K: 16 rows of a multiple of 128
        bytes would meet in one bank."""
        acc = self.tile_vars[s.acc.name][0]
        (m, k), n = s.lhs.shape, s.rhs.shape[1]
        per = form.k_step // 4  # operand elements per lane per instruction
        pitch, zero = k + 16 // SIZES[form.element], self.fresh_acc
        at = self.mfma_stage(form, s.lhs, m, k, pitch, transposed=False)
        bt = self.mfma_stage(form, s.rhs, n, k, pitch, transposed=True)
        acc_t = "int" if form.integer else "float"

        def emit() -> None:
            self.put("{")
            self.put("  const int _w = threadIdx.x >> 6, _l = threadIdx.x & 63, _r = _l & 15, _q = _l >> 4;")
            self.put(f"  for (int _blk = _w; _blk < {(m // 16) * (n // 16)}; _blk += {self.threads // 64}) {{")
            self.put(f"    const int _m0 = (_blk / {n // 16}) * 16, _n0 = (_blk % {n // 16}) * 16;")
            self.put(f"    {form.acc_vec} _c;")
            start = "0" if zero else f"{acc}[(_m0 + 4 * _q + _i) * {n} + _n0 + _r]"
            self.put(f"    for (int _i = 0; _i < 4; ++_i) _c[_i] = {start};")
            self.put(f"    for (int _k = 0; _k < {k}; _k += {form.k_step}) {{")
            vec = form.operand_vec
            self.put(f"      const {vec} _a = *(const {vec}*)&{at}[(_m0 + _r) * {pitch} + _k + _q * {per}];")
            self.put(f"      const {vec} _b = *(const {vec}*)&{bt}[(_n0 + _r) * {pitch} + _k + _q * {per}];")
            self.put(f"      _c = {form.builtin}(_a, _b, _c, 0, 0, 0);")
            self.put("    }")
            self.put(f"    for (int _i = 0; _i < 4; ++_i) {acc}[(_m0 + 4 * _q + _i) * {n} + _n0 + _r] = ({acc_t})_c[_i];")
            self.put("  }")
            self.put("}")
            for name in (at, bt, *(() if zero else (acc,))):
                self.access(name, "any")
            self.access(acc, "any", write=True)

        self.region(emit)
        self.mfma_products += 1

    def mfma_stage(self, form: "MfmaForm", e: ir.Expr, rows: int, k: int, pitch: int, transposed: bool) -> str:
        """An operand in LDS as `rows` K-contiguous rows of the instruction's element bits; `transposed` reads a
        (k, rows) tile. The loop runs along the operand's own rows, so that loads from a tensor are contiguous."""
        name = self.reserve(self.fresh("mf"), form.element, rows * pitch)
        along_rows = transposed != isinstance(e, ir.Transpose)

        def body(idx):
            kk, rr = (idx[0], idx[1]) if along_rows else (idx[1], idx[0])
            x, ok = self.value(e, [kk, rr] if transposed else [rr, kk])
            bits = self.mfma_bits(form, x)
            self.put(f"{name}[{rr} * {pitch} + {kk}] = {bits if ok == '1' else f'({ok}) ? {bits} : ({form.element})0'};")
            self.access(name, "any", write=True)

        self.loop((k, rows) if along_rows else (rows, k), body)
        return name

    def stmt_For(self, s: ir.For) -> None:
        if self.pipelined_product(s):
            return
        var = user(s.var.name)
        if self.pending:
            self.barrier()  # the body's first accesses are checked against its own last ones only
        self.put(f"for (long long {var} = {self.scalar(s.lo)}; {var} < {self.scalar(s.hi)}; {var} += {s.step}) {{")
        self.depth += 1
        self.body(s.body)
        if self.pending:
            self.barrier()
        self.depth -= 1
        self.put("}")

    def pipelined_product(self, s: ir.For) -> bool:
        """The loop of a matrix product, `acc += a[.., ks] @ b[ks, ..]` (or the transpose of b[.., ks]) alone in its body:
        the accumulators stay in registers over the whole loop, the next step's elements are loaded while this one
        multiplies, and two LDS stages leave one barrier per step (f32 256^3 with 32 x 32 tiles, 16 steps of one load's
        latency each: 21.6 us before, 13.4 now). Anything else (other statements in the body, computed operands, tiles with more
        outputs than the threads hold) is False, and runs statement by statement."""
        if len(s.body) != 1 or not isinstance(s.body[0], ir.Accumulate):
            return False
        product = s.body[0]
        lhs, rhs = product.lhs, product.rhs
        turned = isinstance(rhs, ir.Transpose)
        loads = (lhs, rhs.operand if turned else rhs)
        if not all(isinstance(e, ir.TileLoad) and len(e.shape) == 2 for e in loads):
            return False
        (m, k), n, var = lhs.shape, rhs.shape[1], user(s.var.name)
        axes = [[a for a, sl in enumerate(e.slices) if not sl.squeeze] for e in loads]
        k_axes = [axes[0][1], axes[1][1] if turned else axes[1][0]]
        if any(self.mentions(sl.start, s.var.name) for e, ka in zip(loads, k_axes) for a, sl in enumerate(e.slices) if a != ka):
            return False
        form, integer = mfma_form(product), product.acc.dtype == I32
        acc, valid = self.tile_vars[product.acc.name]
        waves = self.threads // 64
        if form is not None:
            element, pitches = form.element, (k + 16 // SIZES[form.element],) * 2
            sizes = (m * pitches[0], n * pitches[1])
            held = -(-(m // 16) * (n // 16) // waves)
            if held > 16:
                return False
        else:
            element, pitches = ("int" if integer else "float"), (m + 4, n + 4)
            sizes = (k * pitches[0], k * pitches[1])
            shape = next((r for r in ((1, 1), (1, 2), (2, 2), (2, 4), (4, 4), (4, 8), (8, 8))
                          if m % r[0] == 0 and n % r[1] == 0 and (m // r[0]) * (n // r[1]) <= self.threads), None)
            if shape is None:
                return False
        if self.top + 2 * sum(sizes) * SIZES[element] + 64 > LDS_LIMIT:
            return False
        stages = [self.reserve(self.fresh("st"), element, 2 * size) for size in sizes]
        counts = [-(-m * k // self.threads), -(-n * k // self.threads)]
        regs = [self.fresh("r"), self.fresh("r")]

        def each(body) -> None:
            """`body(stage, registers, index, expression, row, k position)` for every element a thread moves."""
            for i, (e, rows) in enumerate(((lhs, m), (rhs, n))):
                along_rows = i == 1 and not turned
                inner = rows if along_rows else k
                self.put(f'_Pragma("unroll") for (int _u = 0; _u < {counts[i]}; ++_u) {{')
                self.depth += 1
                self.put(f"const int _e = threadIdx.x + _u * {self.threads}, _i0 = _e / {inner}, _i1 = _e % {inner};")
                whole = rows * k % self.threads == 0
                self.put("{" if whole else f"if (_e < {rows * k}) {{")
                self.memo = {}
                row, at = ("_i1", "_i0") if along_rows else ("_i0", "_i1")
                body(i, e, row, at)
                self.put("}")
                self.depth -= 1
                self.put("}")

        def fetch() -> None:
            self.node, reads = {}, self.reads
            for e in (lhs, rhs):
                self.prepare(e, product=True)

            def one(i, e, row, at):
                x, ok = self.value(e, [row, at] if i == 0 else [at, row])
                if form is None:
                    x = f"k8dec({x})" if e.dtype.is_narrow else f"({element}){x}"
                else:
                    x = self.mfma_bits(form, x)
                self.put(f"{regs[i]}[_u] = ({ok}) ? {x} : ({element})0;")

            each(one)
            self.reads, self.memo = reads, {}

        def stage(i, e, row, at):
            place = f"{row} * {pitches[i]} + {at}" if form is not None else f"{at} * {pitches[i]} + {row}"
            self.put(f"{stages[i]}[_p * {sizes[i]} + {place}] = {regs[i]}[_u];")

        if self.pending:
            self.barrier()
        hi = self.scalar(s.hi)
        self.put(f"long long {var} = {self.scalar(s.lo)};")
        self.put(f"if ({var} < {hi}) {{")
        self.depth += 1
        for name, count in zip(regs, counts):
            self.put(f"{element} {name}[{count}];")
        self.put("int _p = 0; unsigned char _kok = 1;")
        kind = "unsigned" if integer else "float"
        if form is not None:
            at16 = f"[(_m0 + 4 * _q + _i) * {n} + _n0 + _r]"
            self.put("const int _w = threadIdx.x >> 6, _l = threadIdx.x & 63, _r = _l & 15, _q = _l >> 4;")
            self.put(f"{form.acc_vec} _c[{held}];")
            blocks = (f'_Pragma("unroll") for (int _b = 0; _b < {held}; ++_b) {{ const int _blk = _w + _b * {waves}, '
                      f"_m0 = _blk / {n // 16} * 16, _n0 = _blk % {n // 16} * 16; "
                      f"if (_blk < {(m // 16) * (n // 16)}) {{")
            self.put(f"{blocks} for (int _i = 0; _i < 4; ++_i) _c[_b][_i] = {acc}{at16}; }} }}")
        else:
            rm, rn = shape
            live = f"if (threadIdx.x < {(m // rm) * (n // rn)})"
            self.put(f"const int _i = threadIdx.x / {n // rn} * {rm}, _j = threadIdx.x % {n // rn} * {rn};")
            self.put(f"{kind} _s[{rm}][{rn}];")
            cell = (f'_Pragma("unroll") for (int _y = 0; _y < {rm}; ++_y) _Pragma("unroll") '
                    f"for (int _x = 0; _x < {rn}; ++_x)")
            self.put(f"{live} {{ {cell} _s[_y][_x] = ({kind}){acc}[(_i + _y) * {n} + _j + _x]; }}")
        self.put("{")
        self.depth += 1
        fetch()
        self.depth -= 1
        self.put("}")
        self.put("for (;;) {")
        self.depth += 1
        each(stage)
        self.put("__syncthreads();")  # the other stage's readers are a whole step behind
        self.put(f"const long long _next = {var} + {s.step};")
        self.put(f"if (_next < {hi}) {{")
        self.depth += 1
        self.put(f"const long long {var} = _next;")
        fetch()
        self.depth -= 1
        self.put("}")
        for e, ka in zip(loads, k_axes):
            start = self.scalar(e.slices[ka].start)
            self.put(f"_kok &= ({start}) < {dim(e.tensor.name, ka)} && ({start}) + {k} > 0;")
        if form is not None:
            per, vec = form.k_step // 4, form.operand_vec
            self.put(f"{blocks} _Pragma(\"unroll\") for (int _k = 0; _k < {k}; _k += {form.k_step}) {{")
            for name, stem, origin, i in (("_a", stages[0], "_m0", 0), ("_b2", stages[1], "_n0", 1)):
                self.put(f"  const {vec} {name} = *(const {vec}*)&{stem}[_p * {sizes[i]} + ({origin} + _r) * {pitches[i]}"
                         f" + _k + _q * {per}];")
            self.put(f"  _c[_b] = {form.builtin}(_a, _b2, _c[_b], 0, 0, 0);")
            self.put("} } }")
            self.mfma_products += 1
        else:
            self.put(f"{live} {{")
            self.put(f'  _Pragma("unroll 8") for (int _k = 0; _k < {k}; ++_k) {{')
            self.put(f"    {element} _f[{rm}], _g[{rn}];")
            self.put(f"    for (int _y = 0; _y < {rm}; ++_y) _f[_y] = "
                     f"{stages[0]}[_p * {sizes[0]} + _k * {pitches[0]} + _i + _y];")
            self.put(f"    for (int _x = 0; _x < {rn}; ++_x) _g[_x] = "
                     f"{stages[1]}[_p * {sizes[1]} + _k * {pitches[1]} + _j + _x];")
            step = ("_s[_y][_x] += (unsigned)(_f[_y] * _g[_x]);" if integer
                    else "_s[_y][_x] = fmaf(_f[_y], _g[_x], _s[_y][_x]);")
            self.put(f"    {cell} {step}")
            self.put("  }")
            self.put("}")
        self.put(f"if (_next >= {hi}) break;")
        self.put(f"{var} = _next; _p ^= 1;")
        self.depth -= 1
        self.put("}")
        if form is not None:
            cast = "int" if form.integer else "float"
            self.put(f"{blocks} for (int _i = 0; _i < 4; ++_i) {acc}{at16} = ({cast})_c[_b][_i]; }} }}")
        else:
            self.put(f"{live} {{ {cell} {acc}[(_i + _y) * {n} + _j + _x] = ({element})_s[_y][_x]; }}")
        self.node = {}
        for e in (lhs, rhs):
            self.prepare(e, product=True)
        rows, cols = self.any_valid(lhs, m, k, False)[1], self.any_valid(rhs, n, k, True)[1]
        self.put(f"for (int _e = threadIdx.x; _e < {m * n}; _e += {self.threads}) {{")
        self.put(f"  const int _i0 = _e / {n}, _i1 = _e % {n};")
        self.put(f"  {valid}[_e] = {valid}[_e] & _kok & ({rows('_i0')}) & ({cols('_i1')});")
        self.put("}")
        self.depth -= 1
        self.put("}")
        self.barrier()
        return True

    @staticmethod
    def mentions(e: ir.Expr, name: str) -> bool:
        return (isinstance(e, (ir.Var, ir.Param)) and e.name == name) or any(
            Emitter.mentions(child, name) for child in ir.children(e))

    @staticmethod
    def mfma_bits(form: "MfmaForm", x: str) -> str:
        """An element as the bits of a matrix-core operand."""
        return {"f16": f"__builtin_bit_cast(unsigned short, (_Float16){x})",
                "bf16": f"(unsigned short)(__float_as_uint({x}) >> 16)",
                "fp8": f"(unsigned char){x}",  # the e4m3 code as the tile holds it
                "i8": f"(signed char){x}"}[form.name]

    def stmt_If(self, s: ir.If) -> None:
        if self.pending:
            self.barrier()
        self.put(f"if ({self.scalar(s.cond)}) {{")
        self.depth += 1
        self.body(s.then)
        if self.pending:
            self.barrier()
        self.depth -= 1
        self.put("} else {")
        self.depth += 1
        self.body(s.orelse)
        if self.pending:
            self.barrier()
        self.depth -= 1
        self.put("}")

    def stmt_Assign(self, s: ir.Assign) -> None:
        self.put(f"const {ctype(s.var.dtype)} {user(s.var.name)} = {self.scalar(s.value)};")

    def scalar(self, e: ir.Expr) -> str:
        match e:
            case ir.Const(value=v):
                if e.dtype == BOOL:
                    return "1" if v else "0"
                if e.dtype.is_float or e.dtype == PY_FLOAT:
                    return f"(({ctype(e.dtype)}){float(v)!r})"
                return f"(({ctype(e.dtype)}){int(v)}LL)"
            case ir.Var(name=n) | ir.Param(name=n):
                return user(n)
            case ir.Dim(tensor=t, axis=a):
                return dim(t.name, a)
            case ir.BlockIndex(axis=a):
                return f"b{a}"
            case ir.Cast(operand=o):
                return self.cast(self.scalar(o), o.dtype, e.dtype)
            case ir.Unary(op=ir.Op.NEG, operand=o):
                return f"(-{self.scalar(o)})"
            case ir.Binary(op=op, lhs=a, rhs=b):
                symbol = {ir.Op.AND: "&&", ir.Op.OR: "||"}.get(op, op.value)
                return f"({self.scalar(a)} {symbol} {self.scalar(b)})"
        raise LoweringError(f"scalar {type(e).__name__} is not lowered")

    def cast(self, text: str, src: Dtype, dst: Dtype) -> str:
        if src == dst:
            return text
        if src.is_narrow:
            text = f"k8dec({text})"
        if dst.is_narrow:
            return f"k8enc((float)({text}))"
        if dst == BF16:
            return f"kb16((float)({text}))"
        if dst == BOOL:
            return f"(({text}) != 0)"
        return f"(({ctype(dst)})({text}))"

    def rounded(self, text: str, dtype: Dtype) -> str:
        return f"kb16({text})" if dtype == BF16 else f"({ctype(dtype)})({text})"


def emit(kernel: ir.Kernel, entry: str, overlapping: bool = False, blocks: int = 1) -> tuple[str, int]:
    """HIP source of `kernel` with the entry point `entry`, and the global scratch bytes each block needs (0 when
    its tiles fit in LDS; otherwise the kernel takes a trailing `_scratch` pointer to blocks x that many bytes).
    `overlapping`: for launches in which a tensor the program stores to shares memory with another one; `blocks`: of
    the launch's x axis, which only the threads of a block depend on."""
    return Emitter(kernel, entry, overlapping, blocks).emit()
