"""ctypes bindings of the C ABI of `libkrn_amd.so` (include/krn_amd.h).

Loading fails loudly: a missing library raises `LibraryNotFound`, and every nonzero return raises `KernelError`
with the library's own message. There is no fallback path.
"""

import ctypes
from ctypes import POINTER, c_char_p, c_float, c_int, c_int64, c_void_p
from functools import cache

from krn_amd.dtypes import BF16, F8E4M3, F16, F32, I8, I32, Dtype
from krn_amd.hw import Libraries

# element kinds of the C ABI (enum Kind in krn_amd/csrc/common.h), by the types' names: hashing a type is a Python call
KINDS = {d.name: code for code, d in enumerate((F32, F16, BF16, F8E4M3, I8, I32))}

# epilogue operations of krn_gemm_nt, applied in order with one float32 rounding each
MUL_SCALAR, MUL_ROW, MUL_COL, ADD_SCALAR, ADD_ROW, ADD_COL, RELU, GELU, SILU = range(9)
ACTIVATIONS = {"relu": RELU, "gelu": GELU, "silu": SILU}
MAX_OPS = 4  # the longest epilogue chain krn_gemm_nt takes (struct Epilogue in krn_amd/csrc/gemm.hip)
# element kind of a row/column vector, added to the operation code (float32 is 0)
VECTOR_KINDS = {F32: 0, F16: 16, BF16: 32}


class KernelError(RuntimeError):
    """A launch the gfx950 kernel library refused or failed, with its message."""


@cache
def lib() -> ctypes.CDLL:
    handle = Libraries.load("krn_amd").handle
    handle.krn_amd_last_error.restype = c_char_p
    handle.krn_amd_last_error.argtypes = []
    handle.krn_gemm_nt.restype = c_int
    handle.krn_gemm_nt.argtypes = [
        c_int, c_void_p, c_void_p, c_void_p, c_int, c_int64, c_int64, c_int64, c_int, POINTER(c_int),
        POINTER(c_float), POINTER(c_void_p), c_void_p,
    ]  # fmt: skip
    handle.krn_gemm.restype = c_int
    handle.krn_gemm.argtypes = [
        c_int, c_int, c_void_p, c_void_p, c_void_p, c_int, c_int64, c_int64, c_int64, c_int, POINTER(c_int),
        POINTER(c_float), POINTER(c_void_p), c_void_p, c_int64, c_void_p,
    ]  # fmt: skip
    handle.krn_gemm_workspace.restype = c_int64
    handle.krn_gemm_workspace.argtypes = [c_int, c_int, c_void_p, c_void_p, c_int64, c_int64, c_int64]
    handle.krn_gemm_workspace_in_place.restype = c_int64
    handle.krn_gemm_workspace_in_place.argtypes = [c_int64, c_int64]
    handle.krn_attention_fwd.restype = c_int
    handle.krn_attention_fwd.argtypes = [
        c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_float, c_int, c_void_p,
    ]  # fmt: skip
    handle.krn_attention_fwd_ws.restype = c_int
    handle.krn_attention_fwd_ws.argtypes = [
        c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_float, c_int, c_void_p,
        c_int64, c_void_p,
    ]  # fmt: skip
    handle.krn_attention_workspace.restype = c_int64
    handle.krn_attention_workspace.argtypes = [c_int64, c_int64, c_int64, c_int64, c_int]
    handle.krn_gemm_nn.restype = c_int
    handle.krn_gemm_nn.argtypes = [
        c_int, c_void_p, c_void_p, c_void_p, c_int, c_int64, c_int64, c_int64, c_int, POINTER(c_int),
        POINTER(c_float), POINTER(c_void_p), c_void_p, c_int64, c_void_p,
    ]  # fmt: skip
    handle.krn_gemm_nn_workspace.restype = c_int64
    handle.krn_gemm_nn_workspace.argtypes = [c_int64, c_int64]
    handle.krn_gemm_nn_workspace_for.restype = c_int64
    handle.krn_gemm_nn_workspace_for.argtypes = [c_void_p, c_void_p, c_int64, c_int64, c_int64]
    handle.krn_gemm_nn_noalloc.restype = c_int
    handle.krn_gemm_nn_noalloc.argtypes = [
        c_int, c_void_p, c_void_p, c_void_p, c_int, c_int64, c_int64, c_int64, c_int, POINTER(c_int),
        POINTER(c_float), POINTER(c_void_p), c_void_p,
    ]  # fmt: skip
    handle.krn_gemm_nn_noalloc_limit.restype = c_int64
    handle.krn_gemm_nn_noalloc_limit.argtypes = []
    handle.krn_transpose16.restype = c_int
    handle.krn_transpose16.argtypes = [c_void_p, c_void_p, c_int64, c_int64, c_void_p]
    handle.krn_softmax_rows.restype = c_int
    handle.krn_softmax_rows.argtypes = [c_int, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_void_p]
    return handle


def check(code: int, what: str) -> None:
    if code != 0:
        raise KernelError(f"{what}: {lib().krn_amd_last_error().decode()} (code {code})")


def kind(dtype: Dtype) -> int:
    try:
        return KINDS[dtype.name]
    except KeyError:
        raise KernelError(f"{dtype} has no kind in the kernel library's C ABI") from None


def gemm_workspace(layout: str, in_dtype: Dtype, a: int, b: int, m: int, n: int, k: int) -> int:
    """Bytes of device workspace `gemm_call` of these arguments uses (`layout` "nt" or "nn")."""
    return lib().krn_gemm_workspace(int(layout == "nn"), kind(in_dtype), a, b, m, n, k)


def gemm_workspace_in_place(m: int, n: int) -> int:
    """Bytes of device workspace with which `gemm_call` may write its result over an operand."""
    return lib().krn_gemm_workspace_in_place(m, n)


def gemm_call(layout: str, in_dtype: Dtype, a: int, b: int, c: int, out_dtype: Dtype, m: int, n: int, k: int,
              ops: list[tuple[int, float, int]], workspace_bytes: int):
    """The product (`layout` "nt": B is N x K, "nn": K x N) as a function of the workspace and the stream, with the
    other arguments marshalled once."""
    codes, scalars, vectors = marshal_ops(ops)
    entry = lib().krn_gemm
    head = (int(layout == "nn"), kind(in_dtype), a, b, c, kind(out_dtype), m, n, k, len(ops), codes, scalars, vectors)

    def call(workspace: int, stream: int) -> None:
        check(entry(*head, workspace, workspace_bytes, stream), "krn_gemm")

    return call


def gemm_nt_call(in_dtype: Dtype, a: int, b: int, c: int, out_dtype: Dtype, m: int, n: int, k: int,
                 ops: list[tuple[int, float, int]]):
    """`gemm_nt` of these arguments as a function of the stream, with the arguments marshalled once."""
    count = len(ops)
    codes = (c_int * max(count, 1))(*(op for op, _, _ in ops))
    scalars = (c_float * max(count, 1))(*(s for _, s, _ in ops))
    vectors = (c_void_p * max(count, 1))(*(v for _, _, v in ops))
    entry = lib().krn_gemm_nt
    head = (kind(in_dtype), a, b, c, kind(out_dtype), m, n, k, count, codes, scalars, vectors)

    def call(stream: int) -> None:
        check(entry(*head, stream), "krn_gemm_nt")

    return call


def marshal_ops(ops: list[tuple[int, float, int]]):
    """The (codes, scalars, vectors) arrays of an epilogue chain for the GEMM entry points."""
    count = len(ops)
    return ((c_int * max(count, 1))(*(op for op, _, _ in ops)), (c_float * max(count, 1))(*(s for _, s, _ in ops)),
            (c_void_p * max(count, 1))(*(v for _, _, v in ops)))


def gemm_nn_workspace(n: int, k: int) -> int:
    """Bytes of device workspace krn_gemm_nn needs for a K x N operand B."""
    return lib().krn_gemm_nn_workspace(n, k)


def gemm_nn_workspace_for(a: int, b: int, m: int, n: int, k: int) -> int:
    """Bytes of workspace this NN product needs: 0 when the kernel reads B as it lies."""
    return lib().krn_gemm_nn_workspace_for(a, b, m, n, k)


def gemm_nt(in_dtype: Dtype, a: int, b: int, c: int, out_dtype: Dtype, m: int, n: int, k: int,
            ops: list[tuple[int, float, int]], stream: int) -> None:
    """C[m, n] = epilogue(sum_k A[m, k] B[n, k]); `ops` are (operation, scalar, vector pointer)."""
    gemm_nt_call(in_dtype, a, b, c, out_dtype, m, n, k, ops)(stream)


def attention_fwd(dtype: Dtype, q: int, k: int, v: int, o: int, bh: int, sq: int, sk: int, d: int, scale: float,
                  causal: bool, stream: int) -> None:
    check(lib().krn_attention_fwd(kind(dtype), q, k, v, o, bh, sq, sk, d, scale, int(causal), stream),
          "krn_attention_fwd")


def attention_workspace(bh: int, sq: int, sk: int, d: int, causal: bool) -> int:
    """Bytes of device workspace `attention_call` of these arguments uses."""
    return lib().krn_attention_workspace(bh, sq, sk, d, int(causal))


def attention_call(dtype: Dtype, q: int, k: int, v: int, o: int, bh: int, sq: int, sk: int, d: int, scale: float,
                   causal: bool, workspace_bytes: int):
    """The attention as a function of the workspace and the stream, with the other arguments marshalled once."""
    entry = lib().krn_attention_fwd_ws
    head = (kind(dtype), q, k, v, o, bh, sq, sk, d, scale, int(causal))

    def call(workspace: int, stream: int) -> None:
        check(entry(*head, workspace, workspace_bytes, stream), "krn_attention_fwd")

    return call


def transpose16(src: int, dst: int, rows: int, cols: int, stream: int) -> None:
    """dst (cols x rows) = src (rows x cols) transposed, 16-bit elements."""
    check(lib().krn_transpose16(src, dst, rows, cols, stream), "krn_transpose16")


def softmax_rows(dtype: Dtype, x: int, y: int, rows: int, width: int, ldx: int, ldy: int, stream: int) -> None:
    """y = softmax over the first `width` columns of each row of x (row strides ldx, ldy in elements)."""
    check(lib().krn_softmax_rows(kind(dtype), x, y, rows, width, ldx, ldy, stream), "krn_softmax_rows")
