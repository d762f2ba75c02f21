"""Tile programs for the generic lowering alone: none is a product, softmax or attention that has a kernel of its own."""

from krn_amd import Const, Matrix, T, block, kernel, struct, where, zeros


@struct
class Extent:
    rows: Const[int] = 16
    cols: Const[int] = 16


@kernel
def reductions(t: Extent, x: Matrix[T.f32], top: Matrix[T.f32], total: Matrix[T.f32]) -> None:
    tile = x[0 : t.rows, 0 : t.cols]
    top[0 : t.rows, 0:1] = tile.max(axis=1, keepdims=True)
    total[0:1, 0 : t.cols] = tile.sum(axis=0, keepdims=True)


@kernel
def turned(t: Extent, x: Matrix[T.f32], y: Matrix[T.f32]) -> None:
    tile = x[0 : t.rows, 0 : t.cols] + 0.0
    tile = tile.transpose()
    tile = tile * 2.0 + tile.transpose().transpose()
    tile = tile + 1.0
    y[0 : t.cols, 0 : t.rows] = tile


@kernel
def in_place(t: Extent, x: Matrix[T.f32]) -> None:
    x[0 : t.cols, 0 : t.rows] = x[0 : t.rows, 0 : t.cols].transpose()


@kernel
def product_nn(t: Extent, a: Matrix[T.f32], b: Matrix[T.f32], c: Matrix[T.f32]) -> None:
    rows, cols = block.tile(t.rows, t.cols)
    acc = zeros(T.f32, t.rows, t.cols)
    for k in range(0, a.shape[1], 8):
        acc += a[rows, k : k + 8] @ b[k : k + 8, cols]
    c[rows, cols] = acc


@kernel
def product_nt(t: Extent, a: Matrix[T.f32], b: Matrix[T.f32], c: Matrix[T.f32]) -> None:
    rows, cols = block.tile(t.rows, t.cols)
    acc = zeros(T.f32, t.rows, t.cols)
    for k in range(0, a.shape[1], 8):
        acc += a[rows, k : k + 8] @ b[cols, k : k + 8].transpose()
    c[rows, cols] = acc


@kernel
def product_scaled(t: Extent, a: Matrix[T.f32], b: Matrix[T.f32], c: Matrix[T.f32]) -> None:
    """An operand that is computed, and an accumulator that the loop also changes."""
    rows, cols = block.tile(t.rows, t.cols)
    acc = zeros(T.f32, t.rows, t.cols)
    for k in range(0, a.shape[1], 8):
        acc *= 0.5
        acc += (a[rows, k : k + 8] * 2.0) @ b[k : k + 8, cols]
    c[rows, cols] = acc


@kernel
def centred(t: Extent, x: Matrix[T.f32], y: Matrix[T.f32]) -> None:
    """Every element of a row reads the row's first one."""
    rows, cols = block.tile(t.rows, t.cols)
    y[rows, 0 : t.cols] = x[rows, 0 : t.cols] - x[rows, 0:1]


@kernel
def moved(t: Extent, x: Matrix[T.f32], y: Matrix[T.f32]) -> None:
    """A load of one statement, stored one column to the left by the next."""
    rows, cols = block.tile(t.rows, t.cols)
    tile = x[rows, 1 : t.cols + 1]
    y[rows, 0 : t.cols] = tile


@kernel
def doubled(t: Extent, x: Matrix[T.f32], y: Matrix[T.f32]) -> None:
    rows = block.tile(t.rows)
    tile = x[rows, 0 : t.cols] * 2.0
    y[rows, 0 : t.cols] = tile


@kernel
def mirrored(t: Extent, x: Matrix[T.f32], y: Matrix[T.f32]) -> None:
    """Two stores, the second of what the first statement's tensor held before."""
    tile = x[0 : t.rows, 0 : t.rows]
    y[0 : t.rows, 0 : t.rows] = tile.transpose() + x[0 : t.rows, 0:1]
    y[0 : t.rows, 0:1] = y[0 : t.rows, 1:2] + x[0 : t.rows, 2:3]


@kernel
def below(t: Extent, x: Matrix[T.i8], y: Matrix[T.i8], n: T.i8) -> None:
    """A scalar sum of a type narrower than C's int: 100 + 100 is -56."""
    y[0 : t.rows, 0 : t.cols] = where(x[0 : t.rows, 0 : t.cols] < n + n, T.i8(1), T.i8(0))
