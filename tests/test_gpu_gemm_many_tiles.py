"""Products of so many rows or columns that small tiles would pass a launch's limit of fewer than 2^32 threads. int8 with
int32 results, exact, checked in rows (columns) of the start, around the limits and of the end; the other rows hold
whatever the memory held."""

import numpy as np
import pytest

from krn_amd import T
from tests.kernels import tile_programs as programs

pytestmark = pytest.mark.gpu


def window(t, first, count):
    row = t.nbytes // t.shape[0]
    return type(t)(t.device, t.pointer + first * row, t.dtype, (count, *t.shape[1:]), owner=t)


@pytest.mark.parametrize("rows,k", [(2**30 + 5, 17), (2**31 + 100, 16)])
@pytest.mark.parametrize("many", ["m", "n"])
def test_products_of_a_billion_rows_or_columns(device, many, rows, k):
    if many == "n" and rows > 2**31:
        pytest.skip("more than 2^24 tiles in one row of tiles of any size")
    rng = np.random.default_rng(k)
    long, short = device.empty(T.i8, rows, k), rng.integers(-127, 128, (1, k), dtype=np.int8)
    starts = [0, 2**29 - 32, rows - 64] + [2**30 - 32, 2**31 - 32] * (rows > 2**31)
    pieces = {first: rng.integers(-127, 128, (64, k), dtype=np.int8) for first in starts}
    for first, piece in pieces.items():
        window(long, first, 64).copy_from(piece)
    c = device.empty(T.i32, *((rows, 1) if many == "m" else (1, rows)))
    operands = (long, device.to_device(short)) if many == "m" else (device.to_device(short), long)
    programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)](*operands, c)
    column = type(c)(device, c.pointer, c.dtype, (rows, 1), owner=c)
    for first, piece in pieces.items():
        want = piece.astype(np.int32) @ short.astype(np.int32).T
        np.testing.assert_array_equal(window(column, first, 64).to_host(), want)
