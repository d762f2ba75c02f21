"""The generic lowering's fused statements, shared reductions and staged products at the places where they can go wrong:
reductions over extents and axes that do not divide the threads, a variable assigned from its own transpose and from a
broadcast of itself, a store to the tensor that is read, tiles that reach past their tensors, and products of every
operand order. Against the C oracle: exact for integer and selecting work, float32 sums within 2 * extent ulps of the
sum of magnitudes (the parts of a shared sum are added in another order)."""

import numpy as np
import pytest

from krn_amd import Blocks
from krn_amd.compiler.capture import capture
from oracle import cbackend
from tests.kernels import generic_programs as programs

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 5), (16, 24), (15, 23), (20, 40)]


def both(device, name, arrays, consts, launch=Blocks(1)):
    from pathlib import Path

    tensors = [device.to_device(a) for a in arrays]
    getattr(programs, name)(programs.Extent(**consts), *tensors, launch=launch)
    copies = [a.copy() for a in arrays]
    cbackend.run(capture(Path(programs.__file__), name, consts={"t": consts}), launch, copies)
    return [t.to_host() for t in tensors], copies


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("rows,cols", [(16, 24), (7, 33), (1, 64), (64, 3)])
def test_reductions_over_both_axes(device, size, rows, cols):
    x = np.random.default_rng(sum(size)).standard_normal(size).astype(np.float32)
    top, total = np.full((size[0], 1), -7, np.float32), np.full((1, size[1]), -7, np.float32)
    got, want = both(device, "reductions", [x, top, total], {"rows": rows, "cols": cols})
    np.testing.assert_array_equal(got[1], want[1])
    bound = np.zeros(size[1])  # per column; nothing past the tile is written
    bound[:cols] = 2 * rows * 2.0**-24 * np.abs(x[:rows, :cols].astype(np.float64)).sum(axis=0)
    assert np.all(np.abs(got[2].astype(np.float64) - want[2]) <= bound)


@pytest.mark.parametrize("size", SIZES)
def test_a_variable_assigned_from_its_own_transpose_and_broadcast(device, size):
    x = np.random.default_rng(sum(size)).integers(-9, 9, size).astype(np.float32)
    y = np.full(size[::-1], -7, np.float32)
    got, want = both(device, "turned", [x, y], {"rows": 16, "cols": 16})
    np.testing.assert_array_equal(got[1], want[1])


@pytest.mark.parametrize("size", [(16, 16), (13, 13)])
def test_a_transposed_store_to_the_tensor_that_is_read(device, size):
    x = np.random.default_rng(1).standard_normal(size).astype(np.float32)
    got, want = both(device, "in_place", [x], {"rows": 16, "cols": 16})
    np.testing.assert_array_equal(got[0], want[0])


@pytest.mark.parametrize("m,n,k", [(16, 16, 16), (33, 29, 50), (7, 64, 5), (70, 40, 128)])
@pytest.mark.parametrize("rows,cols", [(16, 16), (12, 20), (5, 7)])
def test_f32_products_of_every_operand_order_are_one_fused_step_per_k(device, m, n, k, rows, cols):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    launch = Blocks(-(-n // cols), -(-m // rows))
    for name, operands in (("product_nn", [a, b]), ("product_nt", [a, np.ascontiguousarray(b.T)]),
                           ("product_scaled", [a, b])):
        c = np.full((m, n), -7, np.float32)
        got, want = both(device, name, [*operands, c], {"rows": rows, "cols": cols}, launch)
        np.testing.assert_array_equal(got[2], want[2])
