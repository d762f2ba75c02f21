"""Scalars in tile expressions keep their own type in the generic lowering, as the C oracle's one-element tiles do: the
emitted source on the CPU."""

from pathlib import Path

import numpy as np
import pytest

from krn_amd import Blocks
from krn_amd.compiler.capture import capture
from oracle import cbackend
from tests import host_threads
from tests.kernels import generic_programs as programs


@pytest.mark.parametrize("n", [3, 63, 64, 100, -100])
def test_a_narrow_scalar_sum_wraps_before_the_tile_reads_it(n):
    kernel = capture(Path(programs.__file__), "below", consts={"t": {"rows": 16, "cols": 16}})
    x = np.arange(-128, 128, dtype=np.int8).reshape(16, 16)
    want, got = np.full((2, 16, 16), -7, np.int8)
    cbackend.run(kernel, Blocks(1), [x, want, n])
    host_threads.run(kernel, [x, got, n], Blocks(1))
    np.testing.assert_array_equal(want, x < np.int8((2 * n + 128) % 256 - 128))
    np.testing.assert_array_equal(got, want)
