"""The generic lowering's launches of many blocks: a block of 1024 threads 2^22 times and more would pass a launch's limit
of fewer than 2^32 threads along an axis, so such launches take 256."""

from pathlib import Path
from types import SimpleNamespace

import numpy as np
import pytest

from krn_amd import Blocks
from krn_amd.compiler import hipgen
from krn_amd.compiler.capture import capture
from krn_amd.dtypes import F32
from krn_amd.runtime import hip
from tests.kernels import generic_programs as programs


def doubled():
    return capture(Path(programs.__file__), "doubled", consts={"t": {"rows": 64, "cols": 64}})


def test_the_grid_decides_the_threads_of_a_block(monkeypatch):
    made = []

    made, ran = [], []

    class Program(hip.Program):
        def __init__(self, source, entry, threads, scratch=0):
            made.append(threads)
            assert f"__launch_bounds__({threads})" in source and f"_e += {threads}" in source
            self.scratch, self.threads = 0, threads

        def launch(self, grid, threads, table, stream):
            ran.append((grid[0], threads))

    monkeypatch.setattr(hip, "Program", Program)
    monkeypatch.setattr(hip, "_programs", {})
    launch = hip.Launch(doubled(), None)
    tensors = [hip.HIPTensor(None, p, F32, (64, 64), owner=object()) for p in (1 << 20, 1 << 21)]
    for blocks in (1, 2**22 - 1, 2**22, 2**24 - 1, 7):
        launch._generic(tensors, Blocks(blocks))(SimpleNamespace(handle=0))
    assert ran == [(1, 1024), (2**22 - 1, 1024), (2**22, 256), (2**24 - 1, 256), (7, 1024)] and made == [1024, 256]
    assert all(blocks * threads < 2**32 for blocks, threads in ran)


@pytest.mark.gpu
@pytest.mark.parametrize("blocks", [2**22 - 1, 2**22, 2**24 - 1])
def test_a_launch_of_millions_of_blocks_runs(device, blocks):
    assert hipgen.threads(doubled()) == 1024
    x = np.random.default_rng(0).standard_normal((100, 64)).astype(np.float32)
    y = device.to_device(np.zeros_like(x))
    programs.doubled(programs.Extent(64, 64), device.to_device(x), y, launch=Blocks(blocks))
    np.testing.assert_array_equal(y.to_host(), 2 * x)
