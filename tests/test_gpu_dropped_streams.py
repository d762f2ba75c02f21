"""Streams that a program makes, uses and drops, with launches that may still run: results, the memory they leave and the
handles they use."""

import numpy as np
import pytest

from krn_amd import T
from krn_amd.runtime import hipapi
from tests.kernels import tile_programs as programs

pytestmark = pytest.mark.gpu


def test_a_stream_for_every_product_leaves_its_result_and_no_memory(device):
    m, n, k = 130, 512, 16384  # K parts in the stream's workspace
    rng = np.random.default_rng(4)
    a, w = rng.integers(-127, 128, (m, k), dtype=np.int8), rng.integers(-127, 128, (n, k), dtype=np.int8)
    want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32)
    x, y = device.to_device(a), device.to_device(w)
    results = [device.empty(T.i32, m, n) for _ in range(60)]
    device.sync()
    handles, free = set(), []
    for c in results:
        with device.stream() as stream:
            programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)](x, y, c)
            handles.add(stream.handle)
        free.append(hipapi.memory_free())
    del stream
    device.sync()
    for c in results:
        np.testing.assert_array_equal(c.to_host(), want)
    assert len(handles) < 60 and free[-1] >= free[20] - (64 << 20)


def test_arguments_of_a_dropped_stream_outlive_its_work(device):
    """Operands that only the dropped stream's launches refer to, and memory that is allocated and overwritten right
    after the drop."""
    m, n, k = 130, 96, 8192
    rng = np.random.default_rng(6)
    a, w = rng.integers(-127, 128, (m, k), dtype=np.int8), rng.integers(-127, 128, (n, k), dtype=np.int8)
    want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32)
    for _ in range(10):
        c = device.empty(T.i32, m, n)
        operands = device.to_device(a), device.to_device(w)
        with device.stream():
            for _ in range(20):
                programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)](*operands, c)
        del operands
        scratch = [device.to_device(np.full((n, k), 5, np.int8)) for _ in range(2)]
        device.sync()
        np.testing.assert_array_equal(c.to_host(), want)
        del scratch
