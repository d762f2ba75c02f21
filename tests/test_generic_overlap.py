"""The generic lowering when one tensor is passed as two parameters, or two that share memory: a block loads what a
statement reads before that statement, or a later one, stores. Exact against the C oracle on the same memory, the
emitted source on the CPU with the lowest thread first and the highest first; and the launch that decides by the
tensors' addresses."""

from pathlib import Path
from types import SimpleNamespace

import numpy as np
import pytest

from krn_amd import Blocks
from krn_amd.compiler.capture import capture
from krn_amd.dtypes import F16, F32
from krn_amd.runtime import hip
from oracle import cbackend
from tests import host_threads
from tests.kernels import generic_programs as programs


def program(name, rows, cols):
    return capture(Path(programs.__file__), name, consts={"t": {"rows": rows, "cols": cols}})


@pytest.mark.parametrize("last_first", [False, True])
@pytest.mark.parametrize("rows,cols", [(16, 512), (16, 24), (5, 7)])
@pytest.mark.parametrize("name", ["centred", "moved", "mirrored"])
def test_a_program_on_one_tensor_as_two_parameters(name, rows, cols, last_first):
    kernel = program(name, rows, cols)
    x = np.random.default_rng(rows + cols).standard_normal((rows, max(cols, rows))).astype(np.float32)
    want, got = x.copy(), x.copy()
    cbackend.run(kernel, Blocks(1), [want, want])
    host_threads.run(kernel, [got, got], Blocks(1), last_first, overlapping=True)
    np.testing.assert_array_equal(got, want)


def tensor(pointer, shape, dtype=F32):
    return hip.HIPTensor(None, pointer, dtype, shape, owner=object())


@pytest.mark.parametrize("x,y,shared", [
    (tensor(4096, (16, 64)), tensor(4096, (16, 64)), True),
    (tensor(4096, (16, 64)), tensor(8192, (16, 64)), False),  # one ends where the other begins
    (tensor(4096, (16, 64)), tensor(8188, (16, 64)), True),
    (tensor(8188, (16, 64)), tensor(4096, (16, 64)), True),
    (tensor(4096, (16, 64)), tensor(6143, (16, 64), F16), True),
    (tensor(4096, (0, 64)), tensor(4096, (16, 64)), False),
])
def test_the_launch_tells_overlapping_tensors_by_their_addresses(monkeypatch, x, y, shared):
    asked = []

    def generic_program(kernel, overlapping=False, blocks=1):
        asked.append(overlapping)
        return SimpleNamespace(scratch=0, threads=256)

    monkeypatch.setattr(hip, "generic_program", generic_program)
    launch = hip.Launch(program("centred", 16, 64), None)
    launch._generic([x, y], Blocks(1))
    launch._generic([tensor(1 << 20, (16, 64)), tensor(1 << 21, (16, 64))], Blocks(1))
    launch._generic([x, y], Blocks(1))
    assert asked == ([True, False] if shared else [False])


def test_two_tensors_that_are_only_read_may_be_one():
    kernel = capture(Path(programs.__file__), "product_nn", consts={"t": {"rows": 16, "cols": 16}})
    launch, a = hip.Launch(kernel, None), tensor(4096, (16, 16))
    assert not launch._overlapping([a, a, tensor(1 << 20, (16, 16))])
    assert launch._overlapping([a, tensor(1 << 20, (16, 16)), a])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(16, 512), (16, 24), (5, 7)])
@pytest.mark.parametrize("name", ["centred", "moved", "mirrored"])
def test_in_place_launches_on_the_gpu(device, name, rows, cols):
    x = np.random.default_rng(rows + cols).standard_normal((rows, max(cols, rows))).astype(np.float32)
    want = x.copy()
    cbackend.run(program(name, rows, cols), Blocks(1), [want, want])
    t = device.to_device(x)
    getattr(programs, name)(programs.Extent(rows, cols), t, t, launch=Blocks(1))
    np.testing.assert_array_equal(t.to_host(), want)
