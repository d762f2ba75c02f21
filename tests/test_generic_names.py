"""The generic lowering's own names never meet a program's: loop variables and parameters of any name, used as slice
starts, inside tile expressions and around product loops, against the C oracle. Runs the emitted source on the CPU
(tests/host_threads.py); the arithmetic is one operation per element or one fused step per k, so results are exact."""

import numpy as np
import pytest

from krn_amd import Blocks
from krn_amd.compiler.capture import capture
from oracle import cbackend
from tests import host_threads

PROGRAM = """
from krn_amd import Matrix, T, arange, kernel, where, zeros


@kernel
def scalars(x: Matrix[T.f32], y: Matrix[T.f32], {p}: T.f32) -> None:
    acc = zeros(T.f32, 8, 16)
    for {a} in range(0, 4):
        for {b} in range(0, 3):
            acc = where(arange(16, 1, rank=2) <= {a} + 2 * {b}, acc + x[0:8, 0:16] * {p}, acc)
    y[0:8, 0:16] = acc


@kernel
def starts(x: Matrix[T.f32], y: Matrix[T.f32], {p}: T.i32) -> None:
    for {a} in range(0, x.shape[0], 8):
        for {b} in range(0, x.shape[1], 16):
            acc = x[{a} : {a} + 8, {b} : {b} + 16] + x[{b} : {b} + 8, {a} : {a} + 16]
            y[{a} : {a} + 8, {b} : {b} + 16] = acc + acc.sum(axis=0, keepdims=True).to(T.f32)


@kernel
def product(x: Matrix[T.f32], y: Matrix[T.f32], {p}: T.i32) -> None:
    for {a} in range(0, 2):
        for {b} in range(0, 2):
            for {c} in range(0, 2):
                acc = zeros(T.f32, 8, 16)
                for {d} in range(0, x.shape[1], 8):
                    acc += x[{a} * 8 : {a} * 8 + 8, {d} : {d} + 8] @ x[{d} : {d} + 8, {b} * 16 : {b} * 16 + 16]
                for {d} in range(0, x.shape[1], 16):
                    acc += x[{a} * 8 : {a} * 8 + 8, {d} : {d} + 16] @ x[{d} : {d} + 16, {b} * 16 : {b} * 16 + 16]
                y[{a} * 8 : {a} * 8 + 8, {b} * 16 : {b} * 16 + 16] = acc
"""
NAMES = [("i", "s", "r", "x1", "p"), ("s", "i", "r", "e", "scale"), ("s", "i", "e", "r", "bx"), ("x", "t", "o", "s", "_e"),
         ("i", "i0", "r", "r", "_i0"), ("st", "any", "mf", "k", "kmax"), ("u", "w", "l", "q", "y_n0"),
         ("blk", "m0", "n0", "next", "threadIdx"), ("_s", "_x", "_r", "_i", "_s1"), ("acc", "seen", "y1", "p", "int_"),
         ("c", "j", "g", "kok", "_block")]
ORACLES = ("bx", "_e", "y_n0", "kmax", "_block")  # parameters with names of the oracle's C


@pytest.mark.parametrize("program", ["scalars", "starts", "product"])
@pytest.mark.parametrize("names", NAMES, ids=lambda names: "-".join(names))
def test_programs_whose_names_the_lowering_might_use_itself(tmp_path, names, program):
    loops = [name if name not in ("x", "acc") else name + "_" for name in names[:4]]
    path = tmp_path / "program.py"
    path.write_text(PROGRAM.format(**dict(zip("abcd", loops)), p=names[4]))
    kernel = capture(path, program)
    x = np.random.default_rng(3).integers(-4, 5, (32, 32)).astype(np.float32)
    want = np.full((32, 32), -7, np.float32)
    plain = tmp_path / "plain.py"
    plain.write_text(PROGRAM.format(a="one", b="two", c="three", d="four", p="five"))
    cbackend.run(capture(plain, program), Blocks(1), [x.copy(), want, 3])
    if names[4] not in ORACLES:  # loop variables get a number, parameters keep their name
        named = np.full((32, 32), -7, np.float32)
        cbackend.run(kernel, Blocks(1), [x.copy(), named, 3])
        np.testing.assert_array_equal(named, want)
    for last_first in (False, True):
        got = np.full((32, 32), -7, np.float32)
        host_threads.run(kernel, [x.copy(), got, 3], Blocks(1), last_first)
        np.testing.assert_array_equal(got, want)


def test_the_sources_of_such_programs_compile_for_the_gpu(tmp_path):
    from krn_amd.compiler import hipgen
    from krn_amd.runtime import hip, hipapi

    for index, names in enumerate(NAMES):
        loops = [name if name not in ("x", "acc") else name + "_" for name in names[:4]]
        path = tmp_path / f"program{index}.py"
        path.write_text(PROGRAM.format(**dict(zip("abcd", loops)), p=names[4]))
        for program in ("scalars", "starts", "product"):
            kernel = capture(path, program)
            assert hipapi.rtc().compile(hipgen.emit(kernel, "entry")[0], "entry", hip.HIPRTC_OPTIONS)
