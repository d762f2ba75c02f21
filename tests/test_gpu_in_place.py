"""Calls whose result is written over an operand: a product over A or B, attention over its keys or values. The result is
the one of separate tensors: products of small integers are exact in every order, attention is held to a float64
softmax with the tolerance of the other attention tests (f16 3e-3)."""

import math

import numpy as np
import pytest

from krn_amd import Blocks, T
from krn_amd.compiler import cdna4
from krn_amd.compiler.capture import capture
from krn_amd.dtypes import BF16, F16
from krn_amd.lib import lib
from krn_amd.runtime import hip, library
from oracle.numerics import bf16_values, bf16_words
from tests.conftest import KERNELS
from tests.kernels import tile_programs as programs
from tests.test_gpu_attention_split import reference


@pytest.mark.gpu
@pytest.mark.parametrize("over", ["a", "b"])
# A as large as the result (N = K): one tile column, several, whole and partial slices, unaligned rows; square for B
@pytest.mark.parametrize("m,n", [(5, 5), (64, 64), (100, 100), (128, 128), (256, 256), (333, 333), (700, 128), (1000, 104),
                                 (300, 9), (2048, 64)])
def test_matmul_over_an_operand(device, over, m, n):
    if over == "b":
        m = n  # B is K x N, the result M x N
    rng = np.random.default_rng(m + n)
    a, b = rng.integers(-2, 3, (m, n)).astype(np.float16), rng.integers(-2, 3, (n, n)).astype(np.float16)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float16)
    for _ in range(3):
        x = {"a": device.to_device(a), "b": device.to_device(b)}
        lib.matmul(x["a"], x["b"], out=x[over], library="ours")
        np.testing.assert_array_equal(x[over].to_host(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(128, 128), (333, 128), (100, 100)])
def test_a_linear_layer_over_its_input(device, m, n):
    rng = np.random.default_rng(m)
    a, b = (rng.integers(-1, 2, shape).astype(np.float32) for shape in ((m, n), (n, n)))  # sums that bf16 holds
    x = device.to_device(bf16_words(a), T.bf16)
    programs.gemm_nt[programs.Tiling(bm=64, bn=64, bk=32)](x, device.to_device(bf16_words(b), T.bf16), x)
    np.testing.assert_array_equal(bf16_values(x.to_host()), a @ b.T)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("over", ["q", "k", "v"])
@pytest.mark.parametrize("bh,s", [(16, 200), (4, 256), (64, 33), (3, 31), (40, 100)])
def test_attention_over_its_inputs(device, over, bh, s, d):
    rng = np.random.default_rng(s + d)
    words = {name: rng.standard_normal((bh, s, d)).astype(np.float16) for name in "qkv"}
    scale = math.log2(math.e) / math.sqrt(d)
    want = reference(*(w.astype(np.float64) for w in words.values()), scale, False)
    tensors = {name: device.to_device(w) for name, w in words.items()}
    need = library.attention_workspace(bh, s, s, d, False)
    scratch = device.empty(T.u8, max(need, 1))
    library.attention_call(F16, *(t.pointer for t in tensors.values()), tensors[over].pointer, bh, s, s, d, scale, False,
                           need)(scratch.pointer if need else 0, device.default_stream.handle)
    np.testing.assert_allclose(tensors[over].to_host().astype(np.float64), want, atol=3e-3)


@pytest.mark.parametrize("c,in_place", [(1 << 20, True), ((1 << 20) + 2 * 512 * 128 - 2, True), (1 << 21, True),
                                        ((1 << 20) + 2 * 512 * 128, False), (1 << 24, False)])
def test_a_launch_over_an_operand_asks_for_the_planes(monkeypatch, c, in_place):
    """A result that shares memory with an operand gets the workspace of two K parts, so that it is written after both
    operands have been read; other launches get what the product alone needs."""
    asked = []
    monkeypatch.setattr(library, "gemm_workspace", lambda *a: 0)
    monkeypatch.setattr(library, "gemm_workspace_in_place", lambda m, n: 2 * m * n * 4)
    monkeypatch.setattr(library, "gemm_call", lambda *a: asked.append(a[-1]) or (lambda workspace, stream: None))
    monkeypatch.setattr(library, "gemm_nt_call", lambda *a: asked.append(0) or (lambda stream: None))
    kernel = capture(KERNELS, "gemm_nt", consts={"t": {"bm": 64, "bn": 64, "bk": 32}})
    plan = cdna4.lower(kernel)
    tensor = {"a": ((512, 128), 1 << 20), "b": ((128, 128), 1 << 21), "c": ((512, 128), c)}
    params = {name: hip.HIPTensor(None, pointer, BF16, shape, owner=object()) for name, (shape, pointer) in tensor.items()}
    assert hip.Launch(kernel, plan)._gemm(plan, params, Blocks(2, 8)) is not None
    assert asked == [2 * 512 * 128 * 4 if in_place else 0]
