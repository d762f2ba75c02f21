"""The key-split attention kernel (krn_amd/csrc/attention_split.hip): launches of few query rows, whose keys are shared
by the waves of a workgroup and by several workgroups. Against a float64 softmax on the 16-bit operands, with the
tolerances of the other attention tests: P and O each round once to 16 bits (bf16 atol 2e-2, f16 3e-3)."""

import math

import numpy as np
import pytest

from krn_amd import T
from krn_amd.dtypes import BF16, F16
from krn_amd.runtime import library
from oracle.numerics import bf16_values, bf16_words

pytestmark = pytest.mark.gpu

# one query, a few, a whole block, one row more than a block; keys fewer than a tile, one more than a tile, several parts;
# 128 MiB of keys and values (d = 128), read non-temporally
SHAPES = [(1, 1, 1), (2, 1, 33), (3, 5, 333), (8, 1, 16384), (32, 1, 8200), (128, 8, 2000), (2, 33, 31), (4, 100, 1000),
          (16, 300, 300), (5, 31, 4097), (3, 32, 500), (32, 3, 8193)]


def attend(device, dtype, q, k, v, scale, causal, workspace=True):
    (bh, sq, d), sk = q.shape, k.shape[1]
    kind = T.bf16 if dtype == BF16 else T.f16
    tensors = [device.to_device(x, kind) for x in (q, k, v)]
    o = device.to_device(np.full((bh * sq + 1, d), 7, q.dtype), kind)  # one row past the end must stay
    need = library.attention_workspace(bh, sq, sk, d, causal) if workspace else 0
    scratch = device.empty(T.u8, max(need, 1))
    library.attention_call(dtype, *(t.pointer for t in tensors), o.pointer, bh, sq, sk, d, scale, causal, need)(
        scratch.pointer if need else 0, device.default_stream.handle)
    got = o.to_host()
    assert np.all(got[-1] == q.dtype.type(7))
    return got[:-1].reshape(bh, sq, d), need


def reference(q, k, v, scale, causal):
    s = np.einsum("hqd,hkd->hqk", q, k) * (scale * math.log(2))
    if causal:
        s = np.where(np.arange(k.shape[1])[None, None, :] <= np.arange(q.shape[1])[None, :, None], s, -1e30)
    p = np.exp(s - s.max(axis=-1, keepdims=True))
    return np.einsum("hqk,hkd->hqd", p / p.sum(axis=-1, keepdims=True), v)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bh,sq,sk", SHAPES)
def test_few_query_rows_match_a_float64_softmax(device, dtype, d, causal, bh, sq, sk):
    rng = np.random.default_rng(bh + sq + sk + d)
    raw = [rng.standard_normal((bh, n, d)).astype(np.float32) for n in (sq, sk, sk)]
    words = [bf16_words(x) if dtype == BF16 else x.astype(np.float16) for x in raw]
    scale = math.log2(math.e) / math.sqrt(d)
    values = [(bf16_values(w) if dtype == BF16 else w).astype(np.float64) for w in words]
    want = reference(*values, scale, causal)
    for workspace in (True, False):
        got, _ = attend(device, dtype, *words, scale, causal, workspace)
        got = (bf16_values(got) if dtype == BF16 else got).astype(np.float64)
        np.testing.assert_allclose(got, want, atol=2e-2 if dtype == BF16 else 3e-3)


@pytest.mark.parametrize("bh,s", [(32, 512), (33, 512), (48, 320), (48, 333), (32, 768)])
def test_causal_launches_around_two_workgroups_for_every_compute_unit(device, bh, s):
    """On both sides of the estimate's step at 512 workgroups of 32 rows, d = 128, whichever kernel it takes."""
    rng = np.random.default_rng(bh + s)
    words = [rng.standard_normal((bh, s, 128)).astype(np.float16) for _ in range(3)]
    got, _ = attend(device, F16, *words, 0.13, True)
    some = [0, 1, bh // 2, bh - 1]
    want = reference(*(w[some].astype(np.float64) for w in words), 0.13, True)
    np.testing.assert_allclose(got[some].astype(np.float64), want, atol=3e-3)


def test_decoding_shares_a_head_among_workgroups_and_keeps_it_in_one_without_memory():
    assert library.attention_workspace(32, 1, 8192, 128, False) > 0
    assert library.attention_workspace(128, 4096, 4096, 128, True) == 0


@pytest.mark.parametrize("scale", [-0.2, 0.0, 3.0])
def test_scores_that_climb_and_scales_of_either_sign(device, scale):
    """Row maxima that grow from tile to tile (the lazy rescale fires in every wave), negative and zero scales."""
    rng = np.random.default_rng(7)
    bh, sq, sk, d = 3, 4, 2048, 64
    q = np.abs(rng.standard_normal((bh, sq, d))).astype(np.float32)
    k = (rng.standard_normal((bh, sk, d)) * 0.1 + np.linspace(0, 2, sk)[None, :, None]).astype(np.float32)
    v = rng.standard_normal((bh, sk, d)).astype(np.float32)
    words = [bf16_words(x) for x in (q, k, v)]
    got, _ = attend(device, BF16, *words, scale, False)
    want = reference(*(bf16_values(w).astype(np.float64) for w in words), scale, False)
    np.testing.assert_allclose(bf16_values(got).astype(np.float64), want, atol=2e-2)


def test_a_nan_or_infinite_key_reaches_only_the_rows_that_read_it(device):
    bh, sq, sk, d = 2, 2, 600, 128
    rng = np.random.default_rng(9)
    words = [rng.standard_normal((bh, n, d)).astype(np.float16) for n in (sq, sk, sk)]
    words[2][0, 577, 5] = np.nan
    words[2][1, 3, 7] = np.inf
    got, _ = attend(device, F16, *words, 0.1, False)
    assert np.all(np.isnan(got[0, :, 5])) and np.all(np.isposinf(got[1, :, 7]))
    got[0, :, 5] = got[1, :, 7] = 0
    assert np.all(np.isfinite(got))
