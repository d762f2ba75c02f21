"""krn_softmax_rows on rows that start at any element and at the widths where its routes change: one wave, four and
sixteen waves per row, rows longer than the registers hold, a last chunk of every length, and few and many rows. Against
a float64 softmax with the bounds of the other softmax tests; nothing past a row's width is written."""

import numpy as np
import pytest

from krn_amd import T
from krn_amd.dtypes import BF16, F16, F32
from krn_amd.runtime import library
from oracle.numerics import bf16_values, bf16_words

pytestmark = pytest.mark.gpu

WIDTHS = [1, 7, 8, 9, 63, 511, 513, 1023, 2049, 4095, 4097, 8191, 16383, 16385, 50001, 65535, 65537, 70001]
BOUND = {F32: (2e-5, 1e-12), F16: (1.5e-3, 3e-8), BF16: (8e-3, 1e-30)}
KIND = {F32: T.f32, F16: T.f16, BF16: T.bf16}


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("pad", [0, 3])
def test_rows_at_any_alignment(device, dtype, width, pad):
    rng = np.random.default_rng(width + pad)
    rows, ld = (5, width + pad)
    x = (rng.standard_normal((rows, ld)) * 4).astype(np.float32)
    words = {F32: lambda v: v, F16: lambda v: v.astype(np.float16), BF16: bf16_words}[dtype](x)
    values = (bf16_values(words) if dtype == BF16 else words).astype(np.float64)[:, :width]
    out = device.to_device(np.full((rows, ld), 7, words.dtype), KIND[dtype])
    source = device.to_device(words, KIND[dtype])
    library.softmax_rows(dtype, source.pointer, out.pointer, rows, width, ld, ld, device.default_stream.handle)
    got = out.to_host()
    assert np.all(got[:, width:] == words.dtype.type(7))
    got = (bf16_values(got) if dtype == BF16 else got).astype(np.float64)[:, :width]
    p = np.exp(values - values.max(axis=1, keepdims=True))
    rtol, atol = BOUND[dtype]
    np.testing.assert_allclose(got, p / p.sum(axis=1, keepdims=True), rtol=rtol, atol=atol)


@pytest.mark.parametrize("width", [300, 3001])
def test_many_rows_take_one_wave_each(device, width):
    rng = np.random.default_rng(width)
    x = (rng.standard_normal((4099, width)) * 4).astype(np.float16)
    y = device.empty(T.f16, *x.shape)
    source = device.to_device(x)
    library.softmax_rows(F16, source.pointer, y.pointer, 4099, width, width, width, device.default_stream.handle)
    v = x.astype(np.float64)
    p = np.exp(v - v.max(axis=1, keepdims=True))
    np.testing.assert_allclose(y.to_host().astype(np.float64), p / p.sum(axis=1, keepdims=True), rtol=1.5e-3, atol=3e-8)


def test_infinities_and_nan_stay_in_their_rows(device):
    x = np.random.default_rng(3).standard_normal((4, 10001)).astype(np.float32)
    x[0, 17], x[1, 9000], x[2, :] = np.nan, np.inf, -np.inf
    x[3, :9000] = -np.inf
    x[2, 40:48] = np.nan  # a whole chunk of them
    y = device.empty(T.f32, *x.shape)
    source = device.to_device(x)
    library.softmax_rows(F32, source.pointer, y.pointer, 4, 10001, 10001, 10001, device.default_stream.handle)
    got = y.to_host()
    assert np.all(np.isnan(got[0])) and np.all(np.isnan(got[2])) and np.isnan(got[1, 9000])
    assert np.all(got[3, :9000] == 0) and abs(got[3].astype(np.float64).sum() - 1) < 1e-5


def test_a_chunk_of_nan_makes_its_row_nan(device):
    x = np.zeros((2, 4096), np.float16)
    x[0, 800:816] = np.nan
    y = device.empty(T.f16, *x.shape)
    source = device.to_device(x)
    library.softmax_rows(F16, source.pointer, y.pointer, 2, 4096, 4096, 4096, device.default_stream.handle)
    got = y.to_host()
    assert np.all(np.isnan(got[0])) and np.all(np.isfinite(got[1]))
