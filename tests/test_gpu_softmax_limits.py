"""krn_softmax_rows on both sides of every row length at which the waves of a row or the chunks that they keep change, and
on both sides of the row count that decides for the longest of them. Against a float64 softmax; the columns past a row's
width keep what they held, and the last column holds the row's maximum, so a chunk that is left out shows."""

import numpy as np
import pytest

from krn_amd.dtypes import BF16, F16, F32
from krn_amd.runtime import library
from oracle.numerics import bf16_values, bf16_words

pytestmark = pytest.mark.gpu

# half an ulp of the rounding and the float32 exp and sum; f16 results below 2^-14 are spaced by 2^-24
BOUND = {F32: (2e-5, 1e-30), F16: (1.5e-3, 3e-8), BF16: (8e-3, 1e-30)}
CASES = [(5, chunks) for chunks in (64, 128, 256, 320, 384, 512, 768, 1024, 1280, 1536, 1792, 2048, 2560, 3072)]
CASES += [(rows, chunks) for chunks in (4096, 7168, 8192) for rows in (5, 257)]


@pytest.mark.parametrize("dtype", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,chunks", CASES)
@pytest.mark.parametrize("pad", [0, 3])
def test_both_sides_of_every_limit(device, dtype, rows, chunks, pad):
    for width in (chunks * (4 if dtype == F32 else 8), chunks * (4 if dtype == F32 else 8) + 1):
        x = (np.random.default_rng(width + pad).standard_normal((rows, width + pad)) * 4).astype(np.float32)
        x[:, width - 1] = 24.0
        words = {F32: lambda v: v, F16: lambda v: v.astype(np.float16), BF16: bf16_words}[dtype](x)
        source, out = device.to_device(words, dtype), device.to_device(np.full_like(words, 7), dtype)
        library.softmax_rows(dtype, source.pointer, out.pointer, rows, width, width + pad, width + pad,
                             device.default_stream.handle)
        got = out.to_host()
        assert np.all(got[:, width:] == words.dtype.type(7))
        values, got = ((bf16_values(w) if dtype == BF16 else w).astype(np.float64)[:, :width] for w in (words, got))
        p = np.exp(values - values.max(axis=1, keepdims=True))
        rtol, atol = BOUND[dtype]
        np.testing.assert_allclose(got, p / p.sum(axis=1, keepdims=True), rtol=rtol, atol=atol)
