"""krn_softmax_rows: a NaN makes its whole row NaN wherever it lies, also among -infinity in a thread, a half wave or a
wave that holds no other value, while the finite values of the row lie in other lanes. One, four, eight and sixteen
waves a row, and rows longer than the registers hold."""

import numpy as np
import pytest

from krn_amd import T
from krn_amd.dtypes import BF16, F16, F32
from krn_amd.runtime import library
from oracle.numerics import bf16_words

pytestmark = pytest.mark.gpu

KIND = {F32: T.f32, F16: T.f16, BF16: T.bf16}


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("width", [40, 511, 1500, 4000, 6000, 16000, 20001, 40001, 70001, 140000])
def test_a_nan_among_minus_infinity_reaches_every_element_of_its_row(device, dtype, width):
    rng = np.random.default_rng(width)
    rows = 96
    x = np.full((rows, width), -np.inf, np.float32)
    finite = [0, 3, width // 3, width - 1]  # one or two lanes of a wave have a value
    x[:, finite] = rng.standard_normal((rows, len(finite)))
    x[: rows // 2, finite[1:]] = -np.inf
    at = np.setdiff1d(np.linspace(1, width - 2, rows).astype(int), finite)
    x[np.arange(len(at)), at] = np.nan
    for first in (0, 1):  # row 0 aligned, and every row one element further
        words = {F32: lambda v: v, F16: lambda v: v.astype(np.float16), BF16: bf16_words}[dtype](x)
        padded = np.concatenate([np.zeros(first, words.dtype), words.ravel()])
        source = device.to_device(padded, KIND[dtype])
        out = device.to_device(np.zeros_like(padded), KIND[dtype])
        skip = first * padded.itemsize
        library.softmax_rows(dtype, source.pointer + skip, out.pointer + skip, rows, width, width, width,
                             device.default_stream.handle)
        got = out.to_host()[first:].reshape(rows, width)
        nan = (got & 0x7FFF) > 0x7F80 if dtype == BF16 else np.isnan(got)
        missed = [(row, int((~nan[row]).sum())) for row in range(len(at)) if not nan[row].all()]
        assert not missed, f"rows that keep elements that are not NaN: {missed[:8]}"
        assert not nan[len(at):].any()
