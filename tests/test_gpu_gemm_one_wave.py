"""Products whose 128 x 128 tiles fill at most one wave of the chip, on both sides of the line between their two loops (up
to 32 slices of 128 bytes in 16 bits, 18 of int8, 8 or 4 of fp8, and columns that are no multiple of the store blocks),
and products of few rows on both sides of the rule that splits K. int8 is bit-exact; 16-bit and fp8 products are checked
against float64 within 8 * 2^-24 * (k + 8) * |A| |B| plus the rounding of the result."""

import numpy as np
import pytest

from krn_amd import T
from krn_amd.dtypes import BF16
from krn_amd.runtime import library
from oracle.numerics import bf16_values, e4m3_decode, e4m3_encode
from tests.helpers import assert_agrees, bf16_normal
from tests.kernels import tile_programs as programs

pytestmark = pytest.mark.gpu

TILING = programs.Tiling(bm=64, bn=64, bk=64)


@pytest.mark.parametrize("m,n,k", [(1930, 1280, 64), (1930, 1296, 2048), (1930, 1296, 2112), (1930, 1290, 256),
                                   (1301, 1536, 4096), (129, 16384, 192), (2048, 2048, 128)])
def test_bf16(device, m, n, k):
    rng = np.random.default_rng(m + n + k)
    (aw, a), (bw, b) = bf16_normal(rng, (m, k)), bf16_normal(rng, (n, k))
    c = device.empty(T.bf16, m, n)
    programs.gemm_nt[TILING](device.to_device(aw, T.bf16), device.to_device(bw, T.bf16), c)
    assert_agrees(bf16_values(c.to_host()), a, b.T, k, "bf16")


@pytest.mark.parametrize("m,n,slices", [(1931, 1280, 18), (1931, 1280, 19), (1931, 1296, 3), (129, 16384, 1),
                                        (2048, 2048, 2)])
def test_int8(device, m, n, slices):
    rng = np.random.default_rng(m + n + slices)
    a, w = (rng.integers(-127, 128, (rows, slices * 128), dtype=np.int8) for rows in (m, n))
    c = device.empty(T.i32, m, n)
    programs.gemm_i8_i32[TILING](device.to_device(a), device.to_device(w), c)
    np.testing.assert_array_equal(c.to_host(), (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32))


@pytest.mark.parametrize("m,n,slices", [(1920, 1280, 8), (1920, 1280, 9), (1931, 1280, 4), (1931, 1280, 5),
                                        (1920, 1296, 2)])
def test_fp8(device, m, n, slices):
    rng = np.random.default_rng(m + n + slices)
    k = slices * 128
    a, b = (e4m3_encode(rng.standard_normal((rows, k)).astype(np.float32)) for rows in (m, n))
    c = device.empty(T.bf16, m, n)
    programs.gemm_fp8[TILING](device.to_device(a, T.f8e4m3fn), device.to_device(b, T.f8e4m3fn), c, 1.0, 1.0)
    assert_agrees(bf16_values(c.to_host()), e4m3_decode(a), e4m3_decode(b).T, k, "bf16")


@pytest.mark.parametrize("m,n,k,split", [(1, 4096, 16384, False), (12, 4096, 16384, False), (13, 4096, 16384, True),
                                         (8, 4096, 12288, True), (16, 1536, 6144, True), (12, 1536, 4096, False)])
def test_few_rows_split_k_where_that_pays(device, m, n, k, split):
    rng = np.random.default_rng(m + n + k)
    (aw, a), (bw, b) = bf16_normal(rng, (m, k)), bf16_normal(rng, (n, k))
    da, db, c = device.to_device(aw, T.bf16), device.to_device(bw, T.bf16), device.empty(T.bf16, m, n)
    assert (library.gemm_workspace("nt", BF16, da.pointer, db.pointer, m, n, k) > 0) == split
    programs.gemm_nt[TILING](da, db, c)
    assert_agrees(bf16_values(c.to_host()), a, b.T, k, "bf16")
