"""The split GEMM kernels (krn_amd/csrc/gemm_split.hip): products of too few tiles for the chip, K split over
workgroups, unaligned rows and B stored K x N, at the edges of tiles, slices and 16-byte pieces. int8 products are
bit-exact in any order of their sums; 16-bit ones are checked against float64 within the accumulation bound of
`agree` (8 * 2^-24 * (k + 8) * |A| |B|) plus the rounding of the result."""

import numpy as np
import pytest

from krn_amd import T
from oracle.numerics import bf16_values, bf16_words
from tests.helpers import assert_agrees
from tests.kernels import tile_programs as programs

pytestmark = pytest.mark.gpu

# rows of 16 bytes and less, one byte more than a slice, ragged tiles, K split (few tiles, long K), unaligned K
INT8 = [(129, 64, 16), (130, 65, 144), (64, 64, 17), (5, 40, 129), (300, 200, 1000), (129, 31, 8192), (257, 129, 4099),
        (1, 33, 8195), (128, 40, 16384), (16, 1024, 8192), (200, 190, 12288), (133, 70, 6160), (513, 512, 2048),
        (640, 900, 4096), (400, 3000, 1040)]


@pytest.mark.parametrize("m,n,k", INT8)
def test_int8_products_of_every_split_and_alignment_are_bit_exact(device, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, w = rng.integers(-127, 128, (m, k), dtype=np.int8), rng.integers(-127, 128, (n, k), dtype=np.int8)
    c = device.empty(T.i32, m, n)
    programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)](device.to_device(a), device.to_device(w), c)
    want = a.astype(np.int64) @ w.astype(np.int64).T
    np.testing.assert_array_equal(c.to_host(), want.astype(np.int32))


@pytest.mark.parametrize("k", [16, 128, 144, 272, 400, 512, 528, 640, 656, 1040])
def test_int8_products_of_one_to_nine_slices_on_128_by_128_tiles_are_bit_exact(device, k):
    rng = np.random.default_rng(k)
    a, w = rng.integers(-127, 128, (2000, k), dtype=np.int8), rng.integers(-127, 128, (2010, k), dtype=np.int8)
    c = device.empty(T.i32, 2000, 2010)
    programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)](device.to_device(a), device.to_device(w), c)
    np.testing.assert_array_equal(c.to_host(), (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32))


@pytest.mark.parametrize("m,n,k", [(129, 130, 8192), (128, 520, 16384), (257, 100, 5000)])
def test_w8a8_scales_apply_once_to_the_sum_of_the_parts(device, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, w = rng.integers(-127, 128, (m, k), dtype=np.int8), rng.integers(-127, 128, (n, k), dtype=np.int8)
    sa = (rng.uniform(0.5, 1.5, (m, 1)) / 127).astype(np.float32)
    sw = (rng.uniform(0.5, 1.5, (1, n)) / 127).astype(np.float32)
    c = device.empty(T.bf16, m, n)
    tiling = programs.Tiling(bm=64, bn=64, bk=64)
    programs.gemm_w8a8[tiling](device.to_device(a), device.to_device(w), device.to_device(sa), device.to_device(sw), c)
    acc = (a.astype(np.int64) @ w.astype(np.int64).T).astype(np.float32)
    np.testing.assert_array_equal(c.to_host(), bf16_words((acc * sa) * sw))


NN = [(1, 8, 8), (70, 9, 64), (65, 136, 200), (100, 333, 13), (129, 64, 63), (64, 65, 129), (130, 1000, 776),
      (300, 301, 777), (200, 264, 8192), (33, 72, 8195), (1024, 1000, 1016), (50, 7, 40), (50, 64, 7)]


@pytest.mark.parametrize("m,n,k", NN)
def test_f16_products_with_b_stored_k_by_n(device, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.uniform(-1, 1, (m, k)).astype(np.float16), rng.uniform(-1, 1, (k, n)).astype(np.float16)
    c = device.empty(T.f32, m, n)
    programs.matmul_f16_f32[programs.Tiling(bm=64, bn=64, bk=32)](device.to_device(a), device.to_device(b), c)
    assert_agrees(c.to_host(), a.astype(np.float32), b.astype(np.float32), k, "f16")


@pytest.mark.parametrize("m,n,k", [(200, 130, 6001), (129, 257, 16384), (140, 33, 9)])
def test_bf16_parts_meet_within_the_accumulation_bound_and_nothing_past_the_result_is_written(device, m, n, k):
    rng = np.random.default_rng(k)
    a, b = (bf16_words(rng.standard_normal(s).astype(np.float32)) for s in ((m, k), (n, k)))
    c = device.to_device(np.full((m + 1, n), -7.0, np.float32))
    view = type(c)(device, c.pointer, c.dtype, (m, n), owner=c)
    programs.gemm_nt_f32[programs.Tiling(bm=64, bn=64, bk=64)](device.to_device(a, T.bf16), device.to_device(b, T.bf16),
                                                               view)
    got = c.to_host()
    assert np.all(got[m] == -7.0)
    x, y = bf16_values(a).astype(np.float64), bf16_values(b).astype(np.float64)
    bound = 8 * 2.0**-24 * (k + 8) * (np.abs(x) @ np.abs(y).T)
    assert np.all(np.abs(got[:m] - x @ y.T) <= bound)


def test_a_split_product_replays_from_a_graph_between_eager_calls_and_on_two_streams(device):
    """The parts' workspace belongs to the stream, and to the graph for a recorded launch."""
    m, n, k = 130, 96, 8192
    rng = np.random.default_rng(5)
    pairs = [(rng.integers(-127, 128, (m, k), dtype=np.int8), rng.integers(-127, 128, (n, k), dtype=np.int8))
             for _ in range(2)]
    wants = [(a.astype(np.int64) @ w.astype(np.int64).T).astype(np.int32) for a, w in pairs]
    inputs = [(device.to_device(a), device.to_device(w), device.empty(T.i32, m, n)) for a, w in pairs]
    launcher = programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)]
    bounds = [launcher.bind(*args) for args in inputs]
    recorded = device.graph(bounds[0])
    other = device.stream()
    for _ in range(4):
        for _, _, c in inputs:
            c.copy_from(np.zeros((m, n), np.int32))
        recorded()
        with other:
            bounds[1]()
        bounds[1]()
        device.sync()
        for (_, _, c), want in zip(inputs, wants):
            np.testing.assert_array_equal(c.to_host(), want)


@pytest.mark.parametrize("kept", [0, 1 << 30])
def test_a_workspace_above_what_a_stream_keeps_is_the_launches_own(device, monkeypatch, kept):
    monkeypatch.setattr("krn_amd.runtime.hip.WORKSPACE_KEPT", kept)
    rng = np.random.default_rng(kept)
    a, w = rng.integers(-127, 128, (129, 8192), dtype=np.int8), rng.integers(-127, 128, (31, 8192), dtype=np.int8)
    want = a.astype(np.int64) @ w.astype(np.int64).T
    with device.stream() as stream:
        c = device.empty(T.i32, 129, 31)
        for _ in range(3):
            programs.gemm_i8_i32[programs.Tiling(bm=64, bn=64, bk=64)](device.to_device(a), device.to_device(w), c)
            np.testing.assert_array_equal(c.to_host(), want.astype(np.int32))
        assert (stream._workspace is None) == (kept == 0)
