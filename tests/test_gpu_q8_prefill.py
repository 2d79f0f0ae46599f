"""The exact-integer Q8_0 prefill tiles (q8_0_prefill_ring.hpp), reached through
the multi-pair Q8_0 variants where K is a multiple of 256 and the operands are
16-byte aligned, and the tiles that serve the other calls of the same variants:
every output judged against the oracle, as in test_gpu_q8_0.py or, where the
exact tiles run, by the error of an f32 sum of exact products (K
additions that round a partial sum of about sqrt(K) max|w| max|x| by 2^-24 each,
independently, come to K 2^-24 max|w| max|x|; four times that is allowed)."""

from __future__ import annotations

import numpy as np
import pytest

from helpers import bits_to_f32, block_scales, linear_f64_full, linear_tolerance, wide_q8_0_weights
from mote_amd import ops, workloads as wl
from mote_amd.device import DeviceBuffer
from mote_amd.hip_runtime import HipRuntime
from test_gpu_q8_0 import check, normal_x, run, weights

pytestmark = pytest.mark.gpu

EXACT = [
    # (M, N, K): one super-pair (the second half of K idle), uneven halves, tiles
    # of 64, 96 and 128 rows with one row more and less, one column, K parts
    (65, 1, 256),
    (97, 129, 768),
    (129, 127, 1280),
    (200, 300, 2304),
    (300, 14336, 256),  # 96-row tiles
    (385, 14336, 256),  # 128-row tiles
    (70, 40, 14336),
    (130, 60, 9472),
]
OTHERS = [(70, 40, 128), (70, 50, 640), (130, 33, 1408)]  # K not a multiple of 256


@pytest.mark.parametrize("m,n,k", EXACT)
def test_exact_tiles(stream, oracle, m, n, k):
    d = ops.Q4_0Dispatch()
    d.force("q8_mfma_x32s_m128_n128_w1_k2")
    x, w = normal_x(wl.seed_for(71, m + k), m, k), weights(wl.seed_for(71, n + k), n, k)
    y = run(stream, x, w, m, n, k, dispatch=d)
    max_w = 128.0 * float(np.abs(block_scales(w, n, k, 34)).max())
    y64 = linear_f64_full(oracle, x, w, m, n, k, oracle.Q8_0)
    bound = 4.0 * k * 2.0 ** -24 * max_w * float(np.abs(bits_to_f32(x)).max())
    assert float(np.abs(y - y64).max()) <= bound, f"{m}x{n}x{k}: past f32 summation of exact products"
    y16 = run(stream, x, w, m, n, k, dispatch=d, f16_out=True)
    assert np.all(np.abs(y16 - y64) <= bound + 2.0 ** -11 * np.abs(y64)), f"{m}x{n}x{k} f16"


@pytest.mark.parametrize("variant", ["q8_mfma_x32s_m128_n256_w1_k2", "q8_mfma_x32s_m128_n128_w1_k2"])
@pytest.mark.parametrize("m,n,k", OTHERS)
def test_other_k_keep_the_staging_tiles(stream, oracle, variant, m, n, k):
    d = ops.Q4_0Dispatch()
    d.force(variant)
    x, w = normal_x(wl.seed_for(72, m + k), m, k), weights(wl.seed_for(72, n + k), n, k)
    check(oracle, run(stream, x, w, m, n, k, dispatch=d), x, w, m, n, k, what=f"{variant} {m}x{n}x{k}")


@pytest.mark.parametrize("m,n,k", [(406, 150, 2176), (300, 200, 1152)])
def test_dispatched_ragged_k(stream, oracle, m, n, k):
    """The linear's own choice at K a multiple of 128 only."""
    x, w = normal_x(wl.seed_for(73, m + k), m, k), weights(wl.seed_for(73, n + k), n, k)
    check(oracle, run(stream, x, w, m, n, k), x, w, m, n, k, what=f"{m}x{n}x{k}")


@pytest.mark.parametrize("m,n,k", [(70, 100, 1024), (130, 60, 9472)])
@pytest.mark.parametrize("scales", ["full", "special"])
@pytest.mark.parametrize("special_x", [False, True])
def test_exact_tiles_not_finite(stream, oracle, m, n, k, scales, special_x):
    """Infinite and NaN scales and activations, and both: the outputs' NaN and
    infinities are where the f64 judge has them."""
    rng = np.random.default_rng(74 + k)
    w = wide_q8_0_weights(75 + n, n, k, scales)
    if scales == "special":  # few of the blocks, so that not every output is NaN
        keep = wide_q8_0_weights(75 + n, n, k, "full").reshape(-1, 34)
        pick = rng.random(len(keep)) < 0.05
        w = np.where(pick[:, None], w.reshape(-1, 34), keep)
        # blocks of one sign: with x > 0, infinite sums that stay infinite
        w[pick & (rng.random(len(keep)) < 0.5), 2:] = 3
        w = w.reshape(-1)
    x = normal_x(wl.seed_for(76, k), m, k).copy()
    x[: m * k // 2] &= 0x7FFF
    if special_x:
        at = rng.choice(x.size, m // 4, replace=False)
        x[at] = rng.choice(np.array([0x7C00, 0xFC00, 0x7E00], dtype=np.uint16), at.size)
    d = ops.Q4_0Dispatch()
    d.force("q8_mfma_x32s_m128_n128_w1_k2")
    y = run(stream, x, w, m, n, k, dispatch=d)
    y64 = linear_f64_full(oracle, x, w, m, n, k, oracle.Q8_0)
    for cls in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(cls(y), cls(y64)), f"{cls.__name__}: {int(cls(y).sum())} against {int(cls(y64).sum())}"
    if scales == "special":
        assert np.isinf(y64).any() and np.isnan(y64).any()
    scale = np.abs(block_scales(w, n, k, 34))
    max_d, max_x = float(scale[np.isfinite(scale)].max()), np.abs(bits_to_f32(x))
    ok = np.isfinite(y64)
    tol = linear_tolerance(y64, k, max_d, float(max_x[np.isfinite(max_x)].max()))
    assert np.all(np.abs(y[ok] - y64[ok]) <= tol[ok])


def test_not_finite_activations_cost_no_more(stream):
    """300 tokens of NaN, and of one infinity each, against finite ones: the time of
    a call may triple at most (recomputed output by output it grows a
    hundredfold)."""
    m, n, k = 300, 4096, 4096
    hip = HipRuntime()
    w = DeviceBuffer.from_array(weights(wl.seed_for(77, n), n, k))
    x = normal_x(wl.seed_for(77, k), m, k)
    nan, inf = np.full_like(x, 0x7E00), x.copy()
    inf[5::k] = 0x7C00
    y = DeviceBuffer(m * n * 4)
    times = []
    begin, end = hip.create(), hip.create()
    for bits in (x, nan, inf):
        xb = DeviceBuffer.from_array(bits)
        best = 1e9
        for _ in range(4):
            hip.record(begin, stream)
            ops.quantized_linear_q8_0_f32(xb.ptr, w.ptr, y.ptr, m, n, k, stream)
            hip.record(end, stream)
            best = min(best, hip.elapsed_ms(begin, end))
        times.append(best)
    for e in (begin, end):
        hip.destroy(e)
    assert max(times) <= 3.0 * times[0], f"finite, NaN, infinite: {times} ms"


@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (33, 127, 512), (129, 128, 768), (257, 200, 1280), (95, 129, 2304)])
@pytest.mark.parametrize("special", [False, True])
def test_every_tile(stream, oracle, m, n, k, special):
    """64-, 96- and 128-row tiles without scratch and over 1 to 5 K parts."""
    w, x = weights(wl.seed_for(78, n), n, k), normal_x(wl.seed_for(78, k), m, k).copy()
    if special:
        rng = np.random.default_rng(79 + k)
        at = rng.choice(x.size, max(1, m // 4), replace=False)
        x[at] = rng.choice(np.array([0x7C00, 0xFC00, 0x7E00], dtype=np.uint16), at.size)
        blocks = w.reshape(-1, 34).copy()
        blocks[rng.random(len(blocks)) < 0.01, 0:2] = np.array([0x00, 0x7C], dtype=np.uint8)
        w = blocks.reshape(-1)
    y64 = linear_f64_full(oracle, x, w, m, n, k, oracle.Q8_0)
    scale, max_x = np.abs(block_scales(w, n, k, 34)), np.abs(bits_to_f32(x))
    bound = 4.0 * k * 2.0 ** -24 * 128.0 * float(scale[np.isfinite(scale)].max()) * float(max_x[np.isfinite(max_x)].max())
    ok = np.isfinite(y64)
    xb, wb, yb = DeviceBuffer.from_array(x), DeviceBuffer.from_array(w), DeviceBuffer(m * n * 4)
    for rows in (64, 96, 128):
        for parts in (p for p in (0, 1, 2, 3, 5) if p <= k // 256):
            yb.upload(np.full(yb.nbytes, 0xA5, dtype=np.uint8))
            ops.prompt_linear_tiles("q8_0", xb.ptr, wb.ptr, yb.ptr, m, n, k, stream, rows, parts)
            stream.synchronize()
            y = yb.download(np.float32).reshape(y64.shape).astype(np.float64)
            for cls in (np.isnan, np.isposinf, np.isneginf):
                assert np.array_equal(cls(y), cls(y64)), f"{rows} rows, {parts} parts: {cls.__name__} positions differ"
            assert float(np.abs(y[ok] - y64[ok]).max(initial=0.0)) <= bound, f"{rows} rows, {parts} parts"


def test_long_k_takes_128_row_tiles_over_two_parts(stream):
    """128 x 8192 x 11 008: two rows of 64-row tiles over all of K wait for the
    weights (66 us), one row of 128-row tiles over two parts does not (56)."""
    m, n, k = 128, 11008, 8192
    xb = DeviceBuffer.from_array(normal_x(wl.seed_for(80, k), m, k))
    wb = DeviceBuffer.from_array(np.tile(weights(wl.seed_for(80, n), n // 43, k).reshape(-1), 43))
    ys = []
    for call in (
        lambda y: ops.quantized_linear_q8_0_f32(xb.ptr, wb.ptr, y.ptr, m, n, k, stream),
        lambda y: ops.prompt_linear_tiles("q8_0", xb.ptr, wb.ptr, y.ptr, m, n, k, stream, 128, 2),
    ):
        y = DeviceBuffer(m * n * 4)
        call(y)
        stream.synchronize()
        ys.append(y.download(np.uint32))
    assert np.array_equal(ys[0], ys[1])
