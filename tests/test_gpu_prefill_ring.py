"""The 128-row Q4_0 prefill tiles' ring body (q4_0_prefill_ring.hip) against the
staging-wave body of the same tiles, which weights off the 16-byte grid take.
Both decode every weight to the same binary16 value and sum exact products in
f32, in another order: K additions that round a partial sum of about sqrt(K)
max|w| max|x| by 2^-24 each, independently, in either body; twice their sum is
allowed.  (Against the oracle both are judged by test_every_mfma_variant and
the wide-scale tests; a forced variant runs its own tiles, here and there.)"""

from __future__ import annotations

import numpy as np
import pytest

from helpers import bits_to_f32, wide_q4_0_weights
from mote_amd import ops, workloads as wl
from mote_amd._ffi import HipError
from mote_amd.device import DeviceBuffer
from test_gpu_q4_0 import check_against_oracle, run_linear, sample_columns

pytestmark = pytest.mark.gpu


def _at(array, offset):
    b = DeviceBuffer(array.nbytes + offset)
    b.upload(array, offset=offset)
    return b, b.ptr + offset


def _both(stream, call, x, weights, m, n, f16_out, other=None):
    """The output with the weights on and off the 16-byte grid (there by `other`)."""
    out = []
    xb, xp = _at(x, 0)
    for offset, call in ((0, call), (4, other or call)):
        held = [_at(w, offset) for w in weights]
        yb = DeviceBuffer(m * n * (2 if f16_out else 4))
        yb.upload(np.full(yb.nbytes, 0xA5, dtype=np.uint8))
        call(xp, [p for _, p in held], yb.ptr)
        stream.synchronize()
        y = yb.download(np.uint16 if f16_out else np.float32)
        out.append((bits_to_f32(y) if f16_out else y).astype(np.float64))
    return out


SHAPES = [
    # (M, N, K): one super-pair (the second half of K idle), uneven halves, one
    # row past and short of a tile on both sides, one column, several tiles
    (128, 256, 256),
    (129, 255, 768),
    (65, 1, 512),
    (127, 129, 2816),
    (300, 513, 1024),
]


@pytest.mark.parametrize("variant", ["mfma_x32s_m128_n256_w1_k2", "mfma_x32s_m128_n128_w1_k2"])
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("scales", ["ordinary", "wide"])
def test_ring_matches_staging_body(stream, variant, m, n, k, scales):
    d, staging = ops.Q4_0Dispatch(), ops.Q4_0Dispatch()
    d.force(variant)  # its own tiles, or with "/P" the same over K parts
    staging.force(variant.split("/")[0])
    x = wl.normal_f16(wl.seed_for(61, m + k), m * k)
    w = wl.q4_0_weights(wl.seed_for(61, n + k), n, k) if scales == "ordinary" else wide_q4_0_weights(62 + n, n, k, "full")
    max_d = float(np.abs(w.reshape(-1, 18)[:, 0:2].copy().view(np.float16).astype(np.float64)).max())
    bound = 4.0 * k * 2.0 ** -24 * 8.0 * max_d * float(np.abs(bits_to_f32(x)).max())
    for f16_out in (False, True):
        if f16_out and scales == "wide":
            continue  # past binary16's range
        def call(dispatch):
            return lambda xp, wp, yp: dispatch.linear(xp, wp[0], yp, m, n, k, stream, f16_out=f16_out)

        got, want = _both(stream, call(d), x, [w], m, n, f16_out, call(staging))
        tol = bound + (2.0 ** -10 * np.abs(want) if f16_out else 0.0)
        assert np.all(np.abs(got - want) <= tol), f"{variant} {m}x{n}x{k}: {float(np.abs(got - want).max())} > {bound}"


@pytest.mark.parametrize("variant", ["mfma_x32s_m128_n256_w1_k2", "mfma_x32s_m128_n128_w1_k2"])
@pytest.mark.parametrize("parts", [2, 3, 8])
@pytest.mark.parametrize("m,n,k", [(70, 96, 14336), (130, 257, 9472), (33, 300, 768), (128, 256, 256)])
@pytest.mark.parametrize("scales", ["ordinary", "wide"])
def test_k_parts_match_staging_body(stream, variant, parts, m, n, k, scales):
    """K parts, with a short last part (K = 9472 over 3 and 8), parts of one
    super-pair (the second half idle) and fewer parts than asked for."""
    test_ring_matches_staging_body(stream, f"{variant}/{parts}", m, n, k, scales)


@pytest.mark.parametrize("m,n,k", [(70, 96, 14336), (130, 129, 9472), (33, 257, 11008), (500, 14336, 512)])
def test_dispatched_prompts(stream, oracle, m, n, k):
    """The dispatcher's own choice, K parts among it, against the oracle."""
    x, w = wl.normal_f16(wl.seed_for(64, m + k), m * k), wl.q4_0_weights(wl.seed_for(64, n + k), n, k)
    y = run_linear(stream, x, w, m, n, k)
    check_against_oracle(oracle, y, x, w, m, n, k, columns=sample_columns(n, 64), what=f"{m}x{n}x{k}")


def test_forced_names():
    d = ops.Q4_0Dispatch()
    d.force("mfma_x32s_m128_n256_w1_k2/8")
    assert d.select(512, 14336, 4096) == "mfma_x32s_m128_n256_w1_k2"
    for name in ("mfma_x32s_m128_n256_w1_k2/1", "mfma_x32s_m128_n256_w1_k2/9", "mfma_x32s_m128_n256_w1_k2/",
                 "mfma_x32s_m128_n256_w1_k2/22", "gateup_mfma_x32s_m128_n128_w1_k2/2", "/2", "q8_generic/2"):
        with pytest.raises(HipError):
            d.force(name)


def test_parts_need_the_ring_tiles(stream):
    """64-row tiles and weights off the 16-byte grid take no K parts."""
    m, n, k = 70, 64, 1024
    xb, wb = DeviceBuffer(m * k * 2), DeviceBuffer(n * k // 32 * 18 + 16)
    yb = DeviceBuffer(m * n * 4)
    d = ops.Q4_0Dispatch()
    for name, offset in (("mfma_x32s_m64_n64_w2_k4/2", 0), ("mfma_x32s_m128_n128_w1_k2/2", 4)):
        d.force(name)
        with pytest.raises(HipError):
            d.linear(xb.ptr, wb.ptr + offset, yb.ptr, m, n, k, stream)


@pytest.mark.parametrize("m,n,k", [(128, 128, 256), (129, 127, 768), (200, 200, 1024)])
def test_gate_up_ring_matches_staging_body(stream, m, n, k):
    d = ops.Q4_0Dispatch()
    d.force("gateup_mfma_x32s_m128_n128_w1_k2")
    x = wl.normal_f16(wl.seed_for(63, m + k), m * k)
    # unit outputs: the SiLU and the product then move an error by at most its
    # slope (1.1) times the other factor
    scale = np.float16(1.0 / (4.6 * np.sqrt(k)))
    wg, wu = (wl.q4_0_weights(wl.seed_for(63, n + i), n, k).reshape(-1, 18).copy() for i in (0, 1))
    for w in (wg, wu):
        w[:, 0:2] = np.array([scale]).view(np.uint8)
    e = 4.0 * k * 2.0 ** -24 * 8.0 * float(scale) * float(np.abs(bits_to_f32(x)).max())
    got, want = _both(stream, lambda xp, wp, yp: d.gate_up_silu(xp, wp[0], wp[1], yp, m, n, k, stream), x,
                      [wg.reshape(-1), wu.reshape(-1)], m, n, False)
    tol = 8.0 * 2.2 * e + 2.0 ** -20 * np.abs(want)  # factors below 8; the device exponential
    assert np.all(np.abs(got - want) <= tol), f"{float((np.abs(got - want) - tol).max())} past the tolerance"


@pytest.mark.parametrize("m,n,k", [(100, 28672, 256), (100, 28672, 1024), (256, 14336, 512)])
def test_short_k_keeps_the_staging_body(stream, m, n, k):
    """With short K the staging-wave body of the 128-row tiles is the faster one
    (65 x 256 x 28 672 7.5 us against 10.2): the linear runs it, so its outputs
    are bit for bit those with weights off the 16-byte grid."""
    x, w = wl.normal_f16(wl.seed_for(65, m + k), m * k), wl.q4_0_weights(wl.seed_for(65, n + k), n, k)
    got, want = _both(stream, lambda xp, wp, yp: ops.quantized_linear_q4_0_f32(xp, wp[0], yp, m, n, k, stream), x, [w],
                      m, n, False)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m,n,k", [(65, 28672, 768), (300, 28672, 512)])
def test_gate_up_short_k_keeps_the_staging_body(stream, m, n, k):
    x = wl.normal_f16(wl.seed_for(66, m + k), m * k)
    w = [wl.q4_0_weights(wl.seed_for(66, n + i), n, k) for i in (0, 1)]
    got, want = _both(stream, lambda xp, wp, yp: ops.q4_0_gate_up_silu_f32(xp, wp[0], wp[1], yp, m, n, k, stream), x, w,
                      m, n, False)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m,n,k", [(65, 4096, 4096), (64, 2048, 3072), (256, 1024, 4096), (80, 4096, 5120)])
def test_k_parts_only_where_they_pay(stream, m, n, k):
    """Shapes whose 64-row tiles in one round are faster than 128-row ones over K
    parts (65 x 4096 x 4096: 17.0 us against 20.0): no parts, so the outputs are
    bit for bit those with weights off the 16-byte grid."""
    x, w = wl.normal_f16(wl.seed_for(67, m + k), m * k), wl.q4_0_weights(wl.seed_for(67, n + k), n, k)
    got, want = _both(stream, lambda xp, wp, yp: ops.quantized_linear_q4_0_f32(xp, wp[0], yp, m, n, k, stream), x, [w],
                      m, n, False)
    assert np.array_equal(got, want)
