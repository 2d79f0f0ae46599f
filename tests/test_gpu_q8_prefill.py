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

from helpers import bits_to_f32, block_scales, linear_f64_full
from mote_amd import ops, workloads as wl
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
