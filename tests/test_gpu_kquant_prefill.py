"""GPU parity of the many-token K-quant tiles (more than 64 tokens, and 17 to
64 where they are the faster ones), at the edges of their tiles, of their K split between wave groups and of the K parts,
judged on every output as the few-token kernels are (test_gpu_kquant.py):
against the oracle's f64 linear over the oracle-decoded weights.

The tiles' products are exact and summed in f32, so besides the tolerance of
the few-token tests each shape is held to the error of that summation: K
additions that round a partial sum of about sqrt(K) max|w| max|x| by 2^-24 each,
independently, come to K 2^-24 max|w| max|x|; four times that is allowed.
"""

from __future__ import annotations

import functools

import numpy as np
import pytest

from helpers import bits_to_f32
from mote_amd import ops, workloads as wl
from mote_amd.device import DeviceBuffer, Stream
from mote_amd.hip_runtime import HipRuntime
from test_gpu_kquant import FORMATS, _blocks, _check, _fmt, _judge, _run

pytestmark = pytest.mark.gpu

SHAPES = [
    # (M, N, K), each on the tile that the linear picks (64 rows but for the
    # last; test_every_tile runs the others): one super-block (the second wave
    # group idle), odd counts of blocks (uneven groups), one row past and short of
    # a tile on both sides, a single column, several tiles, K parts (few tiles,
    # long K) with a short last part
    (65, 1, 256),
    (128, 128, 512),
    (129, 127, 768),
    (66, 129, 2304),
    (200, 33, 1280),
    (257, 300, 4096),
    (70, 40, 14336),
    (130, 60, 9472),
    # up to 64 tokens, wide enough to come here
    (33, 3001, 768),
    (48, 4100, 512),
    (64, 7000, 1280),
    # 96-row tiles
    (300, 14336, 256),
]
# Every tile form on the same problems: 1, 2, 3, 5 and 9 super-blocks (an idle
# second group, uneven groups, parts of one and short last parts), rows and columns one past
# and short of a tile
TILE_SHAPES = [(1, 1, 256), (33, 127, 512), (129, 128, 768), (257, 200, 1280), (95, 129, 2304)]
# (format, (M, N, K), tile rows, K parts; 0: without scratch)
TILES = [
    (name, shape, rows, parts)
    for name in ("q4_k", "q6_k") for shape in TILE_SHAPES for rows in (64, 96, 128) for parts in (0, 1, 2, 3, 5)
    if parts <= shape[2] // 256 and (name, rows, parts) != ("q4_k", 128, 0)
]


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_linear_many_tokens(stream, oracle, name, m, n, k):
    seed = 800 + m * 3 + n + k
    w = (wl.q4_k_weights if name == "q4_k" else wl.q6_k_weights)(seed, n, k)
    x = wl.normal_f16(wl.seed_for(41, seed), m * k)
    y64, max_w, max_x = _judge(oracle, name, x, w, m, n, k)
    y = _run(stream, name, x, w, m, n, k)
    _check(y, y64, k, max_w, max_x, what=f"{name} {m}x{n}x{k} f32")
    bound = 4.0 * k * 2.0 ** -24 * max_w * max_x
    assert float(np.abs(y - y64).max()) <= bound, f"{name} {m}x{n}x{k}: past f32 summation of exact products"
    y16 = _run(stream, name, x, w, m, n, k, f16_out=True)
    _check(y16, y64, k, max_w, max_x, 2.0 ** -11, what=f"{name} {m}x{n}x{k} f16")


@functools.lru_cache(maxsize=4)
def _problem(name, m, n, k, special):
    """Weights, activations and what the oracle says of them."""
    import oracle

    w = (wl.q4_k_weights if name == "q4_k" else wl.q6_k_weights)(860 + n, n, k)
    x = wl.normal_f16(wl.seed_for(46, m + k), m * k).copy()
    if special:
        rng = np.random.default_rng(47 + k)
        at = rng.choice(x.size, max(1, m // 4), replace=False)
        x[at] = rng.choice(np.array([0x7C00, 0xFC00, 0x7E00], dtype=np.uint16), at.size)
        blocks = w.reshape(n * k // 256, -1).copy()
        bad = rng.random(len(blocks)) < 0.02
        d = 0 if name == "q4_k" else 208
        blocks[bad, d:d + 2] = np.array([0x00, 0x7C], dtype=np.uint8)  # infinite
        w = blocks.reshape(-1)
    x32, fmt = bits_to_f32(x), _fmt(oracle, name)
    y64 = oracle.kquant_linear_f64(x32, w, fmt, m, n, k)
    max_w = np.abs(oracle.dequantize_kquant_row(w, fmt, n * k))
    return w, x, y64, float(max_w[np.isfinite(max_w)].max()), float(np.abs(x32)[np.isfinite(x32)].max())


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("name,shape,rows,parts", TILES)
def test_every_tile(stream, name, shape, special, rows, parts):
    m, n, k = shape
    w, x, y64, max_w, max_x = _problem(name, m, n, k, special)
    xb, wb, yb = DeviceBuffer.from_array(x), DeviceBuffer.from_array(w), DeviceBuffer(m * n * 4)
    yb.upload(np.full(yb.nbytes, 0xA5, dtype=np.uint8))
    ops.prompt_linear_tiles(name, xb.ptr, wb.ptr, yb.ptr, m, n, k, stream, rows, parts)
    stream.synchronize()
    y = yb.download(np.float32).reshape(y64.shape).astype(np.float64)
    for cls in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(cls(y), cls(y64)), f"{cls.__name__} positions differ"
    ok = np.isfinite(y64)
    bound = 4.0 * k * 2.0 ** -24 * max_w * max_x
    assert float(np.abs(y[ok] - y64[ok]).max(initial=0.0)) <= bound, "past f32 summation of exact products"


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,k", [(80, 1536), (72, 8192)])
def test_many_tokens_every_finite_scale(stream, oracle, name, m, k):
    n = 40
    w = _blocks(name, 820 + k, n * k // 256)
    x = wl.normal_f16(wl.seed_for(42, 1), m * k)
    y64, max_w, max_x = _judge(oracle, name, x, w, m, n, k)
    assert np.isfinite(y64).all()
    _check(_run(stream, name, x, w, m, n, k), y64, k, max_w, max_x, what=f"{name} wide scales")


@pytest.mark.parametrize("name", list(FORMATS))
def test_many_tokens_non_finite(stream, oracle, name):
    """Infinite and NaN activations, and activations whose sub-block sums pass
    binary16's range: the outputs are the definition's."""
    m, n, k = 70, 24, 12288
    w = (wl.q4_k_weights if name == "q4_k" else wl.q6_k_weights)(830, n, k)
    x = wl.normal_f16(wl.seed_for(43, m), m * k).copy()
    x[5000] = 0x7C00
    x[(m - 1) * k + 9000] = 0xFC00
    x[k + 100] = 0x7E00
    x[2 * k + 64:2 * k + 96] = 0x7000  # token 2: 32 activations of 8192
    y64 = oracle.kquant_linear_f64(bits_to_f32(x), w, _fmt(oracle, name), m, n, k)
    max_w = float(np.abs(oracle.dequantize_kquant_row(w, _fmt(oracle, name), n * k)).max())
    y = _run(stream, name, x, w, m, n, k)
    for cls in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(cls(y), cls(y64)), f"{name}: {cls.__name__} positions differ"
    ok = np.isfinite(y64)
    _check(y[ok], y64[ok], k, max_w, 8192.0, what=f"{name} finite outputs")


def test_q6_k_many_tokens_at_two_byte_offset(stream, oracle):
    m, n, k = 70, 50, 1280
    w = wl.q6_k_weights(840, n, k)
    x = wl.normal_f16(wl.seed_for(44, 1), m * k)
    y64, max_w, max_x = _judge(oracle, "q6_k", x, w, m, n, k)
    _check(_run(stream, "q6_k", x, w, m, n, k, w_offset=2), y64, k, max_w, max_x, what="q6_k at 2 mod 4")


def test_q4_k_many_tokens_unaligned_weights(stream, oracle):
    """Q4_K weights off the 16-byte grid keep the few-token kernels' route."""
    m, n, k = 66, 20, 512
    w, x = wl.q4_k_weights(851, n, k), wl.normal_f16(wl.seed_for(45, 2), m * k)
    y64, max_w, max_x = _judge(oracle, "q4_k", x, w, m, n, k)
    _check(_run(stream, "q4_k", x, w, m, n, k, w_offset=4), y64, k, max_w, max_x, what="q4_k w unaligned")


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("x_offset", [2, 8])
def test_many_tokens_unaligned_activations(stream, oracle, name, x_offset):
    """Activations off the 16-byte grid keep the few-token kernels' route."""
    m, n, k = 66, 20, 512
    w = (wl.q4_k_weights if name == "q4_k" else wl.q6_k_weights)(850, n, k)
    x = wl.normal_f16(wl.seed_for(45, 1), m * k)
    y64, max_w, max_x = _judge(oracle, name, x, w, m, n, k)
    _check(_run(stream, name, x, w, m, n, k, x_offset=x_offset), y64, k, max_w, max_x, what=f"{name} x unaligned")


def test_long_k_is_no_coarser_than_the_few_token_tiles(stream, oracle):
    """64 tokens, K = 14 336, columns enough for one K part: the many-token tiles
    against the few-token ones, which the same call runs under capture.  Both
    errors are means over 65 536 outputs (0.4 % either way); 3 % is allowed."""
    m, rows, n, k = 64, 1024, 32768, 14336
    w, x = wl.q4_k_weights(860, rows, k), wl.normal_f16(861, m * k)
    y64 = oracle.kquant_linear_f64(bits_to_f32(x), w, oracle.Q4_K, m, rows, k)
    xb, wb = DeviceBuffer.from_array(x), DeviceBuffer.from_array(np.tile(w.reshape(-1), n // rows))
    yb, hip = DeviceBuffer(m * n * 4), HipRuntime()

    def call():
        FORMATS["q4_k"][2](xb.ptr, wb.ptr, yb.ptr, m, n, k, stream)

    def error():
        stream.synchronize()
        y = yb.download(np.float32).reshape(m, n)[:, :rows].astype(np.float64)
        return float(np.linalg.norm(y - y64) / np.linalg.norm(y64))

    call()
    many = error()
    graph = hip.capture(stream, call)
    try:
        hip.launch_graph(graph, stream)
        few = error()
    finally:
        hip.destroy_graph(graph)
    assert many <= 1.03 * few, f"relative error {many:.3e}, few-token tiles {few:.3e}"


@pytest.mark.parametrize("m,n,k", [(70, 300, 4096), (70, 64, 14336), (300, 14336, 512)])
@pytest.mark.parametrize("scratch", [True, False])
def test_q4_k_sums_past_binary16(stream, oracle, m, n, k, scratch):
    """Positive activations whose sub-block sums reach 2^20, and the same over 64:
    the sums are carried in full, so the outputs are the same but for the
    factor, exactly."""
    w = wl.q4_k_weights(870, n, k)
    rng = np.random.default_rng(871)
    x = rng.uniform(100.0, 1000.0, m * k).astype(np.float16)
    large = (x * np.float16(64.0)).view(np.uint16)
    s = stream if scratch else HipRuntime().foreign_stream()
    try:
        y, z = (_run(s, "q4_k", v, w, m, n, k) for v in (x.view(np.uint16), large))
    finally:
        if not scratch:
            s.close()
    rows = [0, 1, 31, 32, 63, 64, m - 1]
    y64, max_w, max_x = _judge(oracle, "q4_k", x.view(np.uint16).reshape(m, k)[rows].reshape(-1), w, len(rows), n, k)
    assert float(np.abs(y.reshape(m, n)[rows] - y64.reshape(len(rows), n)).max()) <= 4.0 * k * 2.0 ** -24 * max_w * max_x
    assert np.array_equal(z, 64.0 * y)


@pytest.mark.parametrize("name", list(FORMATS))
def test_many_tokens_not_finite_time(stream, name):
    """300 tokens of NaN, and of one infinity each: every output is not finite and
    is looked at again over the activations that make it so.  That takes some 50
    times a finite call; over all elements, in one lane each, it took 1000."""
    m, n, k = 300, 4096, 4096
    hip, linear = HipRuntime(), FORMATS[name][2]
    w = DeviceBuffer.from_array((wl.q4_k_weights if name == "q4_k" else wl.q6_k_weights)(880, n, k))
    x = wl.normal_f16(881, m * k)
    nan, inf = np.full_like(x, 0x7E00), x.copy()
    inf[5::k] = 0x7C00
    y = DeviceBuffer(m * n * 4)
    begin, end, times = hip.create(), hip.create(), []
    for bits in (x, nan, inf):
        xb = DeviceBuffer.from_array(bits)
        best = 1e9
        for _ in range(3):
            hip.record(begin, stream)
            linear(xb.ptr, w.ptr, y.ptr, m, n, k, stream)
            hip.record(end, stream)
            best = min(best, hip.elapsed_ms(begin, end))
        times.append(best)
    for e in (begin, end):
        hip.destroy(e)
    assert max(times) <= 200.0 * times[0], f"{name}: finite, NaN, infinite {times} ms"


@pytest.mark.parametrize("name,m,n,k,parts", [("q4_k", 24, 14336, 1024, 1), ("q6_k", 32, 7168, 1024, 2)])
def test_short_k_keeps_the_few_token_tiles(stream, name, m, n, k, parts):
    """Up to 64 tokens with short K the few-token tiles are the faster ones (7.3
    against 10.7 us, 8.0 against 12.9): the linear does not take the many-token
    form that fits best."""
    hip, linear = HipRuntime(), FORMATS[name][2]
    w = DeviceBuffer.from_array((wl.q4_k_weights if name == "q4_k" else wl.q6_k_weights)(890, n, k))
    x, y = DeviceBuffer.from_array(wl.normal_f16(891, m * k)), DeviceBuffer(m * n * 4)
    begin, end = hip.create(), hip.create()

    def time(call):
        best = 1e9
        for _ in range(10):
            hip.record(begin, stream)
            for _ in range(50):
                call()
            hip.record(end, stream)
            best = min(best, hip.elapsed_ms(begin, end))
        return best

    own = time(lambda: linear(x.ptr, w.ptr, y.ptr, m, n, k, stream))
    many = time(lambda: ops.prompt_linear_tiles(name, x.ptr, w.ptr, y.ptr, m, n, k, stream, 64, parts))
    for e in (begin, end):
        hip.destroy(e)
    assert own <= 0.9 * many, f"{name}: {own / 50 * 1e3:.2f} us, many-token tiles {many / 50 * 1e3:.2f}"
