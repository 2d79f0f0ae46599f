"""Prompt linears and the scratch of their K parts and activation sums: a buffer
of its own that only the library's streams have, never used under capture.  So
graphs of prompt calls hold no scratch (they may be replayed at once on several
streams, beside eager calls of their capture stream and after it is gone), a
call on the caller's own stream allocates nothing, and one stream handle that
names another queue in each thread is safe."""

from __future__ import annotations

import threading

import numpy as np
import pytest

import test_gpu_q8_0 as q8
from mote_amd import _ffi, ops, workloads as wl
from mote_amd.device import DeviceBuffer, Stream, memory_info
from mote_amd.hip_runtime import HipRuntime
from test_gpu_kquant import _check, _judge
from test_gpu_q4_0 import check_against_oracle

pytestmark = pytest.mark.gpu

M, N, K = 90, 256, 14336  # few tiles, long K: every format takes K parts on a library stream
LINEAR = {
    "q4_0": ops.quantized_linear_q4_0_f32,
    "q8_0": ops.quantized_linear_q8_0_f32,
    "q4_k": ops.quantized_linear_q4_k_f32,
    "q6_k": ops.quantized_linear_q6_k_f32,
}
WEIGHTS = {"q4_0": wl.q4_0_weights, "q8_0": wl.q8_0_weights, "q4_k": wl.q4_k_weights, "q6_k": wl.q6_k_weights}


class _Calls:
    """Two calls of one format with activations of their own, and a third output."""

    def __init__(self, fmt, m=M, n=N, k=K):
        self.fmt, self.shape = fmt, (m, n, k)
        self.w = WEIGHTS[fmt](900, n, k)
        self.x = [wl.normal_f16(901 + i, m * k) for i in range(2)]
        self.wb = DeviceBuffer.from_array(self.w)
        self.xb = [DeviceBuffer.from_array(x) for x in self.x]
        self.yb = [DeviceBuffer(m * n * 4) for _ in range(3)]

    def call(self, x, y, stream):
        m, n, k = self.shape
        LINEAR[self.fmt](self.xb[x].ptr, self.wb.ptr, self.yb[y].ptr, m, n, k, stream)

    def clear(self):
        for y in self.yb:
            y.upload(np.full(y.nbytes, 0xA5, dtype=np.uint8))

    def result(self, y):
        return self.yb[y].download(np.float32).reshape(self.shape[:2])

    def judge(self, oracle, y, x, what):
        m, n, k = self.shape
        if self.fmt == "q4_0":
            check_against_oracle(oracle, y, self.x[x], self.w, m, n, k, what=what)
        elif self.fmt == "q8_0":
            q8.check(oracle, y, self.x[x], self.w, m, n, k, what=what)
        else:
            y64, max_w, max_x = _judge(oracle, self.fmt, self.x[x], self.w, m, n, k)
            _check(y.astype(np.float64), y64, k, max_w, max_x, what=what)

    def free(self):
        for b in [self.wb, *self.xb, *self.yb]:
            b.free()


@pytest.mark.parametrize("fmt", list(LINEAR))
def test_graphs_of_one_stream_replayed_at_once(oracle, fmt):
    hip, c = HipRuntime(), _Calls(fmt)
    own, others = Stream(), [Stream(), Stream()]
    graphs = [hip.capture(own, lambda i=i: c.call(i, i, own)) for i in range(2)]
    try:
        c.clear()
        for g in graphs:  # alone
            hip.launch_graph(g, others[0])
            others[0].synchronize()
        want = [c.result(i) for i in range(2)]
        for i in range(2):
            c.judge(oracle, want[i], i, f"{fmt} replay")
        for replay in range(20):
            c.clear()
            for g, s in zip(graphs, others):
                hip.launch_graph(g, s)
            c.call(0, 2, own)  # beside an eager call of the capture stream
            for s in (own, *others):
                s.synchronize()
            for i in range(2):
                assert np.array_equal(c.result(i), want[i]), f"{fmt}: replay {replay} of graph {i} differs"
        c.judge(oracle, c.result(2), 0, f"{fmt} eager")
        own.close()
        other = DeviceBuffer(128 << 20)  # memory that the stream's scratch may have been
        other.upload(np.full(other.nbytes, 0x7E, dtype=np.uint8))
        c.clear()
        hip.launch_graph(graphs[0], others[0])
        others[0].synchronize()
        assert np.array_equal(c.result(0), want[0]), f"{fmt}: replay after the capture stream is gone differs"
        assert np.all(other.download(np.uint8) == 0x7E)
        other.free()
    finally:
        for g in graphs:
            hip.destroy_graph(g)
        for s in (own, *others):
            s.close()
        c.free()


@pytest.mark.parametrize("fmt", list(LINEAR))
def test_prompts_beside_a_replayed_decode_graph(fmt):
    """A captured split-K call (16 tokens) holds its capture stream's split-K
    buffer; prompts of that stream leave it alone."""
    hip, c, d = HipRuntime(), _Calls(fmt), _Calls(fmt, 16, 1024, 14336)
    own, other = Stream(), Stream()
    graph = hip.capture(own, lambda: d.call(0, 0, own))
    try:
        hip.launch_graph(graph, other)
        c.call(0, 0, own)
        for s in (own, other):
            s.synchronize()
        want, prompt = d.result(0), c.result(0)
        hip.launch_graph(graph, other)
        other.synchronize()
        assert np.array_equal(d.result(0), want)
        for replay in range(20):
            d.clear()
            hip.launch_graph(graph, other)
            c.call(0, 1, own)
            for s in (own, other):
                s.synchronize()
            assert np.array_equal(d.result(0), want), f"{fmt}: replay {replay} differs"
            assert np.array_equal(c.result(1), prompt), f"{fmt}: prompt {replay} differs"
    finally:
        hip.destroy_graph(graph)
        for s in (own, other):
            s.close()
        for x in (c, d):
            x.free()


@pytest.mark.parametrize("fmt", list(LINEAR))
def test_prompts_on_other_streams_allocate_nothing(oracle, fmt):
    hip, c = HipRuntime(), _Calls(fmt)
    first, second = hip.foreign_stream(), hip.foreign_stream()
    try:
        for s in (first, second):  # loads the kernels; the runtime's cost of a stream
            LINEAR[fmt](c.xb[0].ptr, c.wb.ptr, c.yb[2].ptr, 1, N, K, s)
            s.synchronize()
        c.call(0, 0, first)
        first.synchronize()
        before = memory_info()[0]
        c.call(0, 1, second)
        second.synchronize()
        after = memory_info()[0]
        assert after == before, f"{fmt}: free device memory changed by {before - after} bytes"
        c.judge(oracle, c.result(1), 0, f"{fmt} on a caller's stream")
        assert np.array_equal(c.result(0), c.result(1))
    finally:
        first.close()
        second.close()
        c.free()


class _PerThread:
    handle = 2  # hipStreamPerThread: another queue in each thread

    def synchronize(self):
        _ffi.check(_ffi.lib().mote_hip_stream_synchronize(self.handle), "synchronize stream")


@pytest.mark.parametrize("fmt", list(LINEAR))
def test_threads_on_the_per_thread_stream(oracle, fmt):
    c, s = _Calls(fmt), _PerThread()
    want = []
    for i in range(2):
        c.call(i, i, s)
        s.synchronize()
        want.append(c.result(i))
    for i in range(2):
        c.judge(oracle, want[i], i, f"{fmt} on the per-thread stream")
    start, wrong = threading.Barrier(2), []

    def work(i):
        start.wait()
        for r in range(20):
            c.call(i, i, s)
            s.synchronize()
            if not np.array_equal(c.result(i), want[i]):
                wrong.append((i, r))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    c.free()
    assert not wrong, f"{fmt}: (thread, call) {wrong} differ"


@pytest.mark.parametrize("m,n,k", [(90, 256, 14336), (200, 512, 8192), (130, 300, 4096)])
def test_no_allocation_entry_runs_the_same_prompt_kernels(stream, m, n, k):
    x, w = DeviceBuffer.from_array(wl.normal_f16(910, m * k)), DeviceBuffer.from_array(wl.q4_0_weights(911, n, k))
    ys = []
    for call in (ops.quantized_linear_q4_0_f32, ops.quantized_linear_q4_0_f32_no_alloc):
        y = DeviceBuffer(m * n * 4)
        call(x.ptr, w.ptr, y.ptr, m, n, k, stream)
        stream.synchronize()
        ys.append(y.download(np.uint32))
    assert np.array_equal(ys[0], ys[1])


def test_q4_k_sums_past_the_scratch(stream, oracle):
    """8200 tokens of K = 16 384: their sums take the scratch in two turns.  A
    token's outputs do not depend on its place among the others."""
    rows, m, n, k = 41, 8200, 96, 16384
    w, x = wl.q4_k_weights(920, n, k), wl.normal_f16(921, rows * k)
    y64, max_w, max_x = _judge(oracle, "q4_k", x, w, rows, n, k)
    xb, wb = DeviceBuffer.from_array(np.tile(x, m // rows)), DeviceBuffer.from_array(w)
    yb = DeviceBuffer(m * n * 4)
    yb.upload(np.full(yb.nbytes, 0xA5, dtype=np.uint8))
    ops.quantized_linear_q4_k_f32(xb.ptr, wb.ptr, yb.ptr, m, n, k, stream)
    stream.synchronize()
    y = yb.download(np.float32).reshape(m // rows, rows, n)
    _check(y[0].astype(np.float64), y64, k, max_w, max_x, what="first tokens")
    assert np.array_equal(y, np.broadcast_to(y[0], y.shape))
