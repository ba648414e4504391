"""Split-K scratch under HIP graph capture (MI355X only).

The ops keep one set of split-K counters and partials per stream.  The counters
have to read zero for whichever call on the stream comes next, so nothing that
a capture does may leave them to be cleared by that graph's replays: a stream
whose partials grow while it is captured, and a stream first seen under
capture, are used eagerly and by a graph captured later before the graph that
came first is replayed.  The graphs draw on a memory pool holding 0xFF bytes,
so counters taken from it uncleared would show.  Every result must equal the
call on the default stream bit for bit (same plan, fixed summation order).
"""
from __future__ import annotations

import contextlib
import ctypes
import os

import pytest
import torch

import rhinoforge_amd as rf
from rhinoforge_amd import capi

pytestmark = pytest.mark.gpu
DEV = "cuda"


@contextlib.contextmanager
def _new_stream():
    """A stream whose handle no earlier call has used (torch's own streams come
    from a fixed pool); non-blocking, as torch's are."""
    hip = ctypes.CDLL(os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so"))
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0
    try:
        yield torch.cuda.ExternalStream(handle.value)
    finally:
        assert hip.hipStreamSynchronize(handle) == 0
        assert hip.hipStreamDestroy(handle) == 0


def _poisoned_pool(stream, nbytes):
    """A graph whose memory pool has one free block of `nbytes`, all 0xFF."""
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        t = torch.full((nbytes,), 255, dtype=torch.uint8, device=DEV)
        del t
    graph.replay()
    torch.cuda.synchronize()
    return graph


def _int4_gate_up(gs):
    g = torch.Generator(device=DEV).manual_seed(gs + 1)
    n, k = 12288, 4096
    qs = [torch.randint(-8, 8, (n, k), generator=g, device=DEV, dtype=torch.int8) for _ in range(2)]
    shape = (k // gs, n) if gs else (n,)
    ss = [(torch.rand(shape, generator=g, device=DEV) * 1e-2 + 1e-3).half() for _ in range(2)]
    ws = [rf.pack_weight_int4(q) for q in qs]
    xs = {m: torch.randn(m, k, generator=g, device=DEV).half() for m in (1, 41, 48, 64)}
    return xs, lambda x: rf.linear_multi_w4a16(x, ws, ss), lambda m: capi.plan(
        m, [n, n], k, fmt=2 if gs else 1)


def _int8(ms, n, k):
    g = torch.Generator(device=DEV).manual_seed(n + k)
    w = rf.pack_weight(torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8))
    s = (torch.rand(n, generator=g, device=DEV) * 1e-3 + 1e-4).half()
    xs = {m: torch.randn(m, k, generator=g, device=DEV).half() for m in ms}
    return xs, lambda x: [rf.linear(x, w, s)], lambda m: capi.plan(m, [n], k)


# Each capture order grows the partials past the least size (16 MB).
CASES = {
    "int4 gate/up": (lambda: _int4_gate_up(0), (48, 64, 41)),
    "int4 gate/up gs 32": (lambda: _int4_gate_up(32), (48, 64, 41)),
    "int8 4096 x 8192": (lambda: _int8((1, 500, 600), 4096, 8192), (600, 500)),
}


def _same(got, want, what):
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert torch.equal(a, b), what


@pytest.mark.parametrize("name", CASES)
def test_partials_that_grow_under_capture(name):
    make, order = CASES[name]
    xs, call, plan = make()
    print(f"capture scratch: {name}, captured at M {order}", flush=True)
    plans = {m: plan(m) for m in order}
    assert all(p["splits"] > 1 for p in plans.values()), plans
    assert max(p["workspace_bytes"] for p in plans.values()) > 16 << 20, plans
    want = {m: [y.clone() for y in call(xs[m])] for m in order}
    torch.cuda.synchronize()
    with _new_stream() as stream:
        pool = _poisoned_pool(stream, 96 << 20)
        with torch.cuda.stream(stream):
            call(xs[1])                        # the warm-up: scratch at its least size
        torch.cuda.synchronize()
        graphs, outs = {}, {}
        for m in order:
            graphs[m] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graphs[m], pool=pool.pool(), stream=stream):
                outs[m] = call(xs[m])
        with torch.cuda.stream(stream):        # before any replay
            eager = {m: [y.clone() for y in call(xs[m])] for m in order}
        torch.cuda.synchronize()
        for m in order:
            _same(eager[m], want[m], f"eager M={m} before the first replay")
        for rep in range(3):
            for m in reversed(order):          # the last captured is replayed first
                for y in outs[m]:
                    y.zero_()
                torch.cuda.synchronize()
                with torch.cuda.stream(stream):
                    graphs[m].replay()
                torch.cuda.synchronize()
                _same(outs[m], want[m], f"replay {rep} M={m}")
                with torch.cuda.stream(stream):
                    again = call(xs[m])
                torch.cuda.synchronize()
                _same(again, want[m], f"eager M={m} after replay {rep}")


@pytest.mark.parametrize("m,n,k", [(4, 1024, 16384), (40, 2048, 4096)], ids=["gemv", "gemm"])
def test_a_stream_first_seen_under_capture(m, n, k):
    xs, call, plan = _int8((m,), n, k)
    print(f"capture scratch: first use of a stream M={m} N={n} K={k}", flush=True)
    assert plan(m)["splits"] > 1
    want = [y.clone() for y in call(xs[m])]
    torch.cuda.synchronize()
    with _new_stream() as stream:
        pool = _poisoned_pool(stream, 64 << 20)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, pool=pool.pool(), stream=stream):
            out = call(xs[m])
        with torch.cuda.stream(stream):
            eager = call(xs[m])
        torch.cuda.synchronize()
        _same(eager, want, "eager before the first replay")
        for rep in range(3):
            out[0].zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            _same(out, want, f"replay {rep}")
            with torch.cuda.stream(stream):
                _same([y.clone() for y in call(xs[m])], want, f"eager after replay {rep}")
        torch.cuda.synchronize()


def test_library_counters_per_stream():
    """One region per stream, the same on every call, zero to begin with."""
    lib = capi.load()
    seen = {}
    with _new_stream() as a, _new_stream() as b:
        for s in (a, b, a):
            p = ctypes.c_void_p()
            capi.check(lib.rf_w8a16_stream_counters(ctypes.c_void_p(s.cuda_stream), ctypes.byref(p)),
                       "rf_w8a16_stream_counters")
            assert p.value % 256 == 0 and seen.setdefault(s.cuda_stream, p.value) == p.value
    assert len(set(seen.values())) == 2
    assert abs(list(seen.values())[0] - list(seen.values())[1]) % capi.WS_COUNTER_BYTES == 0
