"""GEMM plans that even out the work per CU (int8): their plan on a 256-CU part
and, on the GPU, every output against the fp64 oracle and the CPU path at
ragged sizes, with K tails and a second call bit-identical to the first.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import rhinoforge_amd as rf
from rhinoforge_amd import capi
from oracle import w4a16 as o4
from oracle import w8a16 as o

# (M, N per projection, K, plan name, K splits)
ROWS = [
    # M 33..64, two splits of 64x256 would make more than one round: unsplit
    (33, [18900, 18948], 1032, "gemm 64x256 3-stage", 1),
    # M 33..64 from 96 tiles of 64x64: the two-K-group forms by estimated time
    (41, [2056, 2056, 2056], 2056, "gemm 64x64 two K groups", 1),
    (64, [8200, 1000, 1032], 5128, "gemm 64x128 two K groups", 3),
    (48, [9728, 9720], 2568, "gemm 64x128 two K groups", 1),
    # M 33..64, K >= 16384 on more than 64 tiles: six splits of 64x128
    (40, [4112], 16392, "gemm 64x128 two K groups", 6),
    # M 65 and more: three splits of a 128-wide form where four do not fit
    (250, [5000], 8200, "gemm 128x128 two K groups", 3),
    (100, [5112], 4104, "gemm 64x128 two K groups", 3),
    # ... at M > 128 from 64 K blocks on
    (256, [1000, 520, 520], 4104, "gemm 64x128 two K groups", 3),
    (250, [5000], 4040, "gemm 128x128 two K groups", 3),
    (250, [5000], 4032, "gemm 64x128 two K groups", 1),
]

# int4 launches of large tiles: (M, N per projection, K, group size, plan, splits)
INT4_ROWS = [
    (640, [5120], 25600, 128, "gemm 128x256 B-in-registers", 5),            # K >= 12288: 128x256 in K splits
    (1000, [2560, 2560], 12352, 32, "gemm 128x256 B-in-registers", 3),      # two projections, K % 128 == 64
    (1300, [4880], 12288, 0, "gemm 128x256 B-in-registers", 2),             # ragged M and N
    (300, [6160], 4160, 64, "gemm 128x128 interleaved", 3),  # three splits of 18 blocks and more
    (500, [5120], 3456, 0, "gemm 128x128 interleaved", 3),   # exactly 18
    (384, [8192], 5120, 128, "gemm 128x128 interleaved", 2),
]

# 128x256 tiles in whole rounds of CUs and a few more, whose K range is split:
# (M, N per projection, K, tiles past the whole rounds, pieces of each)
LAST_TILES = [
    (500, [12800, 38300], 3080, 32, 6),   # 4 x 200 tiles, ragged N, K tail in the last piece
    (1000, [17400, 17408], 4104, 64, 3),  # 8 x 136 tiles, ragged M
    (1300, [24576], 3072, 32, 6),
]


def _id(r):
    return f"{r[0]}x{'_'.join(map(str, r[1]))}x{r[2]}"


@pytest.mark.parametrize("row", ROWS, ids=_id)
def test_plan(row):
    m, ns, k, name, splits = row
    p = capi.plan(m, ns, k, kernel=capi.KERNEL_GEMM, cus=256)
    assert (p["name"], p["splits"]) == (name, splits), p
    assert p["workspace_bytes"] + capi.WS_COUNTER_BYTES <= capi.NOALLOC_SCRATCH_BYTES


@pytest.mark.gpu
@pytest.mark.parametrize("row", ROWS, ids=_id)
def test_parity(row):
    m, ns, k = row[:3]
    print(f"gemm balance M={m} N={ns} K={k}", flush=True)
    x = o.make_activation(o.derive_seed(77, "x", m, k), m, k)
    qs = [o.quantize_linear_per_channel(o.make_weight(o.derive_seed(77, "w", i, n, k), n, k))
          for i, n in enumerate(ns)]
    xd = torch.from_numpy(x).cuda()
    ws = [rf.pack_weight(torch.from_numpy(q).cuda()) for q, _ in qs]
    ss = [torch.from_numpy(s).cuda() for _, s in qs]
    ys = rf.linear_multi(xd, ws, ss, kernel=rf.KERNEL_GEMM)
    again = rf.linear_multi(xd, ws, ss, kernel=rf.KERNEL_GEMM)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[0:3, np.linspace(0, m - 1, 9).astype(int), m - 3:m])
    for (q, s), y, y2 in zip(qs, ys, again):
        assert torch.equal(y, y2)
        rep = o.check_tolerance(y.cpu().numpy()[rows], o.cpu_path(x[rows], q, s),
                                o.oracle_fp64(x[rows], q, s))
        assert rep.ok, str(rep)


@pytest.mark.parametrize("row", LAST_TILES, ids=_id)
def test_last_tiles_plan(row):
    m, ns, k, rem, pieces = row
    tiles = -(-m // 128) * sum(-(-n // 256) for n in ns)
    assert tiles % 256 == rem
    for fmt in (0, 1, 2):
        if fmt and (k % 64 or any(n % 16 for n in ns)):
            continue
        p = capi.plan(m, ns, k, fmt=fmt, cus=256)
        assert (p["name"], p["splits"]) == ("gemm 128x256 B-in-registers", pieces), p
        assert p["workgroups"] == tiles - rem + rem * pieces
        assert p["workspace_bytes"] == rem * pieces * 128 * 256 * 4
        assert p["workspace_bytes"] + capi.WS_COUNTER_BYTES <= capi.NOALLOC_SCRATCH_BYTES


@pytest.mark.gpu
@pytest.mark.parametrize("row", LAST_TILES, ids=_id)
def test_last_tiles_parity(row):
    """Split last tiles, also without the workspace they need (run whole): both
    within the bar, the first bit-identical on a second call."""
    import ctypes
    m, ns, k = row[:3]
    print(f"last tiles M={m} N={ns} K={k}", flush=True)
    x = o.make_activation(o.derive_seed(78, "x", m, k), m, k)
    g = torch.Generator().manual_seed(k)
    qs = [torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8) for n in ns]
    ss = [(torch.rand(n, generator=g) * 1e-3 + 1e-4).half() for n in ns]
    xd = torch.from_numpy(x).cuda()
    ws = [rf.pack_weight(q.cuda()) for q in qs]
    sd = [s.cuda() for s in ss]
    ys = rf.linear_multi(xd, ws, sd)
    again = rf.linear_multi(xd, ws, sd)
    lib = capi.load()
    bare = [torch.empty_like(y) for y in ys]
    projs = (capi.Proj * len(ns))()
    for i, n in enumerate(ns):
        projs[i] = capi.Proj(ws[i].data_ptr(), sd[i].data_ptr(), None, bare[i].data_ptr(), n, n)
    st = lib.rf_w8a16_linear_multi(xd.data_ptr(), k, 1, projs, len(ns), m, k, 0, None, 0,
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert st == capi.OK, capi.status_str(st)
    rows = np.unique(np.r_[0:2, m // 2, 127, 128, m - 2:m])
    tiles_n = [-(-n // 256) for n in ns]
    for q, s, y, y2, y3, n, t in zip(qs, ss, ys, again, bare, ns, tiles_n):
        assert torch.equal(y, y2)
        cols = np.r_[0:40, (t - 1) * 256: n]     # the first and the last tile column
        for out in (y, y3):
            rep = o.check_tolerance(out.cpu().numpy()[rows][:, cols],
                                    o.cpu_path(x[rows], q.numpy()[cols], s.numpy()[cols]),
                                    o.oracle_fp64(x[rows], q.numpy()[cols], s.numpy()[cols]))
            assert rep.ok, str(rep)


def _unsplit(x, packed, scale, n):
    """The launch without a workspace: every tile whole."""
    import ctypes
    m, k = x.shape
    y = torch.empty(m, n, dtype=torch.float16, device=x.device)
    projs = (capi.Proj * 1)(capi.Proj(packed.data_ptr(), scale.data_ptr(), None, y.data_ptr(), n, n))
    st = capi.load().rf_w8a16_linear_multi(
        x.data_ptr(), k, 1, projs, 1, m, k, 0, None, 0,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == capi.OK, capi.status_str(st)
    return y


def _big(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    q = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    s = (torch.rand(n, generator=g, device="cuda") * 1e-3 + 1e-4).half()
    return x, q, s


@pytest.mark.gpu
def test_last_tiles_of_a_launch_beyond_the_counters():
    """More tiles (16416) than split-K counters (16384), 32 of them past the
    whole rounds: only those have counters."""
    m, n, k = 4096, 131328, 3072
    print(f"last tiles M={m} N={n} K={k}", flush=True)
    tiles, rem = m // 128 * (n // 256), 32
    assert tiles * 4 > capi.WS_COUNTER_BYTES and tiles % 256 == rem
    x, q, s = _big(m, n, k)
    packed = rf.pack_weight(q)
    y, whole = rf.linear(x, packed, s), _unsplit(x, packed, s, n)
    torch.cuda.synchronize()
    assert int((y != whole).sum()) <= rem * 128 * 256  # elsewhere the same sums
    rows = np.unique(np.linspace(0, m - 1, 7).astype(int))
    cols = np.unique(np.r_[np.arange(5, n, 1021), n - 256:n])
    xc, qc, sc = (t.cpu().numpy() for t in (x[rows], q[cols], s[cols]))
    rep = o.check_tolerance(y[rows][:, cols].cpu().numpy(), o.cpu_path(xc, qc, sc),
                            o.oracle_fp64(xc, qc, sc))
    assert rep.ok, str(rep)


@pytest.mark.gpu
def test_last_tiles_under_capture():
    """A capture on a stream whose scratch is still at its least size splits the
    last tiles as an eager call does: the same bits in both, whatever ran on the
    stream before, and counters that eager calls find cleared."""
    m, n, k = 1300, 24576, 3072
    print(f"last tiles under capture M={m} N={n} K={k}", flush=True)
    x, q, s = _big(m, n, k)
    packed = rf.pack_weight(q)
    split, whole = rf.linear(x, packed, s), _unsplit(x, packed, s, n)
    assert not torch.equal(split, whole)  # (the comparison below would see the other order)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        rf.linear(x[:1], packed, s)  # the stream's scratch at its least size
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = rf.linear(x, packed, s)
    with torch.cuda.stream(stream):
        eager = rf.linear(x, packed, s)
    torch.cuda.synchronize()
    assert torch.equal(eager, split)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, split)
        assert torch.equal(rf.linear(x, packed, s), split)


@pytest.mark.parametrize("row", INT4_ROWS, ids=_id)
def test_int4_plan(row):
    m, ns, k, gs, name, splits = row
    p = capi.plan(m, ns, k, fmt=2 if gs else 1, cus=256)
    assert (p["name"], p["splits"]) == (name, splits), p


@pytest.mark.gpu
@pytest.mark.parametrize("row", INT4_ROWS, ids=_id)
def test_int4_parity(row):
    m, ns, k, gs = row[:4]
    print(f"int4 gemm balance M={m} N={ns} K={k} gs={gs}", flush=True)
    x = o.make_activation(o.derive_seed(79, "x", m, k), m, k)
    g = torch.Generator().manual_seed(k)
    qs = [torch.randint(-8, 8, (n, k), generator=g, dtype=torch.int8) for n in ns]
    ss = [(torch.rand((k // gs, n) if gs else (n,), generator=g) * 1e-2 + 1e-3).half() for n in ns]
    xd = torch.from_numpy(x).cuda()
    ws = [rf.pack_weight_int4(q.cuda()) for q in qs]
    sd = [s.cuda() for s in ss]
    ys = rf.linear_multi_w4a16(xd, ws, sd)
    again = rf.linear_multi_w4a16(xd, ws, sd)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[0:2, m // 2, 127, m - 2:m])
    for q, s, y, y2, n in zip(qs, ss, ys, again, ns):
        assert torch.equal(y, y2)
        cols = np.r_[0:40, n // 2:n // 2 + 40, n - 300:n]
        s = np.ascontiguousarray(s.numpy()[..., cols])
        rep = o.check_tolerance(y.cpu().numpy()[rows][:, cols],
                                o4.cpu_path(x[rows], q.numpy()[cols], s),
                                o4.oracle_fp64(x[rows], q.numpy()[cols], s))
        assert rep.ok, str(rep)
