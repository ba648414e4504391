"""Decode GEMV with one strip per workgroup where x comes through LDS tiles of
each wavefront (int8 from M 9, int4 from M 5): rows up to and past eight, one
to eight pipeline stages (from four on the steady-state loop refills both
buffers) with a partial last one, K splits, K tails inside a tile, strided rows;
against the fp64 oracle and the CPU path."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import rhinoforge_amd as rf
from rhinoforge_amd import capi
from oracle import w4a16 as o4
from oracle import w8a16 as o

# (M, N, K, group size or None for int8, plan name)
CASES = [
    (9, 1000, 1000, None, "gemv 1x1 strips, 16 waves"),    # one tile a wavefront at most, K tail
    (16, 2056, 4104, None, "gemv 1x1 strips, 16 waves"),   # 65 tiles: 2 / 3 stages, K tail of 8
    (12, 2048, 2048, None, "gemv 1x1 strips, 16 waves"),
    (16, 1024, 5176, None, "gemv 1x1 strips, 8 waves"),    # four splits, K tail of 56
    (5, 2048, 2048, 0, "gemv 1x1 strips, 16 waves"),
    (8, 4096, 4160, 32, "gemv 1x1 strips, 16 waves"),      # K % 128 == 64
    (16, 2048, 3008, 64, "gemv 1x1 strips, 16 waves"),     # K % 128 == 64, 24 tiles
    (9, 1008, 1024, 128, "gemv 1x1 strips, 16 waves"),
    (13, 4096, 4096, 0, "gemv 1x1 strips, 16 waves"),
]

# The same with at least four stages in every format and both tile heights:
# (..., stages of the wavefronts).  A stage is two int8 tiles or one int4 tile.
DEEP = [
    (9, 2048, 7000, None, "gemv 1x1 strips, 16 waves", {3, 4}),    # K tail of 24, last stage of one tile
    (16, 4096, 7936, None, "gemv 1x1 strips, 16 waves", {4}),
    (12, 3000, 8120, None, "gemv 1x1 strips, 16 waves", {4}),      # 127 tiles, ragged N, K tail of 56
    (16, 4096, 7936, 0, "gemv 1x1 strips, 16 waves", {3, 4}),
    (13, 4096, 8000, 64, "gemv 1x1 strips, 16 waves", {3, 4}),     # K % 128 == 64
    (6, 512, 16256, 0, "gemv 1x1 strips, 16 waves", {7, 8}),       # 127 tiles, eight rows
    (5, 1024, 16064, 32, "gemv 1x1 strips, 16 waves", {7, 8}),     # K % 128 == 64
    (7, 1008, 12288, 128, "gemv 1x1 strips, 16 waves", {6}),
    (8, 512, 8064, 32, "gemv 1x1 strips, 16 waves", {3, 4}),
]
CASES += [c[:5] for c in DEEP]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-{c[3]}")
def test_plan(case):
    m, n, k, gs, name = case
    p = capi.plan(m, n, k, fmt=0 if gs is None else 2 if gs else 1, cus=256)
    assert (p["kernel"], p["name"]) == ("gemv", name), p


@pytest.mark.parametrize("case", DEEP, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-{c[3]}")
def test_stage_counts(case):
    m, n, k, gs, _, stages = case
    p = capi.plan(m, n, k, fmt=0 if gs is None else 2 if gs else 1, cus=256)
    tiles, per_stage = -(-k // (64 if gs is None else 128)), 2 if gs is None else 1
    assert p["splits"] == 1 and p["tile_n"] == 16
    assert {-(-((tiles - w + p["waves"] - 1) // p["waves"]) // per_stage)
            for w in range(p["waves"])} == stages


def test_int4_from_m5_takes_no_eight_wavefront_one_strip_plan():
    """That configuration has no x tiles in LDS: it is planned up to M 4 only."""
    for fmt in (1, 2):
        for m in range(5, 65):
            for n in (16, 512, 1024, 1040, 2064, 4096, 8192, 10240, 20480, 40960, 151936):
                for k in (128, 1024, 2048, 4096, 8192, 12288, 16384, 25600, 65536):
                    p = capi.plan(m, n, k, kernel=capi.KERNEL_GEMV, fmt=fmt, cus=256)
                    assert p["name"] != "gemv 1x1 strips, 8 waves", (m, n, k, p)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-{c[3]}")
def test_parity(case):
    m, n, k, gs, _ = case
    print(f"gemv x tiles M={m} N={n} K={k} gs={gs}", flush=True)
    w = o.make_weight(o.derive_seed(55, "w", n, k), n, k)
    x = o.make_activation(o.derive_seed(55, "x", m, k), m, k)
    if gs is None:
        q, s = o.quantize_linear_per_channel(w)
        cpu, ref = o.cpu_path(x, q, s), o.oracle_fp64(x, q, s)
        wp, run = rf.pack_weight(torch.from_numpy(q).cuda()), rf.linear
    else:
        q, s = o4.quantize_int4_group_wise(w, gs) if gs else o4.quantize_int4_per_channel(w)
        cpu, ref = o4.cpu_path(x, q, s), o4.oracle_fp64(x, q, s)
        wp, run = rf.pack_weight_int4(torch.from_numpy(q).cuda()), rf.linear_w4a16
    sd = torch.from_numpy(np.ascontiguousarray(s)).cuda()
    xd = torch.from_numpy(x).cuda()
    wide = torch.full((m, k + 24), float("nan"), dtype=torch.float16, device="cuda")
    wide[:, :k] = xd                                # NaN past the rows is never used
    y = run(xd, wp, sd, kernel=rf.KERNEL_GEMV)
    y2 = run(wide[:, :k], wp, sd, kernel=rf.KERNEL_GEMV)
    torch.cuda.synchronize()
    rep = o.check_tolerance(y.cpu().numpy(), cpu, ref)
    assert rep.ok, str(rep)
    assert torch.equal(y, y2)
