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
