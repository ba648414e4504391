"""The packed-int4 GEMM tiles of 128-wide K blocks (M <= 64, and launches of few
tiles beyond) at the edges of their ranges: one row past a tile, ragged N, a K
that ends 64 positions into its last block (in the last of several K splits
too), every scale form, and several projections in one launch.

Tolerance as in test_gpu_w4a16: max|y - y_cpu| <= 1e-2 * rms(y_cpu), cosine >=
0.9999 per row, against the fp16-dequantize-then-GEMM CPU path and the fp64
oracle; one-hot activations reproduce the dequantized column exactly.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import rhinoforge_amd as rf
from rhinoforge_amd import capi
from oracle import w4a16 as o4
from oracle import w8a16 as o8
from test_gpu_w4a16 import _dev, _say, check, make_w4, run

# (M, N, K, group size, tile_m, tile_n, K splits on a 256-CU part)
TILES = [
    (17, 2064, 1088, 32, 32, 64, 1),       # ragged N, K % 128 == 64
    (17, 1040, 4160, 32, 32, 64, 7),       # seven splits, the K tail in the last
    (32, 19456, 1024, 128, 32, 128, 1),
    (33, 2048, 2048, 0, 32, 64, 4),        # one row in the second row of tiles
    (48, 9728, 2112, 64, 48, 64, 3),       # ragged splits, K tail
    (47, 24576, 1088, 32, 48, 128, 1),
    (49, 12288, 1024, 32, 64, 64, 1),
    (64, 19472, 1088, 0, 64, 128, 1),      # ragged N, K tail, per-channel
    (65, 1008, 4160, 32, 48, 64, 7),       # one row past a tile; tail in the last split
    (129, 4096, 1088, 64, 48, 64, 1),
    (512, 2048, 4096, 128, 64, 128, 2),
    (1500, 528, 1024, 32, 64, 64, 1),
]


@pytest.mark.parametrize("row", TILES, ids=lambda r: f"{r[0]}x{r[1]}x{r[2]}-g{r[3]}")
def test_int4_tile_plan(row):
    m, n, k, gs, tm, tn, splits = row
    p = capi.plan(m, n, k, kernel=capi.KERNEL_GEMM, fmt=2 if gs else 1, cus=256)
    assert (p["tile_m"], p["tile_n"], p["splits"]) == (tm, tn, splits), p
    assert p["name"] == f"gemm {tm}x{tn} 128-wide K blocks"


@pytest.mark.gpu
@pytest.mark.parametrize("row", TILES, ids=lambda r: f"{r[0]}x{r[1]}x{r[2]}-g{r[3]}")
def test_int4_tile_parity(row):
    m, n, k, gs = row[:4]
    _say(f"int4 tile M={m} N={n} K={k} gs={gs}")
    q, s = make_w4(n, k, gs, 11)
    x = o8.make_activation(o8.derive_seed(11, "x4t", m, k), m, k)
    b = (o8.normal(o8.derive_seed(11, "b4t", n), (n,)) * 0.1).astype(np.float16) if m % 2 else None
    packed = rf.pack_weight_int4(_dev(q))
    y = run(x, q, s, b, kernel=rf.KERNEL_GEMM, packed=packed)
    rows = None if m <= 65 else np.unique(np.linspace(0, m - 1, 48).astype(int))
    check(y, x, q, s, b, label=f"int4 tile {m}x{n}x{k} gs={gs}", rows=rows)
    y2 = run(x, q, s, b, kernel=rf.KERNEL_GEMM, packed=packed)
    assert (y.view(np.uint16) == y2.view(np.uint16)).all()  # counters zeroed, fixed sum order
    one = np.zeros((m, k), np.float16)
    cols = [(k - 1 - 37 * i) % k for i in range(m)]         # the last column included
    one[np.arange(m), cols] = 1.0
    want = o4.dequantize_int4(q, s)[:, cols].T
    got = run(one, q, s, kernel=rf.KERNEL_GEMM, packed=packed)
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


@pytest.mark.gpu
def test_int4_tiles_several_projections():
    """Three ragged projections in one launch of the 48-row tiles, AUTO."""
    m, ns, k, gs = 41, [1040, 528, 16], 2112, 64
    x = o8.make_activation(12, m, k)
    ws = [make_w4(n, k, gs, 20 + i) for i, n in enumerate(ns)]
    assert capi.plan(m, ns, k, fmt=2)["kernel"] == "gemm"
    ys = rf.linear_multi_w4a16(_dev(x), [rf.pack_weight_int4(_dev(q)) for q, _ in ws],
                               [_dev(s) for _, s in ws])
    torch.cuda.synchronize()
    for (q, s), y in zip(ws, ys):
        check(y.cpu().numpy(), x, q, s, label=f"int4 multi N={y.shape[1]}")
