"""The device quantizers (one kernel) against the torch arithmetic they stand
for, byte for byte: every weight type, values and steps row-major and packed,
at the edges of the kernels' chunks, tiles and kept rows, on strided and
misaligned inputs, and with rows that hold ties, zeros, infinities and NaN.
"""
from __future__ import annotations

import pytest
import torch

import rhinoforge_amd as rf
from rhinoforge_amd.quant import _common, int4

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _eager(fn, *args, **kw):
    """The quantizer's torch path (the kernels switched off)."""
    keep = _common.on_kernel
    _common.on_kernel = int4.on_kernel = lambda w: False
    try:
        return fn(*args, **kw)
    finally:
        _common.on_kernel = int4.on_kernel = keep


def _weight(n, k, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randn(n, k, generator=g, device=DEV) * 0.02
    w[0] = 0                                       # floored step
    if n > 2:
        w[1, : min(k, 9)] = torch.tensor([127.0, 0.5, 1.5, -2.5, 63.5, -126.5, -127.0, 3.0, -0.5],
                                         device=DEV)[: min(k, 9)]    # ties at step 1
        w[2] *= 1e-4                                # fp16 subnormals
    if n > 5:
        w[3, k // 2] = float("inf")
        w[4, k - 1] = float("nan")
        w[5, 0] = 7e4                               # infinite once rounded to fp16
    return w.to(dtype)


def _same(a, b):
    assert a.dtype == b.dtype and a.shape == b.shape
    assert torch.equal(a.view(torch.int16) if a.dtype == torch.float16 else a,
                       b.view(torch.int16) if b.dtype == torch.float16 else b)


def _steps(s):  # NaN payloads are not part of the contract
    return torch.where(s.isnan(), torch.full_like(s, float("nan")), s)


# K: a partial chunk, one chunk, an odd multiple of 8, the kept 4096 exactly
# and one chunk past it, a long row; N: one row, ragged strips.
SHAPES = [(1, 8), (17, 16), (40, 70), (33, 520), (16, 4096), (7, 4112), (130, 12296)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("bits", [8, 4])
def test_per_channel_matches_torch(dtype, n, k, bits):
    print(f"quantize {n}x{k} {dtype} {bits} bits", flush=True)
    w = _weight(n, k, dtype, n + k)
    q0, s0 = _eager(_common.quantize_linear_per_channel, w, bits=bits)
    q, s = rf.quantize_linear_per_channel(w, bits=bits)
    _same(_steps(s), _steps(s0))
    _same(q, q0)
    if bits == 8 or (n % 16 == 0 and k % 64 == 0):
        pack = rf.pack_weight if bits == 8 else rf.pack_weight_int4
        p, sp = torch.ops.rhinoforge.quantize_pack(w, bits, 0)
        _same(p, pack(q0))
        _same(_steps(sp), _steps(s0))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,k,gs", [(16, 64, 32), (48, 1088, 64), (17, 2048, 128), (256, 4160, 32),
                                    (64, 128, 128)])
def test_group_wise_matches_torch(dtype, n, k, gs):
    print(f"quantize groups {n}x{k} {dtype} gs {gs}", flush=True)
    w = _weight(n, k, dtype, 3 * n + k)
    q0, s0, _ = _eager(int4.quantize_int4_group_wise, w, gs)
    q, s, g = rf.quantize_int4_group_wise(w, gs)
    assert g == gs
    _same(_steps(s), _steps(s0))
    _same(q, q0)
    p, sp = torch.ops.rhinoforge.quantize_pack(w, 4, gs)
    _same(p, rf.pack_weight_int4(q0))
    _same(_steps(sp), _steps(s0))


def test_strided_and_misaligned_inputs():
    base = _weight(40, 300, torch.float16, 1)
    for w in (base[:, 3:260], base.t()[:, :33], base[::3, :128], base[1:2]):
        q0, s0 = _eager(_common.quantize_linear_per_channel, w)
        q, s = rf.quantize_linear_per_channel(w)
        _same(q, q0)
        _same(_steps(s), _steps(s0))


@pytest.mark.parametrize("shape,off,ld", [((48, 256), 0, 256), ((40, 130), 0, 130),
                                          ((48, 256), 8, 264), ((17, 64), 1, 65)])
def test_pack_of_any_alignment(shape, off, ld):
    """16-byte loads where the rows allow them, a load per byte otherwise."""
    n, k = shape
    g = torch.Generator(device=DEV).manual_seed(n)
    flat = torch.randint(-8, 8, (n * ld + 16,), generator=g, device=DEV, dtype=torch.int8)
    q = flat[off: off + n * ld].view(n, ld)[:, :k]
    host = q.cpu().contiguous()
    assert torch.equal(rf.pack_weight(q).cpu(), rf.pack_weight(host))
    qc = flat[off: off + n * k].view(n, k)
    assert torch.equal(rf.pack_weight(qc).cpu(), rf.pack_weight(qc.cpu()))
    assert torch.equal(rf.pack_weight_int4(qc).cpu(), rf.pack_weight_int4(qc.cpu()))


def test_modules_from_linear():
    for dtype in (torch.bfloat16, torch.float32):
        lin = torch.nn.Linear(1088, 48, bias=True, device=DEV, dtype=dtype)
        m = rf.W8A16Linear.from_linear(lin)
        q, s = _eager(_common.quantize_linear_per_channel, lin.weight)
        ref = rf.W8A16Linear.from_quantized(q, s, lin.bias.detach().half())
        for gs in (None, 64):
            m4 = rf.W4A16Linear.from_linear(lin, group_size=gs)
            q4, s4 = (_eager(int4.quantize_int4_group_wise, lin.weight, gs)[:2] if gs
                      else _eager(int4.quantize_int4_per_channel, lin.weight))
            r4 = rf.W4A16Linear.from_quantized(q4, s4, lin.bias.detach().half())
            for name in ("weight", "weight_scale", "bias"):
                _same(getattr(m4, name), getattr(r4, name))
            assert m4.group_size == gs and not m4.weight_scale.requires_grad
        for name in ("weight", "weight_scale", "bias"):
            _same(getattr(m, name), getattr(ref, name))
        assert (m.in_features, m.out_features) == (1088, 48)


def test_from_linear_refuses_a_bias_of_another_shape():
    """As on the CPU: refused when the module is made, not by its first call."""
    for dev in ("cpu", DEV):
        for shape in ((47,), (1, 48), ()):
            lin = torch.nn.Linear(64, 48, device=dev)
            lin.bias = torch.nn.Parameter(torch.zeros(shape, device=dev))
            with pytest.raises(ValueError, match="bias must have shape"):
                rf.W8A16Linear.from_linear(lin)


def test_more_rows_than_one_launch_holds():
    """2^26 rows of one repeated pattern: the torch arithmetic, as on the CPU."""
    n, k = 2**26, 8
    w = torch.tensor([0.5, -1, 0.25, 0, 1.5, -2, 3, 1], device=DEV, dtype=torch.float16)
    q, s = rf.quantize_linear_per_channel(w.expand(n, k))
    q1, s1 = rf.quantize_linear_per_channel(w.expand(1, k).cpu())
    assert q.shape == (n, k) and bool((q == q1.to(DEV)).all()) and bool((s == s1.to(DEV)).all())
    edge = w.expand(_common._KERNEL_SIZE - 1, k)     # the most the kernel takes
    assert _common.on_kernel(edge)
    q, s = rf.quantize_linear_per_channel(edge)
    assert bool((q == q1.to(DEV)).all()) and bool((s == s1.to(DEV)).all())
    x = torch.zeros(1, 2**26, device=DEV, dtype=torch.float16)
    x[0, ::32] = 7.0
    q, s, _ = rf.quantize_int4_group_wise(x, 32)
    assert s.shape == (2**21, 1) and bool((s == 1).all()) and int(q.sum()) == 7 * 2**21
    x = x[:, :_common._KERNEL_SIZE - 32]
    q, s, _ = rf.quantize_int4_group_wise(x, 32)
    assert bool((s == 1).all()) and int(q.sum()) == 7 * (x.size(1) // 32)
