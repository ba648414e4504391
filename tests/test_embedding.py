"""W8A16Embedding's lookup op: every index form that torch indexing takes, on
the CPU and under meta / vmap / autograd, against the torch expression; the HIP
kernel (16-, 8- and 1-wide) byte for byte against the same on the GPU."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import rhinoforge_amd as rf


def _table(v, h, dev="cpu"):
    g = torch.Generator().manual_seed(v + h)
    q = torch.randint(-128, 128, (v, h), generator=g, dtype=torch.int8)
    s = (torch.rand(v, generator=g) * 0.01).half()
    s[0] = 6e-8                                    # fp16 subnormal products
    return q.to(dev), s.to(dev)


def _want(q, s, ids):
    return (q[ids].float() * s[ids].float().unsqueeze(-1)).half()


def _forms(v, dev):
    base = torch.tensor([[0, 1, v - 1], [-1, -v, v // 2]], device=dev)
    mask = torch.zeros(v, dtype=torch.bool, device=dev)
    mask[::3] = True
    return {"int64": base, "int32": base.int(), "transposed": base.t(), "scalar": base[0, 1],
            "empty": base[:0], "mask": mask, "one row": base[0, :1]}


def _check(q, s, dev):
    emb = rf.W8A16Embedding(q, s)
    for name, ids in _forms(q.size(0), dev).items():
        got, want = emb(ids), _want(q, s, ids)
        assert got.shape == want.shape and got.dtype == torch.float16, name
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), name


def test_cpu_forms():
    q, s = _table(50, 24)
    _check(q, s, "cpu")
    with pytest.raises(IndexError):
        rf.W8A16Embedding(q, s)(torch.tensor([50]))
    with pytest.raises(IndexError):
        rf.W8A16Embedding(q, s)(torch.tensor([0.5]))


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_indices_that_are_not_tensors(dev):
    q, s = _table(50, 24, dev)
    emb = rf.W8A16Embedding(q, s)
    for ids in (7, -1, [3, 1, -50], slice(2, 9), np.array([[4, 5]]), ([1, 2],), ...):
        assert torch.equal(emb(ids), _want(q, s, ids)), ids
    with pytest.raises(IndexError):
        emb(50)


def test_scripted_and_traced():
    q, s = _table(50, 24)
    emb = rf.W8A16Embedding(q, s)
    ids = torch.tensor([[3, 1], [-1, 7]])
    for m in (torch.jit.script(emb), torch.jit.trace(emb, ids),
              torch.export.export(emb, (ids,)).module(),
              torch.compile(emb, backend="eager", fullgraph=True)):
        assert torch.equal(m(ids), _want(q, s, ids))


def test_tensor_subclasses(tmp_path):
    """Sharded tables and ids, and fake tensors, through their own indexing."""
    import torch.distributed as dist
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.distributed.tensor import Replicate, Shard, distribute_tensor, init_device_mesh
    q, s = _table(50, 24)
    ids = torch.tensor([[3, 1], [-1, 7]])
    with FakeTensorMode() as mode:
        y = rf.W8A16Embedding(mode.from_tensor(q), mode.from_tensor(s))(mode.from_tensor(ids))
        assert y.shape == (2, 2, 24) and y.dtype == torch.float16
    dist.init_process_group("gloo", init_method=f"file://{tmp_path}/store", rank=0, world_size=1)
    try:
        mesh = init_device_mesh("cpu", (1,))
        di = distribute_tensor(ids, mesh, [Replicate()])
        for place in (Replicate(), Shard(0), Shard(1)):
            emb = rf.W8A16Embedding(distribute_tensor(q, mesh, [place]),
                                    distribute_tensor(s, mesh, [Replicate()]))
            assert torch.equal(emb(di).full_tensor(), _want(q, s, ids)), place
    finally:
        dist.destroy_process_group()


def test_transforms():
    q, s = _table(50, 24)
    ids = torch.tensor([[3, 1], [-1, 7]])
    emb = rf.W8A16Embedding(q, s)
    assert torch.equal(torch.vmap(emb)(ids), _want(q, s, ids))
    sg = s.clone().requires_grad_()
    emb.weight_scale = sg
    emb(ids).float().sum().backward()
    ref = s.clone().requires_grad_()
    _want(q, ref, ids).float().sum().backward()
    assert torch.equal(sg.grad, ref.grad)
    m = torch.ops.rhinoforge.embedding(q.to("meta"), s.to("meta"), ids.to("meta"))
    assert m.shape == (2, 2, 24) and m.dtype == torch.float16


def test_replaced_buffers():
    """The lookup reads what the module holds: another tensor, a parameter in the
    buffer's place, a parametrization, functional_call's tensors."""
    from torch.nn.utils import parametrize
    q, s = _table(50, 24)
    ids = torch.tensor([[3, 1], [-1, 7]])

    class Halve(torch.nn.Module):
        def forward(self, t):
            return t * 0.5

    emb = rf.W8A16Embedding(q, s)
    emb.weight = q.flip(0).contiguous()
    assert torch.equal(emb(ids), _want(q.flip(0), s, ids))
    swap = {"weight": q, "weight_scale": s * 2}
    assert torch.equal(torch.func.functional_call(emb, swap, (ids,)), _want(q, s * 2, ids))
    parametrize.register_parametrization(emb, "weight_scale", Halve())
    assert torch.equal(emb(ids), _want(q.flip(0), s * 0.5, ids))
    emb = rf.W8A16Embedding(q, s)
    del emb.weight_scale
    emb.weight_scale = torch.nn.Parameter(s * 4)
    assert torch.equal(emb(ids), _want(q, s * 4, ids))


@pytest.mark.gpu
@pytest.mark.parametrize("v,h", [(300, 4096), (97, 4112), (50, 24), (33, 8), (20, 7), (9, 1),
                                 (1000, 5120)])
def test_gpu_forms(v, h):
    print(f"embedding {v}x{h}", flush=True)
    q, s = _table(v, h, "cuda")
    _check(q, s, "cuda")
    wide = torch.zeros(v * h + 3, dtype=torch.int8, device="cuda")   # a misaligned table
    odd = wide[3:].view(v, h).copy_(q)
    ids = torch.randint(-v, v, (3, 70), device="cuda")
    emb = rf.W8A16Embedding(odd, s)
    assert torch.equal(emb(ids), _want(q, s, ids))
    strided = torch.as_strided(ids, (35, 3), (2, 70))
    assert torch.equal(emb(strided), _want(q, s, strided))


@pytest.mark.gpu
@pytest.mark.parametrize("m,h", [((1 << 24) + 5, 16), ((1 << 23) + 3, 257)])
def test_gpu_more_rows_than_one_launch_holds(m, h):
    """A launch holds fewer than 2^24 workgroups of 256 threads, one (16-wide
    rows) or two (257-wide, a value per thread) to a row here."""
    print(f"embedding of {m} ids x {h}", flush=True)
    q, s = _table(1000, h, "cuda")
    for dtype in (torch.int64, torch.int32):
        ids = torch.randint(-1000, 1000, (m,), device="cuda", dtype=dtype)
        got = rf.W8A16Embedding(q, s)(ids)
        for i in range(0, m, 1 << 20):
            part = ids[i:i + (1 << 20)]
            assert torch.equal(got[i:i + (1 << 20)], _want(q, s, part)), i
        del got


@pytest.mark.gpu
@pytest.mark.parametrize("h", [4096, 24, 7])
def test_gpu_ids_outside_the_table(h):
    """Rows of NaN, without a read outside the table; the other rows as always."""
    print(f"embedding ids outside the table, width {h}", flush=True)
    v = 50
    q, s = _table(v, h, "cuda")
    bad = [v, -v - 1, 2**31 - 1, -2**31, 2**40, -2**62]
    for dtype, n in ((torch.int64, 6), (torch.int32, 4)):
        ids = torch.tensor([3, *bad[:n], -1], device="cuda", dtype=dtype)
        y = rf.W8A16Embedding(q, s)(ids)
        assert y[1:-1].isnan().all()
        assert torch.equal(y[[0, -1]], _want(q, s, ids[[0, -1]]))
