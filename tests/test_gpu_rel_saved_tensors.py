"""Hooks on the tensors that the attention with relative positions saves for its backward, on the native host path: what comes back as it went gives the
same gradients, anything that the kernels cannot read is refused, as by the Python function."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
N_TYPES = 1000


def served_call(h, dtype):
    """(a call that the native path knows, its inputs, the gradient of its result, the shapes of what it saves by name)"""
    from bpt_amd import graphbuilder as gb, op
    from bpt_amd._native import native
    src, dst, etype, _, n = gb.merge_graphs_device([gb.BinaryPartition(300, True, 4, 10)], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    args = (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1])
    gen = torch.Generator().manual_seed(3)
    q, k, v, do = (torch.randn(n, h, 64, generator=gen).to(dtype).to(DEV) for _ in range(4))
    table = (torch.randn(N_TYPES, 64, generator=gen) * 0.1).to(dtype).to(DEV)
    x = [t.requires_grad_(True) for t in (q, k, v, table)]
    call = lambda: op.bpt_attention(*args, *x[:3], rel_table=x[3], etype=etype)
    torch.autograd.grad(call(), x, do)
    assert native.rel_attention(*args, *x[:3], 0.125, 0.0, 0, x[3], etype) is not None
    return call, x, do, {"rows": (n, h, 64), "lse": (n, h), "term": (h, etype.numel()), "table": (N_TYPES, 64)}


@pytest.mark.parametrize("h,dtype", [(8, torch.float32), (16, torch.bfloat16)])
def test_tensors_that_come_back_as_they_went(h, dtype):
    call, x, do, _ = served_call(h, dtype)
    want = torch.autograd.grad(call(), x, do)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(DEV)):
        o = call()
    assert all(torch.equal(a, b) for a, b in zip(want, torch.autograd.grad(o, x, do)))


@pytest.mark.parametrize("which", ["rows", "lse", "term", "table"])
@pytest.mark.parametrize("how", ["host", "order", "type", "short"])
def test_tensors_that_come_back_otherwise_are_refused(which, how):
    call, x, do, shapes = served_call(8, torch.float32)
    change = {"host": lambda t: t.cpu(), "order": lambda t: t.transpose(0, 1).contiguous().transpose(0, 1), "type": lambda t: t.double(),
              "short": lambda t: t[:-1].contiguous()}[how]
    assert len(set(shapes.values())) == 4
    hit = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: (hit.append(1), change(t))[1] if tuple(t.shape) == shapes[which] else t):
        o = call()
    with pytest.raises((RuntimeError, ValueError, TypeError)):
        torch.autograd.grad(o, x, do)
    assert hit
