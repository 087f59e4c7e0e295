"""Attention with relative positions on the native host path (bptop.so's rel_attention): a call served from its table gives the bits of the Python
function that was remembered, forward and backward, and whatever it does not recognise goes to that function."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def graph(length=700, k=4, causal=True):
    from bpt_amd import graphbuilder as gb
    src, dst, etype, _, n = gb.merge_graphs_device([gb.BinaryPartition(length, causal, k, 10)], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    return (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]), etype, n


def inputs(n, h, d, dtype, grad=True):
    gen = torch.Generator().manual_seed(1)
    x = [(torch.randn(n, h, d, generator=gen)).to(dtype).to(DEV) for _ in range(4)]
    table = (torch.randn(1000, d, generator=gen) * 0.1).to(dtype).to(DEV)
    return [t.requires_grad_(grad) for t in x[:3]], table.requires_grad_(grad), x[3]


def served(native, monkeypatch):
    """Counts what rel_attention answers itself."""
    from bpt_amd import op
    seen = []

    class Counting:
        def __getattr__(self, name):
            return getattr(native, name)

        def rel_attention(self, *args):
            o = native.rel_attention(*args)
            seen.append(o is not None)
            return o

    monkeypatch.setattr(op, "_native", Counting())
    return seen


@pytest.mark.parametrize("h,d,dtype", [(8, 64, torch.float32), (16, 64, torch.bfloat16), (6, 50, torch.float32)])
@pytest.mark.parametrize("p", [0.0, 0.1])
def test_served_passes_equal_the_remembered_one(h, d, dtype, p, monkeypatch):
    from bpt_amd import op, plan
    from bpt_amd._native import native
    plan.plan_cache.clear()
    op._rel_aux_cache.clear()
    args, etype, n = graph()
    (q, k, v), table, do = inputs(n, h, d, dtype)
    seen, outs = served(native, monkeypatch), []
    for _ in range(3):
        o = op.bpt_attention(*args, q, k, v, dropout_p=p, seed=5, rel_table=table, etype=etype)
        outs.append((o.detach(),) + torch.autograd.grad(o, (q, k, v, table), do))
    assert seen == [False, True, True]
    for other in outs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(outs[0], other))
    with torch.no_grad():                                          # the entry of a training pass serves a forward alone
        assert torch.equal(op.bpt_attention(*args, q, k, v, dropout_p=p, seed=5, rel_table=table, etype=etype), outs[0][0]) and seen[-1]


def test_a_forward_alone_is_remembered_for_forwards_only(monkeypatch):
    from bpt_amd import op, plan
    from bpt_amd._native import native
    plan.plan_cache.clear()
    op._rel_aux_cache.clear()
    args, etype, n = graph()
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)
    seen = served(native, monkeypatch)
    with torch.no_grad():
        first = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
        second = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    assert seen == [False, True] and torch.equal(first, second)
    o = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    grads = torch.autograd.grad(o, (q, k, v, table), do)
    o = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    again = torch.autograd.grad(o, (q, k, v, table), do)
    assert seen == [False, True, False, True] and all(torch.equal(a, b) for a, b in zip(grads, again))


def test_what_changes_a_call_is_not_served(monkeypatch):
    """Other edge types (another version of the tensor, another tensor), a table of another length, tensors that are not contiguous,
    a plan dropped from the cache, a switch: the Python function's result each time."""
    from bpt_amd import graphop, op, plan
    from bpt_amd._native import native
    plan.plan_cache.clear()
    op._rel_aux_cache.clear()
    args, etype, n = graph()
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)
    seen = served(native, monkeypatch)

    def call(q=q, k=k, v=v, table=table, etype=etype):
        o = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
        return (o.detach(),) + torch.autograd.grad(o, (q, k, v, table), do)

    base = call()
    assert all(torch.equal(a, b) for a, b in zip(base, call())) and seen == [False, True]
    other = etype.clone()
    other[:100] = 7
    want = call(etype=other)
    etype.copy_(other)                                             # (a new version: what was remembered of the old values is not used)
    got = call()
    assert seen[2:] == [False, False] and all(torch.equal(a, b) for a, b in zip(want, got)) and not torch.equal(want[0], base[0])
    longer = torch.cat([table.detach(), table.detach()[:5]]).requires_grad_(True)
    got = call(table=longer)
    assert seen[-1] is False and torch.equal(got[0], want[0]) and torch.equal(got[4][:1000], want[4])
    spread = torch.stack([q.detach(), q.detach()], 3)[..., 0].requires_grad_(True)
    assert not spread.is_contiguous()
    with pytest.raises(RuntimeError):                              # as ever
        call(q=spread)
    wide = torch.stack([table.detach()] * 2, 2)[..., 0].requires_grad_(True)
    assert torch.equal(call(table=wide)[4], want[4]) and seen[-1] is False
    call()
    assert seen[-1] is True
    plan.plan_cache.clear()
    assert torch.equal(call()[1], want[1]) and seen[-1] is False
    call()
    assert seen[-1] is True
    old = graphop.set_tiles(False)
    try:
        got = call()
        assert seen[-1] is False and torch.allclose(got[1], want[1], atol=1e-4)
    finally:
        graphop.set_tiles(old)


def test_a_backward_after_its_plans_left_the_cache():
    from bpt_amd import op, plan
    plan.plan_cache.clear()
    op._rel_aux_cache.clear()
    args, etype, n = graph()
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)
    run = lambda: op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    want = torch.autograd.grad(run(), (q, k, v, table), do)
    o = run()
    plan.plan_cache.clear()
    op._rel_aux_cache.clear()
    assert all(torch.equal(a, b) for a, b in zip(want, torch.autograd.grad(o, (q, k, v, table), do)))


def test_captured_passes_replay():
    """A captured forward and backward, replayed with other inputs and eager work in between, give the eager results."""
    from bpt_amd import op
    args, etype, n = graph(300)
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)

    def run():
        o = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
        return (o,) + torch.autograd.grad(o, (q, k, v, table), do)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            run()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        outs = run()
    for i in range(3):
        with torch.no_grad():
            q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(40 + i)).to(DEV))
        want = [x.clone() for x in run()]
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(want, outs))


def test_a_tangent_is_refused():
    from bpt_amd import op
    import torch.autograd.forward_ad as fwAD
    args, etype, n = graph(300)
    (q, k, v), table, _ = inputs(n, 8, 64, torch.float32, grad=False)
    for _ in range(2):
        op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    with fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        op.bpt_attention(*args, fwAD.make_dual(q, torch.ones_like(q)), k, v, rel_table=table, etype=etype)
