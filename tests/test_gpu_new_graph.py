"""A training call on a graph nobody has seen: both sides' plans are built with it and what both passes take is remembered, so
that the backward of that very call is served by the native host path; results are those of the Python functions."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def new_graph(lengths, device=DEV):
    from bpt_amd import graphbuilder as gb
    src, dst, _, _, n = gb.merge_graphs_device([gb.BinaryPartition(m, True, 4, 10) for m in lengths], torch.device(device))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    return (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]), n


@pytest.mark.parametrize("heads,d,dtype,p", [(8, 64, torch.float32, 0.0), (16, 64, torch.bfloat16, 0.1), (6, 50, torch.float32, 0.1)])
def test_first_backward_of_a_new_graph_is_served_natively(heads, d, dtype, p, monkeypatch):
    from bpt_amd import graphop, op, plan
    plan.plan_cache.clear()
    args, n = new_graph([700, 300, 65])
    gen = torch.Generator(device=DEV).manual_seed(5)
    q, k, v, do = (torch.randn(n, heads, d, generator=gen, device=DEV).to(dtype) for _ in range(4))
    leaves = [x.requires_grad_(True) for x in (q, k, v)]
    o = op.bpt_attention(*args, *leaves, dropout_p=p, seed=3)

    def not_here(*a, **kw):
        raise AssertionError("the backward went through Python")

    with monkeypatch.context() as m:
        m.setattr(graphop, "attention_backward", not_here)
        m.setattr(graphop, "attention_backward_narrow", not_here)
        first = (o.detach(),) + torch.autograd.grad(o, leaves, do)
    # the same through plans that are built one by one when they are asked for
    plan.plan_cache.clear()
    monkeypatch.setattr(graphop, "prepare_training", lambda *a, **kw: None)
    o = op.bpt_attention(*args, *leaves, dropout_p=p, seed=3)
    for name, a, b in zip(("o", "dq", "dk", "dv"), first, (o.detach(),) + torch.autograd.grad(o, leaves, do)):
        assert torch.equal(a, b), name


def test_a_malformed_out_side_is_refused_by_the_backward_only():
    from bpt_amd import op, plan
    plan.plan_cache.clear()
    args, n = new_graph([700, 300, 65])
    bad = list(args)
    bad[3] = args[3].clone()
    bad[3][5] = n + 7                                              # an out-side neighbour that does not exist
    q, k, v = (torch.randn(n, 8, 64, device=DEV, requires_grad=True) for _ in range(3))
    o = op.bpt_attention(*bad, q, k, v)
    with pytest.raises(ValueError):
        o.sum().backward()


@pytest.mark.parametrize("heads,d", [(8, 64), (6, 50)])
def test_an_out_side_of_another_graph_is_refused_by_the_backward_only(heads, d):
    """Each side is sound by itself, but they have different numbers of edges: a forward never asks for the out-side."""
    from bpt_amd import op, plan
    args, n = new_graph([700, 300, 65])
    other, m = new_graph([700, 300, 64])
    assert m < n and args[2].numel() != other[2].numel()
    q, k, v = (torch.randn(n, heads, d, device=DEV, requires_grad=True) for _ in range(3))
    plan.plan_cache.clear()
    want = op.bpt_attention(*args, q, k, v)
    plan.plan_cache.clear()
    o = op.bpt_attention(*other[:4], *args[4:], q, k, v)
    assert torch.equal(o, want)
    with pytest.raises(ValueError):
        o.sum().backward()


@pytest.mark.parametrize("limits", [dict(capacity=1), dict(max_bytes=0)])
def test_a_cache_too_small_for_both_sides_builds_neither_again(limits):
    """Both sides are built together once; what the cache has no room for is built where a pass asks for it, as ever."""
    from bpt_amd import graphop, op, plan
    args, n = new_graph([700, 300, 65])
    leaves = [torch.randn(n, 8, 64, device=DEV, requires_grad=True) for _ in range(3)]

    def step():
        o = op.bpt_attention(*args, *leaves)
        return (o.detach(),) + torch.autograd.grad(o.sum(), leaves)

    plan.plan_cache.clear()
    want = step()
    old = plan.plan_cache.set_limits(**limits)
    try:
        plan.plan_cache.clear()
        built = plan.plan_cache.misses
        graphop.prepare_training(*args, *leaves[:2])
        assert plan.plan_cache.misses == built + 2 and len(plan.plan_cache._d) == 1
        plan.plan_cache.clear()
        got = step()
    finally:
        plan.plan_cache.set_limits(*old)
        plan.plan_cache.clear()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("tiles", [False, True])
def test_a_forced_backward_is_chosen_by_the_backward(tiles, monkeypatch):
    """Nothing is remembered ahead while TILE_BACKWARD is set: the first backward reads it."""
    from bpt_amd import graphop, op, plan
    monkeypatch.setattr(graphop, "TILE_BACKWARD", tiles)
    plan.plan_cache.clear()
    args, n = new_graph([700, 300, 65])
    q, k, v = (torch.randn(n, 8, 64, device=DEV, requires_grad=True) for _ in range(3))
    here, real = [], graphop.attention_backward
    monkeypatch.setattr(graphop, "attention_backward", lambda *a, **kw: here.append(1) or real(*a, **kw))
    op.bpt_attention(*args, q, k, v).sum().backward()
    plan.plan_cache.clear()
    assert here
