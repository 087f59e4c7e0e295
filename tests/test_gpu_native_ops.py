"""The native host path of masked_mm, sparse_softmax and vec_spmm: the results and gradients of the autograd functions it stands for, bit for
bit, on a first call and on later ones; what the functions refuse is refused, what they hold is held."""
import math

import pytest
import torch

from test_gpu_product_tiles import DEV, rand, sides

pytestmark = pytest.mark.gpu


def chain(ops, s, q, k, v):
    e = ops[0](*s.out, *s.inn, k, q)
    a = ops[1](*s.inn[:3], e / math.sqrt(q.size(-1)))
    return ops[2](*s.inn, *s.out, a, v)


@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 8, 64), (torch.float32, 6, 50), (torch.bfloat16, 8, 64), (torch.float64, 3, 10)],
                         ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("name", ["bpt512", "multigraph"])
def test_same_bits_as_the_autograd_functions(name, dtype, h, d, monkeypatch):
    from bpt_amd import graphop, op, plan
    s = sides(name)
    x = [rand((s.n, h, d), i).to(dtype).requires_grad_(True) for i in (1, 2, 3)]
    do = rand((s.n, h, d), 4).to(dtype)
    plan.plan_cache.clear()
    native = plan.PlanCache.native

    def run(ops):
        o = chain(ops, s, *x)
        return (o.detach(),) + torch.autograd.grad(o, x, do)

    functions = (op.MaskedMMCSR.apply, op.SparseSoftmax.apply, op.VectorSPMM.apply)
    calls = (op.masked_mm, op.sparse_softmax, op.vec_spmm)
    want = run(functions)
    plan.plan_cache.clear()
    first = run(calls)
    with monkeypatch.context() as known:                          # served from the table, every operator and every backward
        for name in ("maskedmm_csr_forward", "maskedmm_csr_backward", "sparse_softmax_forward", "sparse_softmax_backward", "vector_spmm_forward",
                     "vector_spmm_backward", "prepare_products"):
            known.setattr(graphop, name, lambda *args, **kw: pytest.fail("not in the table"))
        second = run(calls)
        with torch.no_grad():
            third = chain(calls, s, *x)
    assert torch.equal(third, want[0])
    for a, b, c in zip(want, first, second):
        assert torch.equal(a, b) and torch.equal(a, c)
    native.take_used()
    old = graphop.set_tiles(False)                                # a switch: what was chosen under the other one is not used
    try:
        assert not native.take_used()
        off = run(calls)
        assert all(torch.equal(a, b) for a, b in zip(off, run(functions)))
    finally:
        graphop.set_tiles(old)


def test_refused_and_held_as_by_the_autograd_functions():
    import torch.autograd.forward_ad as forward_ad
    from bpt_amd import op
    s = sides("bpt512")
    q, k, v = (rand((s.n, 8, 64), i) for i in (1, 2, 3))
    calls = (op.masked_mm, op.sparse_softmax, op.vec_spmm)
    chain(calls, s, q, k, v)
    chain(calls, s, q, k, v)
    with forward_ad.dual_level():
        for no_grad in (False, True):
            with torch.set_grad_enabled(not no_grad), pytest.raises(RuntimeError):
                op.masked_mm(*s.out, *s.inn, forward_ad.make_dual(k, q), q)
            with torch.set_grad_enabled(not no_grad), pytest.raises(RuntimeError):
                op.vec_spmm(*s.inn, *s.out, rand((s.E, 8), 5), forward_ad.make_dual(v, q))
            with torch.set_grad_enabled(not no_grad), pytest.raises(RuntimeError):
                op.sparse_softmax(*s.inn[:3], forward_ad.make_dual(rand((s.E, 8), 5), rand((s.E, 8), 6)))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: op.masked_mm(*s.out, *s.inn, x, q).sum())(k)
    with pytest.raises(RuntimeError):
        op.masked_mm(*s.out, *s.inn, k.cpu(), q.cpu())
    with pytest.raises(RuntimeError):
        op.masked_mm(*s.out, *s.inn, k.transpose(0, 1), q.transpose(0, 1))
    with pytest.raises(ValueError):
        op.vec_spmm(*s.inn, *s.out, rand((s.E - 1, 8), 5), v)
    packed = []
    x = v.clone().requires_grad_(True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        o = op.vec_spmm(*s.inn, *s.out, rand((s.E, 8), 5), x)
    assert any(t.shape == v.shape for t in packed)
    o = op.vec_spmm(*s.inn, *s.out, rand((s.E, 8), 5), x)
    with torch.no_grad():
        x += 1
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(o, x, q)


def test_first_calls_leave_no_workspace_behind():
    """The second call on a graph is served with workspaces of the allocator's: one kept from the first would lie idle."""
    from bpt_amd import graphop, op, plan
    s = sides("multigraph")
    x = [rand((s.n, 6, 50), i).requires_grad_(True) for i in (1, 2, 3)]
    plan.plan_cache.clear()
    graphop.release_workspaces()
    for _ in range(2):
        o = chain((op.masked_mm, op.sparse_softmax, op.vec_spmm), s, *x)
        torch.autograd.grad(o, x, rand((s.n, 6, 50), 4))
        assert not graphop._SCRATCH
    op.sparse_softmax(*s.inn[:3], rand((s.E,), 5))                # (no native form: what this one asks for is kept for the next)
    assert graphop._SCRATCH
    graphop.release_workspaces()
    graphop.vector_spmm_forward(*s.inn, rand((s.E, 6), 5), x[0].detach())      # nor has a caller of the function itself
    assert graphop._SCRATCH


@pytest.mark.parametrize("limits", [dict(capacity=1), dict(max_bytes=0), dict(max_bytes=1 << 18)])
def test_a_cache_too_small_for_both_sides_builds_neither_for_nothing(limits):
    from bpt_amd import op, plan
    s = sides("bpt512")
    x = [rand((s.n, 8, 64), i).requires_grad_(True) for i in (1, 2, 3)]
    calls = (op.masked_mm, op.sparse_softmax, op.vec_spmm)
    plan.plan_cache.clear()
    want = chain(calls, s, *x)
    old = plan.plan_cache.set_limits(**limits)
    try:
        plan.plan_cache.clear()
        built = plan.plan_cache.misses
        got = chain(calls, s, *x)
        assert plan.plan_cache.misses == built + 3                # one for each operator
    finally:
        plan.plan_cache.set_limits(*old)
        plan.plan_cache.clear()
    assert torch.equal(got, want)


def test_a_plan_that_does_not_cover_every_edge_is_built_once():
    """Two slots with one edge id: the operators on tiles do not take such a graph."""
    from bpt_amd import op, plan
    from test_gpu_product_tiles import product_ok, sum_ok
    s = sides("bpt512")

    def twice(side):
        row, indptr, eid, indices = side
        eid = eid.clone()
        eid[eid == 1] = 0
        return row, indptr, eid, indices

    out, inn = twice(s.out), twice(s.inn)
    k, q, w = rand((s.n, 8, 64), 1), rand((s.n, 8, 64), 2), rand((s.E, 8), 3)
    one_weight = w.clone()
    one_weight[1] = w[0]
    distinct = torch.arange(s.E, device=DEV) > 1                  # (edge 0 is written by two slots, edge 1 by none)
    for grad in (False, True):
        plan.plan_cache.clear()
        built = plan.plan_cache.misses
        e = op.masked_mm(*out, *inn, k.requires_grad_(grad), q)
        assert product_ok(e[distinct], k[s.src[distinct]], q[s.dst[distinct]]) and not e[1].any()
        assert sum_ok(op.vec_spmm(*inn, *out, w, k), s.dst, one_weight, k.detach()[s.src], s.n)
        assert plan.plan_cache.misses == built + 2
    dk, = torch.autograd.grad(e, k, w)
    assert sum_ok(dk, s.src, one_weight, q[s.dst], s.n)


def test_rows_cut_into_many_empty_units():
    """More units than rows and edges together, which the builder on the GPU has no room for: the host's takes them."""
    from bpt_amd import op, plan
    s = sides("bpt512")
    x = [rand((s.n, 8, 64), i).requires_grad_(True) for i in (1, 2, 3)]
    do = rand((s.n, 8, 64), 4)
    calls = (op.masked_mm, op.sparse_softmax, op.vec_spmm)

    def cut(side):
        row, indptr, eid, indices = side
        more = s.E + s.n
        return torch.cat([row[:1].expand(more), row]), torch.cat([indptr[:1].expand(more), indptr]), eid, indices

    class Cut:
        out, inn = cut(s.out), cut(s.inn)

    plan.plan_cache.clear()
    runs = []
    for g in (s, Cut):
        o = chain(calls, g, *x)
        runs.append((o.detach(),) + torch.autograd.grad(o, x, do))
    for a, b in zip(*runs):
        assert ((a - b).norm() <= 1e-6 * a.norm()).all()          # (other groups of rows, other orders of the same float32 sums)
