"""Plan caches with room for fewer plans than a training pass asks for: what a pass prepares or leaves for the next one builds no plan a second time."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def graph(length, k=4):
    from bpt_amd import graphbuilder as gb
    src, dst, etype, _, n = gb.merge_graphs_device([gb.BinaryPartition(length, True, k, 10)], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    return (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]), etype, n


def training_pass(args, etype, x, table):
    from bpt_amd import op
    rel = {} if table is None else dict(rel_table=table, etype=etype)
    o = op.bpt_attention(*args, *x, **rel)
    torch.autograd.grad(o, list(x) + ([] if table is None else [table]), torch.ones_like(o))


@pytest.fixture
def cache_of():
    from bpt_amd import op, plan
    old = plan.plan_cache.set_limits()
    def limit(**limits):
        plan.plan_cache.clear()
        op._rel_aux_cache.clear()
        plan.plan_cache.set_limits(**limits)
        return plan.plan_cache
    yield limit
    plan.plan_cache.set_limits(*old)


def built(cache, passes, call):
    before = cache.misses
    for _ in range(passes):
        call()
    return (cache.misses - before) / passes


def test_relative_positions_with_two_plans(cache_of):
    """Three plans (both sides, the term's gradient), each built once a pass; with room for three, none once they are there."""
    args, etype, n = graph(700)
    x = [torch.randn(n, 8, 64, device=DEV, requires_grad=True) for _ in range(3)]
    table = torch.randn(1000, 64, device=DEV, requires_grad=True)
    for capacity, most in ((2, 3), (3, 0)):
        cache = cache_of(capacity=capacity)
        training_pass(args, etype, x, table)
        assert built(cache, 4, lambda: training_pass(args, etype, x, table)) == most


def test_relative_positions_with_room_for_two_plans_bytes(cache_of):
    """The same where what stands in the way are bytes: what both sides' plans hold, and some more than that of the third."""
    args, etype, n = graph(700)
    x = [torch.randn(n, 8, 64, device=DEV, requires_grad=True) for _ in range(3)]
    table = torch.randn(1000, 64, device=DEV, requires_grad=True)
    cache = cache_of(capacity=64)
    training_pass(args, etype, x, table)
    held = [p.device_bytes() for p, _ in cache._d.values()]
    assert len(held) == 3
    for room, most in ((sum(held) - 1, 3), (sum(held), 0)):
        cache = cache_of(max_bytes=room)
        training_pass(args, etype, x, table)
        assert built(cache, 4, lambda: training_pass(args, etype, x, table)) <= most


@pytest.mark.parametrize("capacity", [1, 2])
def test_new_small_graphs(cache_of, capacity):
    """A new graph that is left to the kernels that walk rows: one plan for each side, with room for one as with room for both."""
    cache = cache_of(capacity=capacity)
    x = None

    def call():
        nonlocal x
        args, etype, n = graph(50)
        x = [torch.randn(n, 8, 64, device=DEV, requires_grad=True) for _ in range(3)]
        training_pass(args, etype, x, None)

    call()
    assert built(cache, 4, call) == 2
