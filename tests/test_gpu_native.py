"""The native host path (bpt_amd/csrc/bptop.cpp): a call served from its table gives the bits of the call that was remembered, a
changed or dropped plan is not served, refused arguments raise as before, threads with streams of their own agree."""
import threading
import time

import numpy as np
import pytest
import torch

from test_gpu_parity import DEV, Case, rand

pytestmark = pytest.mark.gpu


def args_of(c):
    return (*c.out, *c.inn)


def step(op, args, q, k, v, do, p=0.0):
    q, k, v = (x.detach().requires_grad_(True) for x in (q, k, v))
    o = op.bpt_attention(*args, q, k, v, dropout_p=p, seed=7)
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))


def node_tensors(n, dtype=torch.float32, h=8):
    return tuple(rand((n, h, 64), dtype, s, 1.0 / 8).to(DEV) for s in (1, 2, 3, 4))


def same(a, b):
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("gname", ["bpt512_k4", "multigraph"])
def test_served_calls_equal_the_remembered_one(gname, dtype, p):
    from bpt_amd import op, plan
    c = Case(gname)
    x = node_tensors(c.n, dtype)
    plan.plan_cache.clear()
    first = step(op, args_of(c), *x, p)
    assert plan.PlanCache.native.take_used()
    assert same(first, step(op, args_of(c), *x, p))
    assert plan.PlanCache.native.take_used(), "the second call was not served natively"
    with torch.no_grad():
        assert torch.equal(first[0], op.bpt_attention(*args_of(c), *x[:3], dropout_p=p, seed=7))
    plan.plan_cache.clear()
    assert not plan.PlanCache.native.take_used()
    assert same(first, step(op, args_of(c), *x, p))


def test_changed_graphs_and_dropped_plans_are_not_served():
    from bpt_amd import op, plan
    c = Case("bpt512_k4")
    x = node_tensors(c.n)
    args = [t.clone() for t in args_of(c)]
    first = step(op, args, *x)
    assert same(first, step(op, args, *x))
    # other neighbours, written into the same memory: every edge's source moved by one node, on both sides
    src, dst = (np.asarray(c.src) + 1) % c.n, np.asarray(c.dst)
    from bpt_amd import graphbuilder as gb
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, c.n)
    args[7].copy_(in_csr[1].to(DEV))                       # the in-CSR's shape is the same, its columns are not
    moved = (ROW, IR, out_csr[2], out_csr[1])
    args[:4] = [t.to(DEV) for t in moved]
    fresh = [t.clone() for t in args]
    changed = step(op, args, *x)
    assert not torch.equal(changed[0], first[0])
    assert same(changed, step(op, fresh, *x))
    # a cache of one plan drops one of the two sides all the time
    old = plan.plan_cache.set_limits(capacity=1)
    try:
        assert same(changed, step(op, args, *x)) and same(changed, step(op, args, *x))
        assert len(plan.plan_cache._d) == 1
    finally:
        plan.plan_cache.set_limits(*old)


def test_a_known_graph_still_refuses_wrong_arguments():
    from bpt_amd import graphop, op
    c = Case("bpt512_k4")
    q, k, v, do = node_tensors(c.n)
    step(op, args_of(c), q, k, v, do)
    for bad in ((q, k[:, :, :32].contiguous(), v), (q, k, v[:-1].contiguous()), (q, k.bfloat16(), v), (q, k.transpose(0, 1).contiguous().transpose(0, 1), v),
                (q, k.cpu(), v)):
        with pytest.raises((ValueError, RuntimeError)):
            op.bpt_attention(*args_of(c), *bad)
    with pytest.raises((ValueError, RuntimeError)):
        graphop.attention_forward(*c.inn[:3], c.inn[3][:-1].contiguous(), q, k, v)
    o, lse = graphop.attention_forward(*c.inn, q, k, v)
    with pytest.raises(ValueError):
        graphop.attention_backward(*c.out, *c.inn, q, k, v, o, lse[:-1].contiguous(), do)


@pytest.mark.parametrize("h,d", [(8, 64), (6, 50)])
def test_a_malformed_out_side_is_refused_by_the_backward(h, d, monkeypatch):
    """The forward reads the in-side alone, also where both sides' plans are built with it."""
    from bpt_amd import graphop, op, plan
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    c = Case("bpt512_k4")
    q, k, v, do = (rand((c.n, h, d), torch.float32, s, 1.0 / 8).to(DEV) for s in (1, 2, 3, 4))
    q.requires_grad_(True)
    plan.plan_cache.clear()
    with torch.no_grad():
        want = op.bpt_attention(*args_of(c), q, k, v)
    for side, place in ((0, 3), (1, 7)):
        args = [t.clone() for t in args_of(c)]
        args[place][5] = c.n                                  # (a column that is no node: the builder's check refuses it)
        plan.plan_cache.clear()
        if side == 1:
            with pytest.raises(ValueError, match="out of range"):
                op.bpt_attention(*args, q, k, v)
            continue
        o = op.bpt_attention(*args, q, k, v)
        assert torch.equal(o, want)
        with pytest.raises(ValueError, match="out of range"):
            torch.autograd.grad(o, q, do)


@pytest.mark.parametrize("h,d", [(8, 64), (6, 50)])
def test_a_forward_does_without_the_out_side(h, d, monkeypatch):
    """None in place of the out-CSR's tensors: only a backward reads them, also where gradients are recorded."""
    from bpt_amd import graphop, op, plan
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    c = Case("bpt512_k4")
    q, k, v, do = (rand((c.n, h, d), torch.float32, s, 1.0 / 8).to(DEV) for s in (1, 2, 3, 4))
    with torch.no_grad():
        want = op.bpt_attention(*args_of(c), q, k, v)
    for known in (False, True):
        if not known:
            plan.plan_cache.clear()
        with torch.no_grad():
            got = op.bpt_attention(None, None, None, None, *c.inn, q, k, v)
        o = op.bpt_attention(None, None, None, None, *c.inn, q.detach().requires_grad_(True), k, v)
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-6)
        torch.testing.assert_close(o, want, rtol=1e-5, atol=1e-6)


def test_threads_and_streams():
    from bpt_amd import op
    c = Case("bpt512_k4")
    x = node_tensors(c.n)
    want = step(op, args_of(c), *x)
    torch.cuda.synchronize()
    failures = []

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got = step(op, args_of(c), *x)
                stream.synchronize()
                if not same(want, got):
                    failures.append(1)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


@pytest.mark.parametrize("tiles", [False, True], ids=["by-size", "tiles"])
def test_threads_that_build_the_same_graph_at_once(tiles, monkeypatch):
    """From an empty cache, every thread on a stream of its own; then another graph of the same sizes, in memory that the first one's
    index tensors may have left."""
    from bpt_amd import graphbuilder as gb, graphop, op, plan
    if tiles:
        monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    c = Case("bpt512_k4")
    x = node_tensors(c.n)
    want = [step(op, args_of(c), *x)]
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs((np.asarray(c.src) + 1) % c.n, np.asarray(c.dst), c.n)
    other = tuple(t.to(DEV) for t in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))
    want.append(step(op, other, *x))
    torch.cuda.synchronize()
    failures = []

    def work(args, expected, start):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            start.wait()
            for _ in range(2):
                got = step(op, args, *x)
                stream.synchronize()
                if not same(expected, got):
                    failures.append(1)

    for i in range(12):
        plan.plan_cache.clear()
        args = [t.clone() for t in (args_of(c), other)[i % 2]]
        torch.cuda.synchronize()
        start = threading.Barrier(4)
        threads = [threading.Thread(target=work, args=(args, want[i % 2], start)) for _ in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        del args
    assert not failures


def allocated_at_rest():
    """Bytes allocated once autograd's thread has let go of the last step (it drops its reference to the gradients after handing them
    over, which the caller does not wait for)."""
    seen = []
    for _ in range(25):
        seen.append(torch.cuda.memory_allocated())
        time.sleep(0.002)
    return min(seen)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("h,d", [(8, 64), (6, 50)])
def test_no_workspace_lies_idle_beside_that_of_served_calls(h, d, dtype):
    """What a step leaves allocated is its plans, from the first call on; with a score term, whose calls are never served natively, one
    workspace is kept."""
    from bpt_amd import graphbuilder as gb, graphop, op, plan
    g = gb.BinaryPartition(2048, False, 4, 10)
    src, dst, etype, _, n = gb.merge_graphs_device([g], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    args = (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1])
    x = tuple(rand((n, h, d), dtype, s, 1.0 / 8).to(DEV) for s in (1, 2, 3, 4))
    plan.plan_cache.clear()
    graphop.release_workspaces()
    held = []
    for _ in range(3):
        step(op, args, *x)
        held.append(allocated_at_rest())
    assert not graphop._SCRATCH and held[0] == held[1] == held[2]
    if d == 64:
        q = x[0].clone().requires_grad_(True)
        o = op.bpt_attention(*args, q, *x[1:3], rel_table=torch.zeros(1000, d, dtype=dtype, device=DEV), etype=etype)
        torch.autograd.grad(o, q, x[3])
        assert len(graphop._SCRATCH) == 1
    graphop.release_workspaces()


@pytest.mark.parametrize("h,d", [(8, 64), (6, 50)])
@pytest.mark.parametrize("when", ["get", "remember"])
def test_a_choice_made_before_a_switch_changed_is_not_remembered(when, h, d, monkeypatch):
    """Another thread changes a switch or a setting between the moment a call looks and the moment its choice is put into the table."""
    from bpt_amd import graphop, op, plan
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    c = Case("bpt512_k4")
    x = tuple(rand((c.n, h, d), torch.float32, s, 1.0 / 8).to(DEV) for s in (1, 2, 3, 4))
    native = plan.PlanCache.native
    original = getattr(plan.plan_cache, when)
    for change in (lambda: graphop.set_tiles(False), lambda: setattr(graphop, "_MIN_GROUP_ITEMS", 10 ** 9)):
        def meanwhile(*args, **kw):
            if when == "remember":
                change()
                return original(*args, **kw)
            result = original(*args, **kw)
            change()
            return result

        plan.plan_cache.clear()
        setattr(plan.plan_cache, when, meanwhile)
        try:
            step(op, args_of(c), *x)
            served = native.take_used()              # (before the switches are put back, which clears the table)
        finally:
            delattr(plan.plan_cache, when)
            graphop.set_tiles(True)
            graphop._MIN_GROUP_ITEMS = 0
        assert not served


def test_an_entry_holds_its_index_tensors():
    """Their addresses are the key: nothing else may come to lie there while the entry stands."""
    import ctypes
    from bpt_amd import graphop, plan
    native = plan.PlanCache.native
    native.clear()
    struct, before = graphop.PlanStruct(), torch.cuda.memory_allocated()
    index = [torch.zeros(1 << 20, dtype=torch.int64, device=DEV) for _ in range(4)]
    held = torch.cuda.memory_allocated()
    assert native.remember(native.generation(), native.ATTN_FWD, index, [1, 1, 8, 64, 0, 0], ctypes.addressof(struct), 0, (object(),))
    del index
    assert torch.cuda.memory_allocated() == held
    native.clear()
    assert torch.cuda.memory_allocated() == before


@pytest.mark.parametrize("h,d", [(8, 64), (6, 50)])
def test_transforms_that_need_the_autograd_function(h, d):
    """A tangent is refused, not dropped, also where no gradient is asked for; a trace runs the layer again on other inputs."""
    import torch.autograd.forward_ad as forward_ad
    from bpt_amd import op
    c = Case("bpt512_k4")
    q, k, v = (rand((c.n, h, d), torch.float32, s).to(DEV) for s in (1, 2, 3))
    op.bpt_attention(*args_of(c), q, k, v)
    with forward_ad.dual_level():
        for no_grad in (False, True):
            with torch.set_grad_enabled(not no_grad), pytest.raises(RuntimeError):
                op.bpt_attention(*args_of(c), q, forward_ad.make_dual(k, q), v)
    traced = torch.jit.trace(lambda x: op.bpt_attention(*args_of(c), x, k, v), (q,), check_trace=False)
    other = v.clone()
    torch.testing.assert_close(traced(other), op.bpt_attention(*args_of(c), other, k, v), rtol=1e-5, atol=1e-6)
