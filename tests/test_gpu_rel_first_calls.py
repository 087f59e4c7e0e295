"""The first call of a graph, shape and type with relative positions, which leaves the later ones to the native host path: it may be captured into a
graph where its plans and index tensors are at hand, its forward waits for nothing that it has queued, and only calls that ran on the tiles
leave anything."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def graph(length, k=4):
    from bpt_amd import graphbuilder as gb
    src, dst, etype, _, n = gb.merge_graphs_device([gb.BinaryPartition(length, True, k, 10)], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    return (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]), etype, n


def inputs(n, h, d, dtype):
    gen = torch.Generator().manual_seed(1)
    x = [torch.randn(n, h, d, generator=gen).to(dtype).to(DEV) for _ in range(4)]
    table = (torch.randn(1000, d, generator=gen) * 0.1).to(dtype).to(DEV)
    return [t.requires_grad_(True) for t in x[:3]], table.requires_grad_(True), x[3]


def forget_all():
    from bpt_amd import op, plan
    plan.plan_cache.clear()
    op._rel_aux_cache.clear()


def known(args, q, k, v, p, table, etype):
    from bpt_amd._native import native
    return native.rel_attention(*args, q, k, v, 0.125, p, 7, table, etype) is not None


@pytest.mark.parametrize("h,d,dtype", [(8, 64, torch.float32), (16, 64, torch.bfloat16), (6, 50, torch.float32)])
@pytest.mark.parametrize("why", ["dropout", "cleared"])
def test_a_first_call_under_capture(h, d, dtype, why):
    """Warmed up without dropout and captured with it; and warmed up, but forgotten since by a switch set and set back, which leaves plans and
    index tensors."""
    from bpt_amd import graphop, op
    forget_all()
    args, etype, n = graph(300)
    (q, k, v), table, do = inputs(n, h, d, dtype)
    p = 0.2 if why == "dropout" else 0.0

    def run(p):
        o = op.bpt_attention(*args, q, k, v, dropout_p=p, seed=7, rel_table=table, etype=etype)
        return (o,) + torch.autograd.grad(o, (q, k, v, table), do)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run(0.0)
    torch.cuda.current_stream().wait_stream(side)
    if why == "cleared":
        graphop.set_tiles(graphop.set_tiles(False))
    captured = torch.cuda.CUDAGraph()
    with torch.cuda.graph(captured):
        outs = run(p)
    for i in range(4):
        with torch.no_grad():
            q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(40 + i)).to(DEV))
        want = [x.clone() for x in run(p)]
        captured.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(want, outs))


@pytest.mark.parametrize("train", [True, False])
def test_a_new_graphs_forward_waits_for_none_of_its_kernels(train, monkeypatch):
    """Long products are queued in front of the attention's kernels, behind all that a new graph's plans and index tensors wait for: they still
    run when the call returns, and the next call is known."""
    from bpt_amd import graphop, op
    forget_all()
    args, etype, n = graph(1500)
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)
    big = torch.randn(8192, 8192, device=DEV)
    big @ big
    torch.cuda.synchronize()
    real, behind = graphop.attention_forward, torch.cuda.Event()

    def slow(*a, **kw):
        for _ in range(12):                                       # (12 x 1.1 TFLOP in float32: 80 ms and more)
            big @ big
        behind.record()
        return real(*a, **kw)

    monkeypatch.setattr(graphop, "attention_forward", slow)
    with torch.set_grad_enabled(train):
        o = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
        assert not behind.query()
    monkeypatch.undo()
    torch.cuda.synchronize()
    with torch.no_grad():
        assert known(args, q, k, v, 0.0, table, etype)
        again = op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    assert torch.equal(o, again)


def test_a_forward_alone_builds_no_plan_of_the_backward():
    """Inference with parameters that would have gradients: both sides' tile plans, without the gradient's."""
    from bpt_amd import op, plan
    args, etype, n = graph(700)
    (q, k, v), table, _ = inputs(n, 8, 64, torch.float32)
    held = {}
    for train in (False, True):
        forget_all()
        with torch.set_grad_enabled(train):
            op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
        held[train] = len(plan.plan_cache.held())
        with torch.no_grad():
            assert known(args, q, k, v, 0.0, table, etype)
    assert held == {False: 2, True: 3}


def test_calls_off_the_tiles_leave_nothing(monkeypatch):
    from bpt_amd import graphop, op
    forget_all()
    args, etype, n = graph(300)
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)
    left, real = [], graphop.remember_rel
    monkeypatch.setattr(graphop, "remember_rel", lambda *a: left.append(real(*a)))
    call = lambda: op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    call()
    assert len(left) == 1
    old = graphop.set_tiles(False)
    try:
        call()
        assert len(left) == 1
    finally:
        graphop.set_tiles(old)


def test_index_tensors_made_under_capture_are_not_kept():
    """Captured first, then run eagerly before any replay has filled them."""
    from bpt_amd import op
    from bpt_amd._native import native
    forget_all()
    args, etype, n = graph(300)
    (q, k, v), table, do = inputs(n, 8, 64, torch.float32)
    run = lambda: op.bpt_attention(*args, q, k, v, rel_table=table, etype=etype)
    with torch.no_grad():
        want = run()
        aux = next(iter(op._rel_aux_cache.values()))
        del aux["rows_slot"]                                      # (as after a call whose term was not in the order of the tiles)
        native.clear()
        torch.cuda.synchronize()
        captured = torch.cuda.CUDAGraph()
        with torch.cuda.graph(captured):
            out = run()
        assert "rows_slot" not in aux
        assert torch.equal(run(), want)
        for _ in range(3):
            out.zero_()
            captured.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
