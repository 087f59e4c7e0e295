"""The tile kernels that read heads of fewer than 64 columns as they are in memory, at the widths where quads of four columns end,
shift or fall away and at head counts that leave a workgroup half empty; against the float64 oracle at the layer's tolerances
(fp32 outputs rtol / atol 1e-5, gradients rtol 1e-4, bf16 2e-2).  Widths they do not take run on padded copies and are checked with
them.  What stands behind the last head must not matter: the rows are views into memory full of NaN."""
import pytest
import torch

import oracle
from test_gpu_parity import DEV, GTOL, TOL, Case, close, f64, rand

pytestmark = pytest.mark.gpu

_cases = {}


def case(name):
    if name not in _cases:
        _cases[name] = Case(name)
    return _cases[name]


def among_nans(x):
    """x as a contiguous view that starts and ends inside a larger buffer of NaN."""
    buf = torch.full((x.numel() + 128,), float("nan"), dtype=x.dtype, device=x.device)
    view = buf[64:64 + x.numel()].view(x.shape)
    view.copy_(x)
    return view


@pytest.mark.parametrize("gname", ["bpt512_k4", "multigraph"])
@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 1, 4), (torch.float32, 3, 5), (torch.float32, 4, 6), (torch.float32, 5, 7), (torch.float32, 6, 50),
                                       (torch.float32, 7, 61), (torch.float32, 9, 63), (torch.float32, 15, 64), (torch.float32, 2, 3),
                                       (torch.bfloat16, 1, 4), (torch.bfloat16, 5, 6), (torch.bfloat16, 6, 50), (torch.bfloat16, 9, 62),
                                       (torch.bfloat16, 3, 64), (torch.bfloat16, 6, 51)],
                         ids=lambda x: str(x).replace("torch.", ""))
def test_narrow_heads_against_the_oracle(gname, dtype, h, d, monkeypatch):
    from bpt_amd import graphop, op
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)       # (tiles whatever the graph's size)
    c = case(gname)
    q, k, v, do = (among_nans(rand((c.n, h, d), dtype, s, 1.0 / 8).to(DEV)) for s in (71, 72, 73, 74))
    for t in (q, k, v):
        t.requires_grad_(True)
    o = op.bpt_attention(*c.out, *c.inn, q, k, v)
    assert o.shape == (c.n, h, d) and o.is_contiguous()
    grads = torch.autograd.grad(o, (q, k, v), do)
    ro, ra = oracle.attention_forward(c.csr, f64(q), f64(k), f64(v))
    want = oracle.attention_backward(c.csr, f64(q), f64(k), f64(v), ra, f64(do))
    close(o, ro, TOL[dtype], "o")
    for got, ref, name in zip(grads, want, ("dq", "dk", "dv")):
        assert got.shape == q.shape
        close(got, ref, GTOL[dtype], name)


@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 6, 50), (torch.float32, 3, 5), (torch.bfloat16, 6, 50)], ids=lambda x: str(x).replace("torch.", ""))
def test_dropout_of_narrow_heads_is_that_of_the_padded_layer(dtype, h, d):
    from bpt_amd import graphop, op
    c = case("bpt512_k4")
    q, k, v, do = (rand((c.n, h, d), dtype, s, 1.0 / 8).to(DEV) for s in (81, 82, 83, 84))
    hp = graphop.attention_padded_shape(q)[0]
    grow = lambda x: torch.nn.functional.pad(x, (0, 64 - d, 0, hp - h))
    both = []
    for narrow in (True, False):
        x = [t.detach().requires_grad_(True) for t in (q, k, v)]
        rows = x if narrow else [grow(t) for t in x]
        o = op.bpt_attention(*c.out, *c.inn, *rows, scale=d ** -0.5, dropout_p=0.3, seed=5)[:, :h, :d]
        both.append((o.detach(), *torch.autograd.grad(o, x, do)))
    # (the same kernels on the same numbers and zeros: sums over the columns differ in nothing but the zeros' places)
    for got, want, name in zip(both[0], both[1], ("o", "dq", "dk", "dv")):
        close(got, f64(want), TOL[dtype] if name == "o" else GTOL[dtype], name)


@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("d", [50, 64])
def test_bfloat16_rows_that_start_on_two_bytes(d, p):
    """Views one element into their memory, the incoming gradient among them: the bits of the same values from their own memory."""
    from bpt_amd import op
    c = case("bpt512_k4")                                     # (with dropout: the kernels that read the rows as they are, whatever the size)
    x = [rand((c.n, 6, d), torch.bfloat16, s, 1.0 / 8).to(DEV) for s in (91, 92, 93, 94)]

    def shifted(t):
        view = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        return view.copy_(t)

    def step(q, k, v, do):
        q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
        o = op.bpt_attention(*c.out, *c.inn, q, k, v, dropout_p=p, seed=3)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))

    for want, got in zip(step(*x), step(*map(shifted, x))):
        assert torch.equal(want, got)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_small_graphs_keep_the_row_kernels(dtype):
    """A layer too small for tiles takes its padded form's kernels: the bits of the padded layer, and a row that is not finite
    reaches its neighbours and no one else."""
    from bpt_amd import graphbuilder as gb, op
    g = gb.BinaryPartition(300, True, 4, 10)
    src, dst, _, _, n = gb.merge_graphs_device([g, g], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    graph = (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1])
    assert col.numel() < 1536
    q, k, v, do = (rand((n, 6, 50), dtype, s, 1.0 / 8).to(DEV) for s in (61, 62, 63, 64))
    q[5] = float("inf")
    grow = lambda x: torch.nn.functional.pad(x, (0, 14, 0, 2))
    both = []
    for rows in (lambda x: x, grow):
        x = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = op.bpt_attention(*graph, *map(rows, x), scale=50 ** -0.5)[:, :6, :50]
        both.append((o.detach(), *torch.autograd.grad(o, x, do)))
    for got, want in zip(*both):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
        assert not got[n // 2:].isnan().any()                  # the second graph


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_a_small_layer_is_the_same_after_one_with_dropout(dtype):
    """Dropout puts a small layer on tiles; the layer without it keeps the row kernels, whichever call came first."""
    from bpt_amd import graphbuilder as gb, graphop, plan
    g = gb.BinaryPartition(300, True, 4, 10)
    src, dst, _, _, n = gb.merge_graphs_device([g], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    out, inn = (row, ir, out_csr[2], out_csr[1]), (col, ic, in_csr[2], in_csr[1])
    q, k, v, do = (rand((n, 6, 50), dtype, s, 1.0 / 8).to(DEV) for s in (51, 52, 53, 54))
    q[5] = float("inf")
    stand_in = torch.empty(n, 8, 64, dtype=dtype, device="meta")

    def layer(p):
        o, lse = graphop.attention_forward(*inn, stand_in, stand_in, stand_in, 50 ** -0.5, p, 3, narrow=(q, k, v))
        return (o, lse[:, :6], *graphop.attention_backward_narrow(*out, *inn, q, k, v, o, lse, do, 8, 50 ** -0.5, p, 3))

    plan.plan_cache.clear()
    cold = layer(0.0)
    layer(0.1)
    for got, want in zip(layer(0.0), cold):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 8, 40), (torch.float32, 6, 50), (torch.float32, 5, 51), (torch.float32, 3, 5), (torch.bfloat16, 8, 40),
                                       (torch.bfloat16, 6, 50)], ids=lambda x: str(x).replace("torch.", ""))
def test_a_mask_column_of_minus_infinity(dtype, h, d, p, monkeypatch):
    """-inf in one of the last columns of some key rows, where the query rows hold one: their edges have probability zero, and what is
    finite, infinite or NaN is what it is on the padded layer's tiles."""
    from bpt_amd import graphop, op
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)       # (tiles whatever the graph's size)
    c = case("bpt512_k4")
    q, k, v, do = (rand((c.n, h, d), dtype, s, 1.0 / 8).to(DEV) for s in (41, 42, 43, 44))
    hp = graphop.attention_padded_shape(q)[0]
    grow = lambda x: torch.nn.functional.pad(x, (0, 64 - d, 0, hp - h))
    masked = torch.arange(0, c.n, 7, device=DEV)
    for col in range(d - 4, d):
        qm, km = q.clone(), k.clone()
        qm[..., col], km[..., col] = 1.0, 0.0
        km[masked, :, col] = float("-inf")
        both = []
        for narrow in (True, False):
            x = [t.detach().requires_grad_(True) for t in (qm, km, v)]
            o = op.bpt_attention(*c.out, *c.inn, *(x if narrow else [grow(t) for t in x]), scale=d ** -0.5, dropout_p=p, seed=5)[:, :h, :d]
            both.append((o.detach(), *torch.autograd.grad(o, x, do)))
        assert both[1][0].isfinite().all() and not both[0][3][masked].any()
        for got, want, name in zip(both[0], both[1], ("o", "dq", "dk", "dv")):
            assert torch.equal(got.isfinite(), want.isfinite()) and torch.equal(got.isnan(), want.isnan()), name
            close(got.nan_to_num(), f64(want.nan_to_num()), TOL[dtype] if name == "o" else GTOL[dtype], name)


@pytest.mark.parametrize("tiles", [True, False], ids=["tiles", "by-size"])
@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 6, 50), (torch.float32, 3, 5), (torch.bfloat16, 6, 50), (torch.bfloat16, 3, 64)],
                         ids=lambda x: str(x).replace("torch.", ""))
def test_rows_and_result_may_be_written_to_after_the_forward(dtype, h, d, tiles, monkeypatch):
    """As on padded copies: the gradients are those of the values that the forward saw."""
    from bpt_amd import graphop, op
    if tiles:
        monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    c = case("bpt512_k4")
    leaves = [rand((c.n, h, d), dtype, s, 1.0 / 8).to(DEV).requires_grad_(True) for s in (21, 22, 23)]
    do = rand((c.n, h, d), dtype, 24, 1.0 / 8).to(DEV)
    want = torch.autograd.grad(op.bpt_attention(*c.out, *c.inn, *leaves), leaves, 2 * do)
    q, k, v = (x * 1 for x in leaves)
    o = op.bpt_attention(*c.out, *c.inn, q, k, v)
    for x in (q, k, v):
        x.add_(1.0)
    o.mul_(2.0)
    for got, ref in zip(torch.autograd.grad(o, leaves, do), want):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 6, 50), (torch.bfloat16, 8, 40)], ids=lambda x: str(x).replace("torch.", ""))
def test_graph_replay_of_a_training_step_equals_eager(dtype, h, d):
    """A captured forward and backward holds the copies of the rows and of the result, too: replayed on new values, with eager work in
    between, it gives the eager step's bits."""
    from bpt_amd import graphop, op
    c = case("bpt512_k4")
    q, k, v, do = (rand((c.n, h, d), dtype, s, 1.0 / 8).to(DEV) for s in (31, 32, 33, 34))
    assert graphop.attention_reads_narrow(c.inn[0], c.inn[2], q, k, graphop.attention_padded_shape(q)[0], 0.1)

    def step():
        x = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = op.bpt_attention(*c.out, *c.inn, *x, dropout_p=0.1, seed=5)
        return (o.detach(), *torch.autograd.grad(o, x, do))

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):                              # plans are built and cached before the capture
        for _ in range(2):
            step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for rep in range(4):
        for t in (q, k, v, do):
            t.mul_(-0.5).add_(0.01 * rep)
        want = step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, ref, name in zip(captured, want, ("o", "dq", "dk", "dv")):
            assert torch.equal(got, ref), f"replay {rep}: {name}"
