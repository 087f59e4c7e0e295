"""Sentences attending to other sentences (two node sets, half of the nodes without edges), whose work items are as long as the
rows, against the float64 oracle: rows below, at and above the lengths of an item.  And two node sets whose nodes all have
edges, whose items are cut by that average."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# (keys, queries) of a sentence pair: rows of 64 | 65, 128 | 129, 256 | 257 edges.  No rows of a single edge: there bfloat16's p (dO . v -
# delta) is nothing but the rounding of o that delta was formed from, 2^-9 sum |dO| |o| = 0.011, which times |k| / 8 is as large as all
# of dq beside it.
@pytest.mark.parametrize("heads,d,dtype,p", [(8, 64, torch.float32, 0.0), (8, 64, torch.bfloat16, 0.1), (6, 50, torch.float32, 0.1)])
@pytest.mark.parametrize("pairs", [[(64, 64), (65, 500), (20, 960)], [(128, 700), (129, 900), (33, 40)], [(257, 950), (256, 641), (40, 3)]],
                         ids=["short", "medium", "long"])
def test_two_node_sets_match_the_oracle(pairs, heads, d, dtype, p):
    from oracle import torch_ops
    from bpt_amd import graphbuilder as gb
    from bpt_amd import graphop, op, plan
    plan.plan_cache.clear()
    bpt = lambda n: gb.BinaryPartition(n, False, 1, 10)
    src, dst, n_k, n_q = gb.inter_graph_edges([bpt(a) for a, _ in pairs], [bpt(b) for _, b in pairs])
    csr = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    out_csr, in_csr, row, ir, col, ic = csr
    args = tuple(x.to(DEV) for x in (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(41)
    q, do = (torch.randn(n_q, heads, d, generator=gen).to(dtype) for _ in range(2))
    k, v = (torch.randn(n_k, heads, d, generator=gen).to(dtype) for _ in range(2))
    do = (do / 8).to(dtype)
    leaves = [x.to(DEV).requires_grad_(True) for x in (q, k, v)]
    o = op.bpt_attention(*args, *leaves, dropout_p=p, seed=11)
    got = (o.detach(),) + torch.autograd.grad(o, leaves, do.to(DEV))
    drop = None
    if p:
        shape = graphop.attention_padded_shape(q) or (heads, d)
        like = lambda n: torch.empty(n, *shape, dtype=dtype)
        drop = graphop.attention_dropout_mask(*args[4:], like(n_q), like(n_k), p, 11)[:, :heads].double()
    f64 = lambda x: x.detach().cpu().double()
    src, dst = (torch.as_tensor(np.asarray(x)) for x in (src, dst))
    want = torch_ops.attention_fwd_bwd(src, dst, f64(q), f64(k), f64(v), f64(do), drop=drop)
    # float32: sums of at most some 10^3 products of magnitude 1; bfloat16: p and ds rounded to 2^-9 where they enter a product
    tol = 2e-5 if dtype == torch.float32 else 2e-2
    for name, a, b in zip(("o", "dq", "dk", "dv"), got, want[:4]):
        assert (f64(a) - b).norm() / b.norm() < tol, name
        assert ((f64(a) - b).abs() <= tol * 20 * (b.abs() + b.pow(2).mean().sqrt())).all(), name


@pytest.mark.parametrize("every,edges,want", [(1, 20, 64), (2, 20, 64), (2, 40, 128), (1, 40, 128), (2, 100, 256)])
def test_items_follow_the_rows_that_have_edges(every, edges, want, monkeypatch):
    """Every or every second row of either side has `edges` edges: the length of the items is the same, and so are the results
    of plans built together and one by one."""
    from oracle import torch_ops
    from bpt_amd import graphbuilder as gb
    from bpt_amd import graphop, op, plan
    n_q, n_k = every * 1600, every * 1601                         # (one source without edges more)
    dst = np.repeat(np.arange(0, n_q, every), edges).astype(np.int64)
    src = ((dst // every + np.tile(np.arange(edges) * 37, n_q // every)) % 1600 * every).astype(np.int64)
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    args = tuple(x.to(DEV) for x in (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(43)
    q, do = (torch.randn(n_q, 8, 64, generator=gen) for _ in range(2))
    k, v = (torch.randn(n_k, 8, 64, generator=gen) for _ in range(2))
    leaves = [x.to(DEV).requires_grad_(True) for x in (q, k, v)]
    runs = []
    for together in (True, False):
        plan.plan_cache.clear()
        if not together:
            monkeypatch.setattr(graphop, "prepare_training", lambda *a, **kw: None)
        o = op.bpt_attention(*args, *leaves)
        runs.append((o.detach(),) + torch.autograd.grad(o, leaves, do.to(DEV)))
        assert [p.seg_len for p, _ in plan.plan_cache._d.values()] == [want] * 2
    for a, b in zip(*runs):
        assert torch.equal(a, b)
    f64 = lambda x: x.detach().cpu().double()
    ref = torch_ops.attention_fwd_bwd(torch.from_numpy(src), torch.from_numpy(dst), f64(q), f64(k), f64(v), f64(do))
    for name, a, b in zip(("o", "dq", "dk", "dv"), runs[0], ref[:4]):
        assert (f64(a) - b).norm() / b.norm() < 2e-5, name        # float32: sums of at most some 10^2 products of magnitude 1


@pytest.mark.parametrize("n", [0, 1, 2, 255, 256, 257, 16383, 16384, 16385, 40000])
def test_rows_with_edges_are_counted(n):
    """Units of rows in one piece and in several, empty ones before, between and behind the others of a row, rows of nothing else."""
    from bpt_amd import plan
    rng = np.random.default_rng(n)
    sides, want = [], []
    for p_empty, p_more in ((0.0, 0.3), (0.6, 0.7)):
        row = np.cumsum(rng.random(n) >= p_more).astype(np.int64) * 3
        size = np.where(rng.random(n) < p_empty, 0, rng.integers(1, 33, n))
        sides.append(tuple(torch.from_numpy(x).to(DEV) for x in (row, np.concatenate([[0], np.cumsum(size)]).astype(np.int64))))
        want.append(len(np.unique(row[size > 0])))
    assert plan.rows_with_edges(sides) == want
    assert plan.rows_with_edges(sides[:1]) == want[:1]
    assert plan.rows_with_edges([tuple(t.cpu() for t in side) for side in sides]) == want


@pytest.mark.parametrize("heads,d", [(8, 64), (6, 50)])
@pytest.mark.parametrize("n_q,n_k", [(3200, 3201), (3200, 3200)])
def test_index_tensors_of_32_bits(n_q, n_k, heads, d):
    """Widened for the plans that are built on the GPU, as the host builder widens them: the same results."""
    from bpt_amd import graphbuilder as gb
    from bpt_amd import op, plan
    rng = np.random.default_rng(7)
    dst = np.repeat(np.arange(n_q), 12).astype(np.int64)
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_bipartite(rng.integers(0, n_k, len(dst)), dst, n_k, n_q)
    args = tuple(x.to(DEV) for x in (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(47)
    q, do = (torch.randn(n_q, heads, d, generator=gen).to(DEV) for _ in range(2))
    k, v = (torch.randn(n_k, heads, d, generator=gen).to(DEV) for _ in range(2))
    leaves = [x.requires_grad_(True) for x in (q, k, v)]
    runs = []
    for graph in (args, tuple(t.to(torch.int32) for t in args)):
        plan.plan_cache.clear()
        o = op.bpt_attention(*graph, *leaves)
        runs.append((o.detach(),) + torch.autograd.grad(o, leaves, do))
    for a, b in zip(*runs):
        assert torch.equal(a, b)
