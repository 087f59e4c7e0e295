"""Sentences attending to other sentences (two node sets, half of the nodes without edges), whose work items are as long as the
rows, against the float64 oracle: rows below, at and above the lengths of an item."""
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
