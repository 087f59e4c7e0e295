"""The source side of the bfloat16 tile kernels that forms p and ds again instead of reading them back: entry lists that end at, before and
after a block of 16 and a staged piece of 128, fewer edges than rows ((lse, delta) of the rows is then the larger part of the
workspace), rows without edges and split rows on both sides, with and without dropout; float64 oracle, rtol / atol 2e-2 as for
every bfloat16 path (8 significant bits: 2^-8 per rounded operand, three of them in a gradient)."""
import numpy as np
import pytest
import torch

from test_gpu_tiles import BF16_TOL, DEV, check, f64, forced_tiles

pytestmark = pytest.mark.gpu


def graph(name):
    """(src, dst, key nodes, query nodes)"""
    if name == "sparse":                                   # 40 edges among 900 query rows
        rng = np.random.default_rng(1)
        return np.sort(rng.integers(0, 64, 40)), rng.integers(0, 900, 40), 64, 900
    # 16 source rows (one tile) whose list of destinations is `name` entries long, and one row split into work items
    n = int(name)
    src = np.concatenate([np.arange(n) % 16, np.full(n, 3)])
    dst = np.concatenate([np.arange(n), np.arange(n)])
    return src, dst, 40, n + 5


@pytest.mark.parametrize("dropout", [0.0, 0.25])
@pytest.mark.parametrize("heads", [8, 16])
@pytest.mark.parametrize("name", ["sparse", "1", "15", "16", "17", "127", "128", "129", "300"])
def test_pairs_formed_again_match_the_oracle(name, heads, dropout):
    from oracle import torch_ops
    from bpt_amd import graphbuilder as gb
    from bpt_amd import graphop, op
    src, dst, n_k, n_q = graph(name)
    src, dst = src.astype(np.int64), dst.astype(np.int64)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    args = tuple(x.to(DEV) for x in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(31)
    # dO / 8: delta = dO . o is formed from the rounded o, and where a row has one edge p (dO . v - delta) is nothing but that
    # rounding, at most 2^-9 sum |dO| |o| over 64 columns, here 64 x 0.64 / 8 / 0.75 x 2^-9 = 0.013 in ds, 0.013 x scale x |q| (up
    # to 4) = 0.007 in dk (with dO of N(0, 1) it is 0.05, beyond the absolute tolerance)
    q = torch.randn(n_q, heads, 64, generator=gen).to(torch.bfloat16)
    do = (torch.randn(n_q, heads, 64, generator=gen) / 8).to(torch.bfloat16)
    k, v = (torch.randn(n_k, heads, 64, generator=gen).to(torch.bfloat16) for _ in range(2))
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    with forced_tiles(64):
        mask = graphop.attention_dropout_mask(*args[4:], qd, kd, dropout, 77)
        o = op.bpt_attention(*args, qd, kd, vd, fused=True, dropout_p=dropout, seed=77)
        o.backward(do.to(DEV))
        from bpt_amd.plan import plan_cache
        assert [p for p, _ in plan_cache._d.values() if any(key[0] == 16 for key in p._groups)], "the tile kernels did not run"
    ro, rdq, rdk, rdv = torch_ops.attention_fwd_bwd(torch.from_numpy(src), torch.from_numpy(dst), f64(q), f64(k), f64(v), f64(do),
                                                    drop=mask.double() if dropout else None)
    check(o, ro, BF16_TOL, "o")
    for got, want, what, rows in ((qd.grad, rdq, "dq", dst), (kd.grad, rdk, "dk", src), (vd.grad, rdv, "dv", src)):
        # a row of a gradient sums one rounded term per edge of its own: BF16_TOL up to 16 of them (every row of dq has one or two,
        # or 40 / 900 on average), beyond that its absolute part grows with the square root of the row's number of edges
        terms = torch.from_numpy(np.bincount(rows, minlength=want.shape[0])).double()[:, None, None]
        err, bound = (f64(got) - want).abs(), 2e-2 * want.abs() + 2e-2 * (terms / 16).clamp(min=1.0).sqrt()
        assert got.shape == want.shape and bool((err <= bound).all()), f"{what}: {float((err / bound).max()):.2f} times its bound"


@pytest.mark.parametrize("dropout", [0.0, 0.25])
@pytest.mark.parametrize("rel", [False, True], ids=["plain", "rel"])
@pytest.mark.parametrize("name", ["sparse", "17", "300"])
def test_the_backward_stays_inside_its_workspace(name, rel, dropout, monkeypatch):
    """The workspace holds (lse, delta) of the rows without a score term and (p, ds) of the pairs with one, and the split rows' sums."""
    from bpt_amd import graphbuilder as gb
    from bpt_amd import graphop, op
    from bpt_amd.plan import plan_cache
    src, dst, n_k, n_q = graph(name)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    args = tuple(x.to(DEV) for x in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))
    q, k, v = (torch.randn(n, 8, 64, device=DEV).to(torch.bfloat16).requires_grad_(True) for n in (n_q, n_k, n_k))
    real, behind = graphop._workspace, []

    def with_a_mark_behind(*a, **kw):
        n = real(*a, **kw)[1]
        buf = torch.full((n + 65536,), 0x5A, dtype=torch.uint8, device=DEV)
        behind.append(buf[n:])
        return (buf, n) if n else (None, 0)

    monkeypatch.setattr(graphop, "_workspace", with_a_mark_behind)
    plan_cache.clear()
    rel_kw = dict(rel_table=torch.randn(5, 64, device=DEV).to(torch.bfloat16), etype=torch.arange(len(src), device=DEV) % 5) if rel else {}
    with forced_tiles(64):
        o = op.bpt_attention(*args, q, k, v, fused=True, dropout_p=dropout, seed=77, **rel_kw)
        o.backward(torch.randn_like(o))
    torch.cuda.synchronize()
    assert len(behind) >= 2 and all(bool((x == 0x5A).all()) for x in behind)
