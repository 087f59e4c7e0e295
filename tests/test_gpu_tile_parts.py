"""Tiles whose blocks are shared out over two or four wavefronts of a workgroup (chosen by the number of tiles and of their
blocks) against the float64 oracle: entry lists of every length around a block and around a part's share of the blocks, down to
lists that leave parts without a block, rows in one piece and split rows, float32 and bfloat16, with dropout, and heads of
fewer than 64 columns."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
LENGTHS = [0, 1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 81, 127, 128, 129]        # entries of the tiles


def blocky_graph(n_tiles):
    """Sixteen rows after sixteen that share all their neighbours: tiles of LENGTHS entries each."""
    rng = np.random.default_rng(3)
    n = 16 * n_tiles
    src, dst = [], []
    for t in range(n_tiles):
        m = LENGTHS[t % len(LENGTHS)]
        cols = np.sort(rng.choice(min(n, 400), m, replace=False)) + max(0, min(16 * t, n - 400))
        rows = np.arange(16 * t, 16 * t + 16)
        keep = rng.random((16, m)) < 0.9                          # (a few pairs missing)
        r, c = np.nonzero(keep)
        dst.append(rows[r]); src.append(cols[c])
    return np.concatenate(src).astype(np.int64), np.concatenate(dst).astype(np.int64), n


# tiles, heads x columns, dtype, dropout, edges per work item, wavefronts per tile and head that the sizes ask for
CASES = [(36, 8, 64, torch.float32, 0.0, 256, 4), (36, 8, 64, torch.float32, 0.25, 256, 4), (36, 8, 64, torch.bfloat16, 0.0, 256, 4),
         (36, 8, 64, torch.bfloat16, 0.25, 256, 4), (20, 16, 64, torch.float32, 0.0, 32, 4), (40, 4, 64, torch.float32, 0.0, 256, 4),
         (144, 8, 64, torch.float32, 0.0, 256, 2), (108, 8, 64, torch.bfloat16, 0.0, 256, 2), (144, 8, 64, torch.float32, 0.25, 256, 2),
         (36, 6, 50, torch.float32, 0.25, 256, 4), (180, 6, 50, torch.float32, 0.0, 256, 2), (36, 6, 50, torch.bfloat16, 0.0, 256, 4),
         (144, 8, 40, torch.bfloat16, 0.25, 256, 2), (400, 8, 64, torch.float32, 0.0, 256, 1)]


@pytest.mark.parametrize("n_tiles,heads,d,dtype,p,seg,parts", CASES)
def test_tiles_in_parts_match_the_oracle(n_tiles, heads, d, dtype, p, seg, parts, monkeypatch):
    from oracle import torch_ops
    from bpt_amd import graphbuilder as gb
    from bpt_amd import graphop, op, plan
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    monkeypatch.setattr(graphop, "TILE_SEG_LEN", seg)
    plan.plan_cache.clear()
    src, dst, n = blocky_graph(n_tiles)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, n)
    args = tuple(x.to(DEV) for x in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(29)
    q, k, v, do = (torch.randn(n, heads, d, generator=gen).to(dtype) for _ in range(4))
    do = (do / 8).to(dtype)
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    runs = []
    for _ in range(2):
        o = op.bpt_attention(*args, qd, kd, vd, dropout_p=p, seed=11)
        runs.append((o.detach(),) + torch.autograd.grad(o, (qd, kd, vd), do.to(DEV)))
    for a, b in zip(*runs):
        assert torch.equal(a, b)                                  # parts are added in one order
    waves = [hit["struct"].n_groups * heads for pl, _ in plan.plan_cache._d.values() for key, hit in pl._groups.items() if key[0] == 16]
    most = {4: 768, 2: 1536, 1: 1 << 30}[parts] if dtype == torch.float32 else {4: 600, 2: 1200, 1: 1 << 30}[parts]
    assert waves and max(waves) <= most                           # (the in-CSR's; the sizes below which a split is certain)
    drop = None
    if p:
        shape = graphop.attention_padded_shape(q) or (heads, d)   # (the mask's keys count the heads a layer is padded to)
        like = torch.empty(n, *shape, dtype=dtype)
        drop = graphop.attention_dropout_mask(*args[4:], like, like, p, 11)[:, :heads].double()
    f64 = lambda x: x.detach().cpu().double()
    want = torch_ops.attention_fwd_bwd(torch.from_numpy(src), torch.from_numpy(dst), f64(q), f64(k), f64(v), f64(do), drop=drop)
    # float32: sums of at most some 10^3 products of magnitude 1; bfloat16: p and ds rounded to 2^-9 where they enter a product
    tol = 2e-5 if dtype == torch.float32 else 2e-2
    for name, a, b in zip(("o", "dq", "dk", "dv"), runs[0], want[:4]):
        err = (f64(a) - b).norm() / b.norm()
        assert err < tol, f"{name}: {err:.2e}"
        assert ((f64(a) - b).abs() <= tol * 20 * (b.abs() + b.pow(2).mean().sqrt())).all(), name
