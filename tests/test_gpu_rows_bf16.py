"""Bfloat16 heads of 64 columns whose tiles one wavefront walks (rows through LDS for both kinds of product), against the float64 oracle:
entry lists of every length around a block and around a piece of a list on either side, rows in one piece and split rows, with dropout,
heads that take one, two and four workgroups a tile.  (The same kernels in two and four parts: test_gpu_tile_parts.py; with a
score term: test_gpu_rel_pos.py.)  Dropout on lists of the destination side has a test of its own: a query row that one pair is left of
has no gradient in q and k but for the rounding of its bfloat16 result, which a bound by the gradients' size does not hold."""
import ctypes
import math

import pytest
import torch
import test_gpu_tile_parts as tiles

SIZES = ((400, 8), (200, 16), (640, 4))
CASES = [(n_tiles, flip, heads, 64, tiles.BF16, p, seg, 1, 1) for n_tiles, heads in SIZES
         for flip, p, seg in ((False, 0.0, 256), (True, 0.0, 256), (False, 0.0, 32), (True, 0.25, 32))]


@pytest.mark.gpu
@pytest.mark.parametrize("n_tiles,flip,heads,d,dtype,p,seg,parts_dst,parts_src", CASES)
def test_rows_through_lds_match_the_oracle(n_tiles, flip, heads, d, dtype, p, seg, parts_dst, parts_src, monkeypatch):
    tiles.test_tiles_in_parts_match_the_oracle(n_tiles, flip, heads, d, dtype, p, seg, parts_dst, parts_src, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("seg", [256, 32])
@pytest.mark.parametrize("n_tiles,heads", SIZES)
def test_dropout_on_lists_of_the_destination_side(n_tiles, heads, seg, monkeypatch):
    """Every element against 64 bits, within what the roundings to bfloat16 (2^-8 of a value) allow: of the probabilities and of ds where they
    enter a product, of o where it stands for itself in delta = dO . o, and of the result."""
    from bpt_amd import _lib, graphop, op, plan
    from bpt_amd import graphbuilder as gb
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    monkeypatch.setattr(graphop, "TILE_SEG_LEN", seg)
    plan.plan_cache.clear()
    src, dst, n_k, n_q = tiles.blocky_graph(n_tiles, False)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    args = tuple(x.to(tiles.DEV) for x in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(29)
    rand = lambda n, s: (torch.randn(n, heads, 64, generator=gen) * s).to(tiles.DEV, torch.bfloat16)
    q, do, k, v = rand(n_q, 1), rand(n_q, 1 / 8), rand(n_k, 1), rand(n_k, 1)
    leaves = [x.requires_grad_(True) for x in (q, k, v)]
    o = op.bpt_attention(*args, *leaves, dropout_p=0.25, seed=11)
    got = (o.detach(),) + torch.autograd.grad(o, leaves, do)
    for pl, _ in plan.plan_cache._d.values():
        hit, = [hit for key, hit in pl._groups.items() if key[0] == 16]
        assert _lib.attn_lib().bpt_wavefronts_per_item(ctypes.byref(hit["struct"]), tiles.SRC if pl.n_rows == n_k else tiles.DST, heads, 64, 2) == 1
        if seg == 256 and pl.n_rows == n_q:
            assert sorted(hit["dev"]["grp_ptr"].diff().tolist()) == sorted(tiles.LENGTHS[t % len(tiles.LENGTHS)] for t in range(n_tiles))
    shape = graphop.attention_padded_shape(q) or (heads, 64)      # (the mask's keys count the heads a layer is padded to)
    like = [torch.empty(n, *shape, dtype=torch.bfloat16) for n in (n_q, n_k)]
    drop = graphop.attention_dropout_mask(*args[4:], *like, 0.25, 11)[:, :heads].double().to(tiles.DEV)
    src, dst = torch.from_numpy(src).to(tiles.DEV), torch.from_numpy(dst).to(tiles.DEV)
    u, scale = 2.0 ** -8, 1 / math.sqrt(64)
    add = lambda n, to, x: torch.zeros((n,) + x.shape[1:], dtype=torch.float64, device=tiles.DEV).index_add_(0, to, x)
    for h in range(heads):
        Q, K, V, D = (x.detach()[:, h].double() for x in (q, k, v, do))
        s = (Q[dst] * K[src]).sum(1) * scale
        e = torch.exp(s - torch.zeros(n_q, dtype=torch.float64, device=tiles.DEV).scatter_reduce(0, dst, s, "amax", include_self=False)[dst])
        p, m = e / add(n_q, dst, e)[dst], drop[:, h]
        O, size_o = (add(n_q, dst, (p * m).unsqueeze(1) * f(V)[src]) for f in (lambda x: x, torch.abs))
        ds = p * ((D[dst] * V[src]).sum(1) * m - (D * O).sum(1)[dst]) * scale
        of_delta = p * (D * O).abs().sum(1)[dst] * scale          # what a relative error of o makes of ds
        want = (O, add(n_q, dst, ds.unsqueeze(1) * K[src]), add(n_k, src, ds.unsqueeze(1) * Q[dst]), add(n_k, src, (p * m).unsqueeze(1) * D[dst]))
        loose = (ds.abs() + of_delta).unsqueeze(1)
        size = (size_o, add(n_q, dst, loose * K[src].abs()), add(n_k, src, loose * Q[dst].abs()), add(n_k, src, (p * m).unsqueeze(1) * D[dst].abs()))
        for name, x, w, z in zip(("o", "dq", "dk", "dv"), got, want, size):
            off = (x[:, h].double() - w).abs() - (1.02 * u * (z + w.abs()) + 1e-5 * z)      # (2 %: products of two roundings; 1e-5: float32 sums)
            assert (off <= 0).all(), f"{name}, head {h}: {off.max():.2e}"
