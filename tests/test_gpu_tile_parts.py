"""Tiles whose blocks are shared out over two or four wavefronts of a workgroup (chosen by the number of tiles and of their
blocks) against the float64 oracle: entry lists of every length around a block and around a part's share of the blocks, down to
lists that leave parts without a block, on the destination and on the source side, rows in one piece and split rows, float32 and
bfloat16, with dropout, and heads of fewer than 64 columns."""
import ctypes

import numpy as np
import pytest
import torch

DEV = "cuda:0"
LENGTHS = [0, 1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 81, 127, 128, 129]        # entries of the tiles
DST, SRC = 2, 3                                                                            # kernels, as bptattn_measure.h counts them
F32, BF16 = torch.float32, torch.bfloat16


def blocky_graph(n_tiles, flip):
    """Two node sets: sixteen rows after sixteen share all their neighbours, and nobody else has these, so that the tiles have
    LENGTHS entries.  Rows without edges come first, so that no order by neighbour puts them among the others.  flip: the
    lists are those of the source side."""
    rng = np.random.default_rng(3)
    sizes = sorted(LENGTHS[t % len(LENGTHS)] for t in range(n_tiles))
    at = 16 * sizes.count(0)
    a, b = [], []
    for t, m in enumerate(sizes):
        keep = rng.random((16, m)) < 0.9                          # (a few pairs missing, no neighbour and not the ends)
        keep[:, [0, -1] if m else []] = True
        keep[rng.integers(0, 16, m), np.arange(m)] = True
        r, c = np.nonzero(keep)
        a.append(16 * t + r); b.append(at + c)
        at += m
    a, b = np.concatenate(a).astype(np.int64), np.concatenate(b).astype(np.int64)
    return (a, b, 16 * n_tiles, at) if flip else (b, a, at, 16 * n_tiles)                  # source, destination, how many of each


# tiles, lists of the source side, heads x columns, dtype, dropout, edges per work item, wavefronts per tile and head of the
# destination and of the source side
CASES = [(36, False, 8, 64, F32, 0.0, 256, 4, 2), (36, False, 8, 64, F32, 0.25, 256, 4, 2), (36, True, 8, 64, F32, 0.0, 256, 2, 4),
         (36, False, 8, 64, BF16, 0.0, 256, 4, 2), (36, True, 8, 64, BF16, 0.25, 256, 2, 4), (20, False, 16, 64, F32, 0.0, 32, 4, 2),
         (36, False, 4, 64, F32, 0.0, 32, 4, 4), (36, False, 8, 64, F32, 0.25, 32, 4, 2), (36, True, 8, 64, F32, 0.25, 32, 2, 4),
         (36, False, 8, 64, BF16, 0.0, 32, 4, 2), (36, True, 8, 64, BF16, 0.0, 32, 2, 4), (72, False, 8, 64, BF16, 0.25, 32, 2, 1),
         (180, False, 8, 64, F32, 0.0, 256, 2, 1), (180, True, 8, 64, F32, 0.0, 256, 1, 2), (108, False, 8, 64, BF16, 0.0, 256, 2, 1),
         (144, True, 8, 64, BF16, 0.25, 256, 1, 2), (180, False, 8, 64, F32, 0.25, 32, 1, 1),
         (36, False, 6, 50, F32, 0.25, 256, 4, 4), (36, True, 6, 50, F32, 0.0, 256, 4, 4), (180, True, 6, 50, F32, 0.0, 256, 1, 2),
         (180, False, 6, 50, F32, 0.25, 256, 2, 1), (36, False, 6, 50, F32, 0.25, 32, 4, 4), (72, False, 6, 50, F32, 0.0, 32, 2, 2),
         (36, False, 6, 50, BF16, 0.0, 256, 4, 2), (144, True, 8, 40, BF16, 0.25, 256, 1, 2), (36, True, 6, 50, BF16, 0.25, 32, 2, 4),
         (72, False, 16, 64, F32, 0.25, 256, 2, 1), (250, False, 4, 64, F32, 0.0, 256, 2, 1), (400, False, 8, 64, F32, 0.0, 256, 1, 1)]


@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("n_tiles", sorted({c[0] for c in CASES}))
def test_the_graphs_have_lists_of_every_length(n_tiles, flip):
    """On the CPU, by the model of the plan."""
    import parallel_plan_model as model
    from bpt_amd import graphbuilder as gb
    src, dst, n_k, n_q = blocky_graph(n_tiles, flip)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_k, n_q, as_torch=False)
    side, n_rows, n_index = ((ROW, IR, out_csr), n_k, n_q) if flip else ((COL, IC, in_csr), n_q, n_k)
    base, _ = model.base_plan(side[0], side[1], side[2][2], side[2][1], n_rows, n_index, 256)
    lists = np.diff(model.group_plan(base, n_index, 16, 2)["grp_ptr"])
    assert sorted(lists) == sorted(LENGTHS[t % len(LENGTHS)] for t in range(n_tiles))


@pytest.mark.gpu
@pytest.mark.parametrize("n_tiles,flip,heads,d,dtype,p,seg,parts_dst,parts_src", CASES)
def test_tiles_in_parts_match_the_oracle(n_tiles, flip, heads, d, dtype, p, seg, parts_dst, parts_src, monkeypatch):
    from oracle import torch_ops
    from bpt_amd import _lib, graphop, op, plan
    from bpt_amd import graphbuilder as gb
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    monkeypatch.setattr(graphop, "TILE_SEG_LEN", seg)
    plan.plan_cache.clear()
    src, dst, n_k, n_q = blocky_graph(n_tiles, flip)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    args = tuple(x.to(DEV) for x in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))
    gen = torch.Generator().manual_seed(29)
    q, do = (torch.randn(n_q, heads, d, generator=gen).to(dtype) for _ in range(2))
    k, v = (torch.randn(n_k, heads, d, generator=gen).to(dtype) for _ in range(2))
    do = (do / 8).to(dtype)
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    runs = []
    for _ in range(2):
        o = op.bpt_attention(*args, qd, kd, vd, dropout_p=p, seed=11)
        runs.append((o.detach(),) + torch.autograd.grad(o, (qd, kd, vd), do.to(DEV)))
    for a, b in zip(*runs):
        assert torch.equal(a, b)                                  # parts are added in one order
    sides = {}
    for pl, _ in plan.plan_cache._d.values():
        hits = [hit for key, hit in pl._groups.items() if key[0] == 16]
        assert len(hits) == 1
        sides[SRC if pl.n_rows == n_k else DST] = pl, hits[0]
    lib = _lib.attn_lib()
    parts = [lib.bpt_wavefronts_per_item(ctypes.byref(sides[side][1]["struct"]), side, heads, 64, 0 if dtype == F32 else 2) for side in (DST, SRC)]
    assert parts == [parts_dst, parts_src]
    listed, hit = sides[SRC if flip else DST]
    if seg == 256:
        lists = hit["dev"]["grp_ptr"].diff().tolist()
        assert sorted(lists) == sorted(LENGTHS[t % len(LENGTHS)] for t in range(n_tiles))
    else:
        assert listed.struct.n_heavy > 0
    drop = None
    if p:
        shape = graphop.attention_padded_shape(q) or (heads, d)   # (the mask's keys count the heads a layer is padded to)
        like = [torch.empty(n, *shape, dtype=dtype) for n in (n_q, n_k)]
        drop = graphop.attention_dropout_mask(*args[4:], *like, p, 11)[:, :heads].double()
    f64 = lambda x: x.detach().cpu().double()
    want = torch_ops.attention_fwd_bwd(torch.from_numpy(src), torch.from_numpy(dst), f64(q), f64(k), f64(v), f64(do), drop=drop)
    # float32: sums of at most some 10^3 products of magnitude 1; bfloat16: p and ds rounded to 2^-9 where they enter a product
    tol = 2e-5 if dtype == F32 else 2e-2
    for name, a, b in zip(("o", "dq", "dk", "dv"), runs[0], want[:4]):
        err = (f64(a) - b).norm() / b.norm()
        assert err < tol, f"{name}: {err:.2e}"
        assert ((f64(a) - b).abs() <= tol * 20 * (b.abs() + b.pow(2).mean().sqrt())).all(), name
