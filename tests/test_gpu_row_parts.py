"""The kernels that walk single rows, with four or eight wavefronts a work item (small graphs): rows of every length around a batch
and around a wavefront's share, split rows, rows without edges, against the float64 oracle; one path for each size of graph, the
same bits on every run; an infinite row reaches its neighbours and nobody else."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DEGREES = [0, 1, 2, 3, 4, 5, 7, 8, 9, 12, 13, 15, 16, 17, 20, 28, 29, 31, 32, 33, 48, 49, 60, 61, 63, 64, 65, 96, 128, 129, 200, 0]


def graph(n):
    from bpt_amd import graphbuilder as gb
    rng = np.random.default_rng(n)
    deg = np.array([DEGREES[i % len(DEGREES)] for i in range(n)])
    if n not in (33, 128, 800):                                   # (800: the long rows that a float32 forward gives one wavefront each)
        deg = np.minimum(deg, 40)
    dst = np.repeat(np.arange(n), deg)
    src = rng.integers(1, n, len(dst))                            # (node 0 is nobody's neighbour)
    perm = rng.permutation(len(dst))
    src, dst = src[perm].astype(np.int64), dst[perm].astype(np.int64)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, n)
    return src, dst, tuple(x.to(DEV) for x in (ROW, IR, out_csr[2], out_csr[1], COL, IC, in_csr[2], in_csr[1]))


@pytest.mark.parametrize("n", [33, 128, 600, 700, 800, 1000])
@pytest.mark.parametrize("heads,d,dtype", [(8, 64, torch.float32), (16, 64, torch.float32), (4, 64, torch.float32), (8, 32, torch.float32), (8, 64, torch.bfloat16),
                                           (16, 64, torch.bfloat16)])
def test_small_graphs_match_the_oracle(n, heads, d, dtype):
    from oracle import torch_ops
    from bpt_amd import _lib, op, plan
    plan.plan_cache.clear()
    src, dst, args = graph(n)
    gen = torch.Generator().manual_seed(13)
    q, k, v, do = (torch.randn(n, heads, d, generator=gen).to(dtype) for _ in range(4))
    leaves = [x.to(DEV).requires_grad_(True) for x in (q, k, v)]
    runs = []
    for _ in range(2):
        o = op.bpt_attention(*args, *leaves, fused=True)
        runs.append((o.detach(),) + torch.autograd.grad(o, leaves, do.to(DEV)))
    for a, b in zip(*runs):
        assert torch.equal(a, b)
    items = [p.n_items for p, _ in plan.plan_cache._d.values()]
    lib, struct = _lib.attn_lib(), next(iter(plan.plan_cache._d.values()))[0].struct
    want_parts = 8 if n < 289 or (n == 600 and heads * d <= 512) else 1 if n == 800 and dtype == torch.float32 and heads * d >= 512 else 4
    assert lib.bpt_wavefronts_per_item(ctypes.byref(struct), 1, heads, d, 0 if dtype == torch.float32 else 2) == want_parts
    assert max(items) < 1536 and not any(p._groups for p, _ in plan.plan_cache._d.values())       # (rows, not groups of rows)
    f64 = lambda x: x.detach().cpu().double()
    want = torch_ops.attention_fwd_bwd(torch.from_numpy(src), torch.from_numpy(dst), f64(q), f64(k), f64(v), f64(do))
    # float32: sums of at most 10^3 products.  bfloat16: one rounding (2^-9) of each result, and the backward reads the rounded o:
    # its delta = dO . o carries 8 such errors of |dO| |o| into every ds of a row, where p (dO . v - delta) may cancel:
    # errors of a normal kind, the worst of 6e5 five times the typical one of its row, and rows of one or two edges, whose p is near 1,
    # four times the mean row's
    tol = 1e-5 if dtype == torch.float32 else 2 ** -8
    for name, a, b in zip(("o", "dq", "dk", "dv"), runs[0], want[:4]):
        a = f64(a)
        assert (a - b).norm() <= tol * b.norm(), f"{name}: {float((a - b).norm() / b.norm()):.2e}"
        worst = ((a - b).abs() / (b.abs() + b.pow(2).mean().sqrt())).max()
        assert worst <= 20 * tol, f"{name}: {float(worst):.2e}"



@pytest.mark.parametrize("n", [128, 700])
def test_an_infinite_row_reaches_its_neighbours_only(n):
    from bpt_amd import op
    src, dst, args = graph(n)
    q, k, v = (torch.randn(n, 8, 64, device=DEV) for _ in range(3))
    want = op.bpt_attention(*args, q, k, v)
    v2 = v.clone()
    v2[5, 3, 7] = float("inf")
    got = op.bpt_attention(*args, q, k, v2)
    mine = torch.zeros(n, dtype=torch.bool)
    mine[torch.from_numpy(dst[src == 5])] = True
    assert mine.any() and torch.equal(got[~mine], want[~mine])
    assert not got[mine][:, 3, 7].isfinite().any() and torch.equal(got[:, :3], want[:, :3])
