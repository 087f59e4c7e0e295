"""The edge softmax with its split rows taken whole by workgroups of the launch over the items, against float64: rows of the lengths
around a workgroup's one load (512 threads, eight slots each) and around the longest that goes this way, beside rows of the items;
and the same rows where the plan does not say how long the longest is (segments, merged in launches of their own)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


LIMIT = 1024             # the longest row that is taken whole


def degrees(h):
    """Row lengths around what a workgroup loads at once, up to the longest that goes this way."""
    once = 8 * (512 // (h // 4) if h in (4, 8, 16) else 8 * (64 // h))
    return [d for d in (0, 3, 64, 65, 200, once - 1, once, once + 1, 0, 2 * once + 3, LIMIT - 1, LIMIT) if d <= LIMIT]


@pytest.mark.parametrize("known", [True, False])       # (whether the plan says how long its longest row is)
@pytest.mark.parametrize("h,dtype", [(4, torch.float32), (8, torch.float32), (16, torch.bfloat16), (6, torch.float32), (12, torch.bfloat16), (8, torch.float64), (64, torch.float32)])
def test_whole_rows_match_float64(h, dtype, known):
    from bpt_amd import graphbuilder as gb, graphop, plan
    plan.plan_cache.clear()
    deg = degrees(h)
    n, rng = len(deg), np.random.default_rng(5)
    dst = np.repeat(np.arange(n), deg).astype(np.int64)
    rng.shuffle(dst)
    _, in_csr, _, _, col, ic = gb.get_csrs(rng.integers(0, n, len(dst)).astype(np.int64), dst, n)
    csr = tuple(t.to(DEV) for t in (col, ic, in_csr[2]))
    gen = torch.Generator().manual_seed(6)
    x, dy = (torch.randn(len(dst), h, generator=gen) * s for s in (3, 1))
    x[torch.rand(x.shape, generator=gen) < 0.2] = float("-inf")           # masked scores
    x[[int(np.argmax(dst == r)) for r in range(n) if deg[r]]] = 0.5       # (every row keeps an edge)
    x, dy = x.to(dtype), dy.to(dtype)
    struct = plan.plan_cache.get(*csr, None, None, None, prefer_device=True).struct      # (as the op asks for it)
    assert struct.max_degree == LIMIT and struct.n_heavy == sum(d > 64 for d in deg)
    if not known:
        struct.max_degree = 0
    y = graphop.sparse_softmax_forward(*csr, x.to(DEV))
    dx = graphop.sparse_softmax_backward(*csr, y, dy.to(DEV))
    idx = torch.from_numpy(dst).unsqueeze(1).expand(-1, h)
    xd, yh, dyd = x.double(), y.cpu().double(), dy.double()
    m = torch.full((n, h), -1e9, dtype=torch.float64).scatter_reduce(0, idx, xd, "amax")
    e = torch.exp(xd - m.gather(0, idx))
    want = e / torch.zeros_like(m).scatter_add_(0, idx, e).gather(0, idx)
    dot = torch.zeros_like(m).scatter_add_(0, idx, yh * dyd).gather(0, idx)
    want_dx = yh * (dyd - dot)                                             # (the backward is that of the rounded probabilities)
    # float32: exponentials and a division to some ulp, sums of up to 1024 terms over some hundred partial sums; bfloat16: one rounding of the result
    tol = {torch.float32: 3e-6, torch.bfloat16: 2.0 ** -8, torch.float64: 1e-13}[dtype]
    assert ((yh - want).abs() <= tol * (want + 1e-7)).all()
    assert ((dx.cpu().double() - want_dx).abs() <= tol * (want_dx.abs() + yh * (dyd.abs() + dot.abs() + 1))).all()
    assert torch.equal(y, graphop.sparse_softmax_forward(*csr, x.to(DEV)))
