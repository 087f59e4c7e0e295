"""The edge softmax and its backward with four heads a lane (4, 8 or 16 heads, float32 and bfloat16) against float64: rows of every
length around what a wavefront holds at once, split rows of few and of many segments, rows without edges, masked and infinite
scores, tensors that start off a 16-byte boundary (which take the kernels of one head a lane)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DEGREES = [0, 1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 511, 513, 1500, 0, 5000]


def graph(order):
    from bpt_amd import graphbuilder as gb
    rng = np.random.default_rng(7)
    dst = np.repeat(np.arange(len(DEGREES)), DEGREES)
    src = rng.integers(0, len(DEGREES), len(dst))
    if order == "shuffled":
        rng.shuffle(dst)                                          # (edge ids of a row scattered)
    n = len(DEGREES)
    _, in_csr, _, _, col, ic = gb.get_csrs(src.astype(np.int64), dst.astype(np.int64), n)
    return torch.from_numpy(dst.astype(np.int64)), n, tuple(t.to(DEV) for t in (col, ic, in_csr[2]))


def reference(dst, n, x, dy):
    x = x.double().requires_grad_(True)
    idx = dst.unsqueeze(1).expand(-1, x.size(1))
    m = torch.full((n, x.size(1)), -1e9, dtype=torch.float64).scatter_reduce(0, idx, x.detach(), "amax")
    e = torch.exp(x - m[dst])
    y = e / torch.zeros_like(m).index_add_(0, dst, e)[dst]
    return y.detach(), torch.autograd.grad(y, x, dy.double())[0]


@pytest.mark.parametrize("order", ["in order", "shuffled"])
@pytest.mark.parametrize("seg", [64, 24, 256])
@pytest.mark.parametrize("h,dtype", [(4, torch.float32), (8, torch.float32), (16, torch.float32), (8, torch.bfloat16), (16, torch.bfloat16), (2, torch.float32)])
def test_softmax_matches_float64(h, dtype, seg, order, monkeypatch):
    from bpt_amd import graphop, plan
    monkeypatch.setattr(plan, "FORCE_SEG_LEN", seg)
    plan.plan_cache.clear()
    dst, n, csr = graph(order)
    gen = torch.Generator().manual_seed(3)
    x = (torch.randn(len(dst), h, generator=gen) * 3).to(dtype)
    dy = torch.randn(len(dst), h, generator=gen).to(dtype)
    y = graphop.sparse_softmax_forward(*csr, x.to(DEV))
    want, _ = reference(dst, n, x, dy)
    dx = graphop.sparse_softmax_backward(*csr, y, dy.to(DEV))
    yh = y.cpu().double()                                         # (the backward is that of the rounded probabilities)
    dot = torch.zeros(n, h, dtype=torch.float64).index_add_(0, dst, yh * dy.double())
    want_dx = yh * (dy.double() - dot[dst])
    # float32: exp and division to some ulp; sums of 5000 terms.  bfloat16: one rounding of the result
    tol = 3e-6 if dtype == torch.float32 else 2 ** -8
    assert ((yh - want).abs() <= tol * (want.abs() + 1e-7)).all()
    bound = tol * (want_dx.abs() + yh * (dy.double().abs() + dot[dst].abs() + 1))
    assert ((dx.cpu().double() - want_dx).abs() <= bound).all()
    # (rerun: the same bits)
    assert torch.equal(y, graphop.sparse_softmax_forward(*csr, x.to(DEV))) and torch.equal(dx, graphop.sparse_softmax_backward(*csr, y, dy.to(DEV)))


@pytest.mark.parametrize("h", [4, 8, 16])
def test_masked_and_infinite_scores_and_unaligned_tensors(h, monkeypatch):
    from bpt_amd import graphop, plan
    monkeypatch.setattr(plan, "FORCE_SEG_LEN", 64)
    plan.plan_cache.clear()
    dst, n, csr = graph("shuffled")
    gen = torch.Generator().manual_seed(4)
    x = torch.randn(len(dst), h, generator=gen)
    x[torch.rand(x.shape, generator=gen) < 0.3] = float("-inf")    # masked
    first = torch.tensor([int((dst == r).nonzero()[0]) for r in range(n) if DEGREES[r]])
    x[first] = 0.5                                                # (every row keeps an edge)
    long_row, short_row = DEGREES.index(1500), DEGREES.index(33)
    whole = x.clone()
    for r in (long_row, short_row):
        x[int((dst == r).nonzero()[3]), h - 1] = float("inf")     # NaN in that row and head, nowhere else
    y = graphop.sparse_softmax_forward(*csr, x.to(DEV)).cpu()
    touched = ((dst == long_row) | (dst == short_row)).unsqueeze(1) & (torch.arange(h) == h - 1)
    want, _ = reference(dst, n, whole, torch.zeros_like(whole))
    ok = (y.double() - want).abs() <= 3e-6 * (want.abs() + 1e-7)
    assert (ok | touched).all() and y[int((dst == long_row).nonzero()[3]), h - 1].isnan() and y[int((dst == short_row).nonzero()[3]), h - 1].isnan()
    held = torch.empty(len(dst) * h + 1, device=DEV)
    held[1:] = whole.to(DEV).flatten()
    unaligned = held[1:].view(len(dst), h)
    got = graphop.sparse_softmax_forward(*csr, unaligned).cpu().double()
    assert ((got - want).abs() <= 3e-6 * (want.abs() + 1e-7)).all()
