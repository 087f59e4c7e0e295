"""The edge softmax with the heads side by side where its split rows are taken whole by a workgroup each, and just past where they are: the longest row
by the number of heads, the number of split rows beside their length; against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def check(deg, h, dtype):
    from bpt_amd import graphbuilder as gb, graphop, plan
    plan.plan_cache.clear()
    n, rng = len(deg), np.random.default_rng(7)
    dst = np.repeat(np.arange(n), deg).astype(np.int64)
    rng.shuffle(dst)
    _, in_csr, _, _, col, ic = gb.get_csrs(rng.integers(0, n, len(dst)).astype(np.int64), dst, n)
    csr = tuple(t.to(DEV) for t in (col, ic, in_csr[2]))
    gen = torch.Generator().manual_seed(8)
    x, dy = ((torch.randn(len(dst), h, generator=gen) * s).to(dtype) for s in (3, 1))
    y = graphop.sparse_softmax_forward(*csr, x.to(DEV))
    dx = graphop.sparse_softmax_backward(*csr, y, dy.to(DEV)).cpu().double()
    struct = plan.plan_cache.get(*csr, None, None, None, prefer_device=True).struct
    idx = torch.from_numpy(dst).unsqueeze(1).expand(-1, h)
    xd, yh, dyd = x.double(), y.cpu().double(), dy.double()
    e = torch.exp(xd)
    want = e / torch.zeros(n, h, dtype=torch.float64).scatter_add_(0, idx, e).gather(0, idx)
    dot = torch.zeros(n, h, dtype=torch.float64).scatter_add_(0, idx, yh * dyd).gather(0, idx)
    want_dx = yh * (dyd - dot)
    # float32: exponentials and a division to some ulp, sums of up to 1024 terms over some hundred partial sums; bfloat16: one rounding of the result
    tol = {torch.float32: 3e-6, torch.bfloat16: 2.0 ** -8, torch.float64: 1e-13}[dtype]
    assert ((yh - want).abs() <= tol * (want + 1e-7)).all()
    assert ((dx - want_dx).abs() <= tol * (want_dx.abs() + yh * (dyd.abs() + dot.abs() + 1))).all()
    return struct


@pytest.mark.parametrize("longest", [511, 512, 513, 640, 641, 768, 769, 1024])
@pytest.mark.parametrize("h,dtype", [(6, torch.float32), (7, torch.float32), (12, torch.bfloat16), (64, torch.float32), (5, torch.float64), (6, torch.float64), (32, torch.float64)])
def test_longest_row(h, dtype, longest):
    struct = check([3, 65, longest, 0, 200, longest, 64, 129], h, dtype)
    assert struct.max_degree == longest and struct.n_heavy == 5


@pytest.mark.parametrize("rows,deg,h,dtype", [(1536, 65, 3, torch.float64), (1537, 65, 3, torch.float64), (1537, 257, 3, torch.float64), (3072, 66, 1, torch.float32),
                                              (3073, 66, 1, torch.float32), (3073, 193, 2, torch.bfloat16)])
def test_number_of_split_rows(rows, deg, h, dtype):
    assert check([deg] * rows + [5, 0, 64], h, dtype).n_heavy == rows
