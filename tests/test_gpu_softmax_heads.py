"""The edge softmax and its backward with the heads side by side, for counts of heads that do not divide a wavefront and for the largest that it
holds, against float64: the rows of the test of four heads a lane, split into few and into many segments."""
import pytest
import torch

from test_gpu_softmax_quads import DEV, graph, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seg", [64, 24, 256])
@pytest.mark.parametrize("h,dtype", [(1, torch.float32), (3, torch.float32), (5, torch.bfloat16), (6, torch.float32), (7, torch.float64), (10, torch.float32),
                                     (12, torch.bfloat16), (21, torch.float32), (31, torch.float32), (33, torch.float32), (63, torch.float32),
                                     (64, torch.float32), (65, torch.float32)], ids=lambda x: str(x).replace("torch.", ""))
def test_softmax_of_any_number_of_heads(h, dtype, seg, monkeypatch):
    from bpt_amd import graphop, plan
    monkeypatch.setattr(plan, "FORCE_SEG_LEN", seg)
    plan.plan_cache.clear()
    dst, n, csr = graph("shuffled")
    gen = torch.Generator().manual_seed(3)
    x = (torch.randn(len(dst), h, generator=gen, dtype=torch.float64) * 3).to(dtype)
    dy = torch.randn(len(dst), h, generator=gen, dtype=torch.float64).to(dtype)
    y = graphop.sparse_softmax_forward(*csr, x.to(DEV))
    want, _ = reference(dst, n, x, dy)
    dx = graphop.sparse_softmax_backward(*csr, y, dy.to(DEV))
    yh = y.cpu().double()                                         # (the backward is that of the rounded probabilities)
    dot = torch.zeros(n, h, dtype=torch.float64).index_add_(0, dst, yh * dy.double())
    want_dx = yh * (dy.double() - dot[dst])
    # exp and division to some ulp, sums of 5000 terms; bfloat16: one rounding of the result
    tol = {torch.float32: 3e-6, torch.bfloat16: 2 ** -8, torch.float64: 1e-13}[dtype]
    assert ((yh - want).abs() <= tol * (want.abs() + 1e-7)).all()
    bound = tol * (want_dx.abs() + yh * (dy.double().abs() + dot[dst].abs() + 1))
    assert ((dx.cpu().double() - want_dx).abs() <= bound).all()
    assert torch.equal(y, graphop.sparse_softmax_forward(*csr, x.to(DEV))) and torch.equal(dx, graphop.sparse_softmax_backward(*csr, y, dy.to(DEV)))
