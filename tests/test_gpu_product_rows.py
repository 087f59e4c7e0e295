"""The row-group product whose sums over a head's lanes are spread over the members, at row lengths where a batch of entries or a
lane-held list of them ends, for groups of four and eight rows.  Against float64: a float32 sum of 64 products is off by at most
64 x 2^-24 x sum |a b| (stated with a factor 2), and rounding the result to bfloat16 adds 2^-8 of it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

@pytest.fixture
def forced(request):
    from bpt_amd import graphop, plan
    old = plan.FORCE_SEG_LEN, graphop._MIN_GROUP_ITEMS
    plan.FORCE_SEG_LEN, graphop._MIN_GROUP_ITEMS = request.param, 0
    plan.plan_cache.clear()
    yield
    plan.FORCE_SEG_LEN, graphop._MIN_GROUP_ITEMS = old
    plan.plan_cache.clear()


def rows(lengths, seed=0):
    """in-CSR side of rows of these lengths, edge ids shuffled"""
    from bpt_amd import graphbuilder as gb
    rng = np.random.default_rng(seed)
    dst = np.repeat(np.arange(len(lengths)), lengths)[rng.permutation(sum(lengths))].astype(np.int64)
    src = rng.integers(0, len(lengths), len(dst)).astype(np.int64)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, len(lengths))
    return src, dst, tuple(t.to(DEV) for t in (ROW, IR, out_csr[2], out_csr[1])), tuple(t.to(DEV) for t in (COL, IC, in_csr[2], in_csr[1]))


@pytest.mark.parametrize("forced", [64], indirect=True, ids=["seg64"])
@pytest.mark.parametrize("R", [4, 8])
@pytest.mark.parametrize("dtype,h,d", [(torch.float32, 4, 64), (torch.float32, 8, 64), (torch.float32, 16, 64), (torch.float32, 8, 32),
                                       (torch.bfloat16, 8, 64), (torch.bfloat16, 16, 64)], ids=lambda x: str(x).replace("torch.", ""))
def test_products_spread_over_the_members(dtype, h, d, R, forced):
    from bpt_amd import graphop
    lengths = [1, 2, 0, 7, 8, 9, 55, 56, 57, 64, 130, 3] * 3
    src, dst, out, _ = rows(lengths, seed=3)
    gen = torch.Generator().manual_seed(7)
    A, B = (torch.randn(len(lengths), h, d, generator=gen).to(dtype) for _ in range(2))
    A[5], B[6, :, 3] = float("nan"), float("inf")           # stay with the edges that read them
    before = graphop.set_group_rows(R)
    try:
        y = graphop.maskedmm_csr_forward(*out, A.to(DEV), B.to(DEV)).cpu()
    finally:
        graphop.set_group_rows(before)
    a, b = A.double()[src], B.double()[dst]
    want, size = (a * b).sum(-1), (a * b).abs().sum(-1)
    ok = torch.from_numpy((src != 5) & (dst != 6))[:, None].expand_as(want)
    assert ((y.double() - want).abs() <= (2 * 64 * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)) * size)[ok].all()
    assert torch.isnan(y[src == 5]).all() and not torch.isfinite(y[(src != 5) & (dst == 6)]).any()
