"""masked_mm's two gradients, whose split rows one launch adds up, against the same two products with a launch each (vec_spmm's forward): equal
bit for bit, with split rows on both sides, one side or neither, whole heads and narrow ones, rows on 16 bytes and not."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("hubs", ["none", "sources", "destinations", "both"])
@pytest.mark.parametrize("h,d", [(4, 64), (8, 64), (16, 64), (6, 50), (8, 40), (5, 30)])
def test_the_same_bits(h, d, hubs, offset):
    from bpt_amd import graphbuilder as gb, graphop, plan
    plan.plan_cache.clear()
    rng, n = np.random.default_rng(h), 900
    src, dst = [np.repeat(np.arange(n), 6)], [np.clip(np.repeat(np.arange(n), 6) + rng.integers(-30, 31, 6 * n), 0, n - 1)]
    for i, wanted in ((0, hubs in ("sources", "both")), (1, hubs in ("destinations", "both"))):
        if wanted:
            hub, others = np.repeat([7, 450, n - 1], [200, 65, 700]), np.concatenate([rng.permutation(n)[:k] for k in (200, 65, 700)])
            src.append(others if i else hub)
            dst.append(hub if i else others)
    src, dst = np.concatenate(src).astype(np.int64), np.concatenate(dst).astype(np.int64)
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs(src, dst, n)
    side_r, side_c = [t.to(DEV) for t in (row, ir, out_csr[2], out_csr[1])], [t.to(DEV) for t in (col, ic, in_csr[2], in_csr[1])]
    gen = torch.Generator().manual_seed(d)

    def held(*shape):
        x = torch.empty(int(np.prod(shape)) + offset, device=DEV)
        x[offset:] = torch.randn(shape, generator=gen).to(DEV).flatten()
        return x[offset:].view(shape)

    a, b, dy = held(n, h, d), held(n, h, d), held(len(src), h)
    for _ in range(2):                                            # (the second call finds its plans)
        da, db = graphop.maskedmm_csr_backward(*side_r, *side_c, a, b, dy)
        assert torch.equal(da, graphop.vector_spmm_forward(*side_r, dy, b)) and torch.equal(db, graphop.vector_spmm_forward(*side_c, dy, a))
