"""The score term over the tiles (graphop.rel_bias_forward_tiles) where the launch can go wrong: fewer tiles than the chip holds workgroups and
more, which then take several each; tiles of more pairs than a wavefront's first loads; rows without edges; the fewest and the most types in
use; tiles that use a few of the sixteens of types.  Against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def graph(n, kind, rng):
    """degrees of the n rows"""
    if kind == "short":
        deg = rng.integers(0, 6, n)
        deg[:: 7] = 0
    else:
        deg = rng.integers(30, 60, n)
        deg[5:9] = (300, 0, 1, 700)
    return deg


@pytest.mark.parametrize("n_used", [1, 16, 17, 64, 240])
@pytest.mark.parametrize("n,kind", [(40, "long"), (1500, "long"), (13_500, "short"), (33_000, "short")])
@pytest.mark.parametrize("h,dtype", [(4, torch.float32), (8, torch.float32), (16, torch.float32), (8, torch.bfloat16), (16, torch.bfloat16)])
def test_against_float64(h, dtype, n, kind, n_used):
    from bpt_amd import graphbuilder as gb, graphop, plan
    plan.plan_cache.clear()
    rng = np.random.default_rng(n + n_used)
    deg = graph(n, kind, rng)
    E, n_types = int(deg.sum()), 300
    dst = np.repeat(np.arange(n), deg).astype(np.int64)
    src = np.clip(dst + rng.integers(-40, 41, E), 0, n - 1).astype(np.int64)
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs(src, dst, n)
    graph_args = [t.to(DEV) for t in (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1])]
    used_types = rng.permutation(n_types)[:n_used].astype(np.int32)
    number = (dst * n_used // n + rng.integers(0, 20, E)) % n_used               # (neighbouring rows use neighbouring numbers)
    gen = torch.Generator().manual_seed(n_used)
    q, table = torch.randn(n, h, 64, generator=gen).to(dtype), torch.randn(n_types, 64, generator=gen).to(dtype)
    qd = q.to(DEV)
    pair, member = graphop.attention_pair_rows(*graph_args, qd, qd), graphop.attention_pair_members(*graph_args, qd, qd)
    if pair is None:
        pytest.skip("the layer does not run such a graph on tiles")
    tm = torch.empty(E, dtype=torch.int32, device=DEV).index_copy_(0, pair, torch.from_numpy(number.astype(np.int32)).to(DEV)) | (member << 8)
    bias = graphop.rel_bias_forward_tiles(*graph_args, qd, qd, table.to(DEV), torch.from_numpy(used_types).to(DEV), tm.contiguous())
    got = bias.t().index_select(0, pair).cpu().double()
    rows, types = torch.from_numpy(dst), torch.from_numpy(used_types[number].astype(np.int64))
    for e0 in range(0, E, 8192):                                  # (a few edges at a time: an edge gives h x 64 products)
        a, b = q.double()[rows[e0:e0 + 8192]], table.double()[types[e0:e0 + 8192]].unsqueeze(1)
        # 64 float32 products and sums: a rounding (2^-24) of the sum of magnitudes per doubling of the terms, one for the product and one to spare
        assert ((got[e0:e0 + 8192] - (a * b).sum(2)).abs() <= 8 * 2.0 ** -24 * (a * b).abs().sum(2)).all()
