"""The kernels that build a batch's CSRs and plans (libbptplan, include/bptbuild.h) at the sizes where they can go wrong: the edges
of the sort's tiles of 2048 records and of its 9-bit digits, rows of many units, rows without edges.  Every result is integer and
equals the host builder's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def random_edges(n, E, skew, seed=0):
    rng = np.random.default_rng(seed)
    src, dst = rng.integers(0, n, E), rng.integers(0, n, E)
    if skew:                                    # one row holds two thirds of the edges
        dst[: 2 * E // 3] = n - 1
    return src.astype(np.int64), dst.astype(np.int64)


@pytest.mark.parametrize("skew", [False, True], ids=["even", "skewed"])
@pytest.mark.parametrize("n,E", [(1, 1), (3, 2047), (254, 2048), (255, 2049), (256, 4096), (511, 777), (512, 10000), (100000, 3),
                                 (262143, 30000), (262144, 30000), (5000, 600000)])
def test_csrs_at_the_edges_of_tiles_and_digits(n, E, skew):
    from bpt_amd import graphbuilder as gb
    src, dst = random_edges(n, E, skew)
    want = gb.get_csrs(src, dst, n, chunk_size=32, as_torch=False)
    got = gb.get_csrs_device(torch.from_numpy(src).to(DEV), torch.from_numpy(dst).to(DEV), n, chunk_size=32)
    for side in (0, 1):
        for a, b in zip(got[side], want[side]):
            assert a.dtype == torch.int64 and np.array_equal(a.cpu().numpy(), b)
    for a, b in zip(got[2:], want[2:]):
        assert a.dtype == torch.int64 and np.array_equal(a.cpu().numpy(), b)
