"""The kernels that build a batch's CSRs and plans (libbptplan, include/bptbuild.h) at the sizes where they can go wrong: the edges
of the sort's tiles of 2048 records and of its 9-bit digits, rows of many units, rows without edges.  Every result is integer and
equals the host builder's."""
import numpy as np
import pytest
import torch

import parallel_plan_model as model
from test_gpu_device_plan import check_base, check_groups

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


@pytest.mark.parametrize("order", [2, 6, 4], ids=["neighbour", "mask", "mask-local"])
@pytest.mark.parametrize("n,n_index,E,seg,R", [
    (70, 40, 3000, 64, 16),             # a group of the largest size: 1024 edges, many of them repeated
    (70, 300, 5000, 128, 16),           # ... 2048
    (50, 5000, 9000, 256, 16),          # ... 4096
    (50, 5000, 9000, 257, 16),          # one more: groups by device-wide sorts
    (33, 9, 2000, 512, 8),
    (200, 3000000, 4000, 64, 16),       # neighbours that take 64-bit keys
    (1, 1, 1, 1, 1),
    (40000, 700, 20000, 8, 4),          # more groups than are sorted in LDS
    (70000, 700, 20000, 8, 4),          # more groups than one workgroup numbers
])
def test_groups_at_the_edges_of_their_forms(n, n_index, E, seg, R, order):
    from bpt_amd import graphbuilder as gb
    from bpt_amd.plan import DevicePlan
    rng = np.random.default_rng(n + seg)
    rows, cols = rng.integers(0, n, E), rng.integers(0, n_index, E)
    rows[: E // 4] = n // 2                                       # a row of many items
    rows, cols = rows.astype(np.int64), cols.astype(np.int64)
    eid = np.argsort(rows, kind="stable").astype(np.int64)
    indptr = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=indptr[1:])
    row, units = gb.partition_csr(indptr, 32)
    arrs = (row, units, eid, cols[eid])
    want, info = model.base_plan(*arrs, n, n_index, seg)
    by_mask = {2: 0, 6: 1, 4: 5}[order]
    groups = model.group_plan(want, n_index, R, by_mask)
    tens = tuple(torch.from_numpy(a).to(DEV) for a in arrs)
    for asked_first in (True, False):                             # formed along with the base plan, or behind it
        plan = DevicePlan(*tens, n, n_index, DEV, seg, groups=(R, order) if asked_first else None)
        check_base(plan, want, info)
        check_groups(plan.ensure_groups(R, order), groups, E)


@pytest.mark.parametrize("n_graphs", [1, 63, 64, 65, 130])
def test_merge_at_the_edges_of_a_launch(n_graphs):
    from bpt_amd import graphbuilder as gb
    rng = np.random.default_rng(n_graphs)
    graphs = [gb.BinaryPartition(int(L), True, 4, 10) for L in rng.integers(1, 700, n_graphs)] + [gb.FullyConnected(1, True, 2)]
    want, got = gb.merge_graphs(graphs), gb.merge_graphs_device(graphs, DEV)
    assert got[4] == want[4]
    for a, b in zip(got[:4], want[:4]):
        assert a.dtype == torch.int64 and np.array_equal(a.cpu().numpy(), b)
