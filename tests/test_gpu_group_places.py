"""The places of a plan's groups (locality, ranges of equal work, decreasing work inside a range) at the edges of what one workgroup
places and compares with at a time, up to about the largest number of groups (a bound of 16384) that are placed this way; bit for bit the numpy model."""
import numpy as np
import pytest
import torch

import parallel_plan_model as model
from test_gpu_device_plan import check_base, check_groups

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("order", [2, 4], ids=["by-work", "local"])
@pytest.mark.parametrize("groups", [1, 15, 16, 17, 2047, 2048, 2049, 4097, 13700])
def test_groups_at_the_edges_of_a_comparison(groups, order):
    from bpt_amd import graphbuilder as gb
    from bpt_amd.plan import DevicePlan
    R, seg, n_index = 4, 8, 500                          # few neighbours: many groups with the same smallest one
    n = groups * R - (3 if groups > 1 else 0)            # the last group is not full
    rng = np.random.default_rng(groups)
    deg = rng.integers(0, 4, n)
    deg[n // 3: n // 3 + 40] = 0                         # whole groups without edges
    E = int(deg.sum())
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    eid = rng.permutation(E).astype(np.int64)
    row, units = gb.partition_csr(indptr, 32)
    arrs = (row, units, eid, rng.integers(0, n_index, E).astype(np.int64))
    want, info = model.base_plan(*arrs, n, n_index, seg)
    plan = DevicePlan(*(torch.from_numpy(a).to(DEV) for a in arrs), n, n_index, DEV, seg, groups=(R, order))
    check_base(plan, want, info)
    check_groups(plan.ensure_groups(R, order), model.group_plan(want, n_index, R, {2: 0, 4: 5}[order]), E)
