"""CSRs and base plans of small graphs (one workgroup a side) where most rows have no edges and some have most of them, against the host builder and
the numpy model, bit for bit: what fills in the starts of the rows in between, and rows of more units or items than a thread writes by itself."""
import numpy as np
import pytest
import torch

import parallel_plan_model as model
from test_gpu_device_plan import check_base

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
KINDS = {"last": lambda n, E, rng: np.full(E, n - 1), "first": lambda n, E, rng: np.zeros(E), "ends": lambda n, E, rng: np.where(np.arange(E) % 3 == 0, 0, n - 1),
         "few": lambda n, E, rng: rng.choice(rng.integers(0, n, 5), E), "late": lambda n, E, rng: rng.integers(n - max(n // 50, 1), n, E)}


def edges(n, E, kind):
    rng = np.random.default_rng(n + E)
    return rng.integers(0, n, E).astype(np.int64), KINDS[kind](n, E, rng).astype(np.int64)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,E,chunk", [(4096, 10240, 32), (4096, 1, 32), (4095, 70, 8), (1024, 10240, 1), (64, 9, 1), (63, 8, 1), (2, 3000, 300)])
def test_csrs(n, E, chunk, kind):
    from bpt_amd import graphbuilder as gb
    src, dst = edges(n, E, kind)
    want = gb.get_csrs(src, dst, n, chunk_size=chunk, as_torch=False)
    got = gb.get_csrs_device(torch.from_numpy(src).to(DEV), torch.from_numpy(dst).to(DEV), n, chunk_size=chunk)
    for a, b in zip([*got[0], *got[1], *got[2:]], [*want[0], *want[1], *want[2:]]):
        assert a.dtype == torch.int64 and np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,E,seg", [(3904, 12288, 64), (4000, 100, 64), (1, 12288, 3), (1023, 576, 64), (1025, 513, 64), (300, 9000, 64)])
def test_base_plans(n, E, seg, kind):
    from bpt_amd import graphbuilder as gb
    from bpt_amd.plan import DevicePlan
    cols, rows = edges(n, E, kind)
    eid = np.argsort(rows, kind="stable").astype(np.int64)
    indptr = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=indptr[1:])
    row, units = gb.partition_csr(indptr, 32)
    arrs = (row, units, eid, cols[eid])
    want, info = model.base_plan(*arrs, n, n, seg)
    check_base(DevicePlan(*(torch.from_numpy(a).to(DEV) for a in arrs), n, n, DEV, seg), want, info)
