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


def test_merge_keeps_graphs_apart_that_a_subclass_tells_apart():
    """A subclass with a constructor argument of its own, and a class that only has what the merge calls."""
    from bpt_amd import graphbuilder as gb

    class Without(gb.BinaryPartition):                            # leaves out the edges of some types
        def __init__(self, length, types):
            super().__init__(length, True, 4, 10)
            self.types = types

        def __reduce__(self):
            return Without, (self._length, self.types)

        def get_edges_device(self, device, v_shift=0):
            src, dst, etype = super().get_edges_device(device, v_shift)
            keep = ~torch.isin(etype, torch.tensor(self.types, device=device))
            return src[keep], dst[keep], etype[keep]

    class Chain:
        number_of_nodes = 4

        def __reduce__(self):
            return Chain, ()

        def get_edges_device(self, device):
            i = torch.arange(3, device=device)
            return i, i + 1, torch.zeros_like(i)

        def get_pos(self):
            return np.arange(4)

    plain, some, more = gb.BinaryPartition(30, True, 4, 10), Without(30, (0,)), Without(30, (0, 1))
    n = plain.number_of_nodes
    src, dst, etype, pos, nodes = gb.merge_graphs_device([plain, some, more, Chain()], DEV)
    _, _, want = plain.get_edges()
    want = [want, want[want > 0], want[want > 1], np.zeros(3, dtype=np.int64)]
    assert nodes == 3 * n + 4 and pos.numel() == nodes
    assert np.array_equal(etype.cpu().numpy(), np.concatenate(want))
    assert src[-3:].tolist() == [3 * n, 3 * n + 1, 3 * n + 2] and dst[-1].item() == 3 * n + 3


@pytest.mark.parametrize("dtype,step,more", [(torch.int32, 1, 0), (torch.int64, 2, 0), (torch.int64, 1, 3)])
def test_merge_with_lists_that_the_launch_cannot_read(dtype, step, more):
    """A class of the caller's with 32-bit lists, strided views or positions of another length, beside an ordinary graph."""
    from bpt_amd import graphbuilder as gb

    class Chain:
        number_of_nodes = 5

        def __reduce__(self):
            return Chain, (dtype, step, more)

        def get_edges_device(self, device):
            i = torch.arange(4, device=device).repeat_interleave(step).to(dtype)[::step]
            return i, i + 1, i

        def get_pos(self):
            return np.arange(5 + more)

    plain = gb.BinaryPartition(30, True, 4, 10)
    n, (src, dst, etype), pos = plain.number_of_nodes, plain.get_edges(), plain.get_pos()
    got = gb.merge_graphs_device([Chain(), plain, Chain()], DEV)
    i = np.arange(4)
    want = ([i, src + 5, i + 5 + n], [i + 1, dst + 5, i + 6 + n], [i, etype, i], [np.arange(5 + more), pos, np.arange(5 + more)])
    assert got[4] == n + 10
    for a, b in zip(got[:4], want):
        assert a.dtype == torch.int64 and np.array_equal(a.cpu().numpy(), np.concatenate(b))


@pytest.mark.parametrize("n_src,n_dst,E,seg,orders", [(300, 300, 6000, 64, (None, 0)), (40, 900, 5000, 64, (6, 6)), (900, 40, 5000, 128, (4, 2)),
                                                      (1, 1, 1, 64, (None, 0)), (5000, 64, 70000, 64, (None, 0))])
def test_both_sides_built_together(n_src, n_dst, E, seg, orders):
    """DevicePlan.tile_plans: both sides of a graph in shared launches equal the plans built one by one (the model), the second
    linked to the first; sides of different sizes share the launches of the larger one."""
    from bpt_amd import graphbuilder as gb
    from bpt_amd.plan import DevicePlan, pair_numbers_host
    rng = np.random.default_rng(E)
    src, dst = rng.integers(0, n_src, E).astype(np.int64), rng.integers(0, n_dst, E).astype(np.int64)
    dst[: E // 3] = n_dst // 2
    if E > 4:
        src[-3:], dst[-3:] = src[-4], dst[-4]                     # an edge four times
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_src, n_dst, as_torch=False)
    sides = [((COL, IC, in_csr[2], in_csr[1]), n_dst, n_src), ((ROW, IR, out_csr[2], out_csr[1]), n_src, n_dst)]
    plans = DevicePlan.tile_plans([(*(torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in arrs), n, ni, seg, order)
                                   for (arrs, n, ni), order in zip(sides, orders)])
    want = []
    for plan, (arrs, n, ni), order in zip(plans, sides, orders):
        base, info = model.base_plan(*arrs, n, ni, seg)
        check_base(plan, base, info)
        by_mask = plan._by_mask(16, order)
        want.append(model.group_plan(base, ni, 16, by_mask))
        hit = plan.ensure_groups(16, order)
        check_groups(hit, want[-1], E)
        assert list(plan._groups) == [(16, by_mask)], "the groups were built a second time"
    st = plans[1].linked_to(plans[0], 16, order=orders[1], partner_order=orders[0], pair_numbers=True)
    (_, pairs, partner), = plans[1]._links.values()
    assert partner is plans[0] and st.grp_pairs == pairs.data_ptr()
    assert np.array_equal(pairs.cpu().numpy(), pair_numbers_host(want[1], want[0], E))


def test_malformed_sides_are_refused_together():
    from bpt_amd import graphbuilder as gb
    from bpt_amd.plan import DevicePlan
    src, dst = random_edges(50, 400, False)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, 50)
    good = [tuple(t.to(DEV) for t in side) for side in ((COL, IC, in_csr[2], in_csr[1]), (ROW, IR, out_csr[2], out_csr[1]))]
    for side in (0, 1):
        bad = [list(g) for g in good]
        bad[side][3] = bad[side][3].clone()
        bad[side][3][7] = 50
        with pytest.raises(ValueError, match="out of range"):
            DevicePlan.tile_plans([(*g, 50, 50, 64, None) for g in bad])
    assert DevicePlan.tile_plans([(*g, 50, 50, 64, None) for g in good])[0].n_rows == 50
