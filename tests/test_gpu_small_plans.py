"""CSRs and base plans that one workgroup a side builds in a single launch (k_csr_small, k_plan_small) or whose items it orders (k_item_order), at the largest sizes that go this way and one
past them, against the host builder and the numpy model, bit for bit; malformed arrays; and the first training call on a small new graph, whose
two plans are built together and whose backward is served by the native host path."""
import numpy as np
import pytest
import torch

import parallel_plan_model as model
from test_gpu_device_plan import check_base, check_groups

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def edges(n_rows, n_index, E, kind, seed=1):
    rng = np.random.default_rng(seed)
    rows, cols = rng.integers(0, n_rows, E), rng.integers(0, n_index, E)
    if kind == "skewed":                                          # one row holds two thirds, the last rows have none
        rows = rows * 3 // 4
        rows[: 2 * E // 3] = n_rows // 2
    return rows.astype(np.int64), cols.astype(np.int64)


@pytest.mark.parametrize("kind", ["even", "skewed"])
@pytest.mark.parametrize("chunk", [32, 1, 5000])
@pytest.mark.parametrize("n,E", [(4096, 10240), (4096, 10241), (4097, 500), (4096, 1), (1, 10240), (300, 0), (1023, 127), (1025, 129), (7, 4097)])
def test_csrs(n, E, chunk, kind):
    from bpt_amd import graphbuilder as gb
    src, dst = edges(n, n, E, kind)
    want = gb.get_csrs(src, dst, n, chunk_size=chunk, as_torch=False)
    got = gb.get_csrs_device(torch.from_numpy(src).to(DEV), torch.from_numpy(dst).to(DEV), n, chunk_size=chunk)
    for a, b in zip([*got[0], *got[1], *got[2:]], [*want[0], *want[1], *want[2:]]):
        assert a.dtype == torch.int64 and np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("bad", [-1, 50, 1 << 40])
@pytest.mark.parametrize("which", [0, 1])
def test_a_bad_id_is_refused(which, bad):
    from bpt_amd import graphbuilder as gb
    pair = [torch.randint(0, 50, (900,), device=DEV) for _ in range(2)]
    pair[which][333] = bad
    with pytest.raises(ValueError, match="out of range"):
        gb.get_csrs_device(*pair, 50)


def side(n_rows, n_index, E, kind, seed=1):
    from bpt_amd import graphbuilder as gb
    rows, cols = edges(n_rows, n_index, E, kind, seed)
    eid = np.argsort(rows, kind="stable").astype(np.int64)
    indptr = np.zeros(n_rows + 1, dtype=np.int64)
    np.cumsum(np.bincount(rows, minlength=n_rows), out=indptr[1:])
    row, units = gb.partition_csr(indptr, 32)
    return row, units, eid, cols[eid]


SIZES = [(4000, 4000, 12288, 128), (3904, 3904, 12288, 64), (3905, 3905, 12288, 64), (500, 500, 12289, 64), (100, 65535, 3000, 64), (100, 65536, 3000, 64),
         (3, 2, 12000, 7), (1, 1, 1, 1), (1030, 20, 0, 64), (900, 900, 5000, 64), (127, 127, 64, 64), (2049, 2049, 4000, 1),
         (10800, 10800, 29696, 64), (10801, 10801, 29696, 64), (5000, 262143, 20000, 64), (5000, 262144, 20000, 64), (6000, 300, 0, 64)]     # k_item_order


@pytest.mark.parametrize("kind", ["even", "skewed"])
@pytest.mark.parametrize("n,n_index,E,seg", SIZES)
def test_base_plans_and_groups(n, n_index, E, seg, kind):
    from bpt_amd.plan import DevicePlan
    arrs = side(n, n_index, E, kind)
    want, info = model.base_plan(*arrs, n, n_index, seg)
    tens = tuple(torch.from_numpy(a).to(DEV) for a in arrs)
    check_base(DevicePlan(*tens, n, n_index, DEV, seg), want, info)
    other = side(n_index, n, E, kind, 2)                          # a second side of other sizes in the same launch
    want2, info2 = model.base_plan(*other, n_index, n, seg)
    tens2 = tuple(torch.from_numpy(a).to(DEV) for a in other)
    plans = DevicePlan.base_plans([(*tens, n, n_index, seg), (*tens2, n_index, n, seg)])
    check_base(plans[0], want, info)
    check_base(plans[1], want2, info2)
    built = DevicePlan.tile_plans([(*tens, n, n_index, seg, 2), (*tens2, n_index, n, seg, 6)])
    if built is not None:                                         # (items in the order of the groups: left by the same launch)
        check_base(built[0], want, info)
        check_groups(built[0].ensure_groups(16, 2), model.group_plan(want, n_index, 16, 0), E)
        check_groups(built[1].ensure_groups(16, 6), model.group_plan(want2, n, 16, 1), E)


def test_a_plan_without_indices_keeps_the_rows_order():
    from bpt_amd.plan import DevicePlan, Plan
    row, units, eid, _ = side(700, 700, 6000, "skewed")
    tens = tuple(torch.from_numpy(a).to(DEV) for a in (row, units, eid))
    got, want = DevicePlan(*tens, None, 700, 700, DEV, 64), Plan(row, units, eid, None, 700, 700, DEV, 64)
    assert (got.n_items, got.n_heavy, got.n_slots, got.max_degree, got.covers_all_edges) == \
           (want.n_items, want.n_heavy, want.n_slots, want.max_degree, want.covers_all_edges)
    for name, k in (("rowptr", 701), ("eid", 6000), ("items", got.n_items), ("heavy", got.n_heavy)):
        assert torch.equal(got._dev[name][:k], want._dev[name][:k]), name


def test_edge_ids_that_repeat_do_not_cover_the_edges():
    from bpt_amd.plan import DevicePlan
    arrs = [torch.from_numpy(a).to(DEV) for a in side(300, 300, 2000, "even")]
    arrs[2][7] = arrs[2][8]
    assert not DevicePlan(*arrs, 300, 300, DEV, 64).covers_all_edges


@pytest.mark.parametrize("where,at,value,message", [(0, 5, -1, "out of range|not sorted"), (0, 5, 300, "out of range|not sorted"), (0, 50, 0, "not sorted"), (1, 30, 0, "not sorted"),
                                                    (1, 0, -4, None), (1, -1, 2001, None), (1, -1, 1 << 33, None), (2, 9, 2000, "out of range"), (2, 9, -3, "out of range"),
                                                    (3, 9, 300, "out of range"), (3, 9, -1, "out of range"), (3, 9, 1 << 35, "out of range")])
def test_malformed_arrays_are_refused(where, at, value, message):
    from bpt_amd.plan import DevicePlan
    arrs = [torch.from_numpy(a).to(DEV) for a in side(300, 300, 2000, "even")]
    arrs[where][at] = value
    with pytest.raises(ValueError, match=message):
        DevicePlan(*arrs, 300, 300, DEV, 64)
    with pytest.raises(ValueError, match=message):
        DevicePlan.base_plans([(*arrs, 300, 300, 64)])


@pytest.mark.parametrize("heads,dtype", [(8, torch.float32), (16, torch.bfloat16)])
def test_first_call_on_a_small_new_graph(heads, dtype, monkeypatch):
    from bpt_amd import graphbuilder as gb, graphop, op, plan
    plan.plan_cache.clear()
    src, dst, _, _, n = gb.merge_graphs_device([gb.BinaryPartition(m, True, 4, 10) for m in (16, 3, 40, 90)], torch.device(DEV))
    out_csr, in_csr, row, ir, col, ic = gb.get_csrs_device(src, dst, n)
    args = (row, ir, out_csr[2], out_csr[1], col, ic, in_csr[2], in_csr[1])
    gen = torch.Generator(device=DEV).manual_seed(5)
    q, k, v, do = (torch.randn(n, heads, 64, generator=gen, device=DEV).to(dtype) for _ in range(4))
    leaves = [x.requires_grad_(True) for x in (q, k, v)]

    def not_here(*a, **kw):
        raise AssertionError("this went through Python")

    with monkeypatch.context() as m:
        m.setattr(graphop, "attention_backward", not_here)
        o = op.bpt_attention(*args, *leaves)
        first = (o.detach(),) + torch.autograd.grad(o, leaves, do)
    assert len(plan.plan_cache.held()) == 2
    plan.plan_cache.clear()
    monkeypatch.setattr(graphop, "prepare_training", lambda *a, **kw: None)       # one by one, when they are asked for
    o = op.bpt_attention(*args, *leaves)
    for name, a, b in zip(("o", "dq", "dk", "dv"), first, (o.detach(),) + torch.autograd.grad(o, leaves, do)):
        assert torch.equal(a, b), name
    plan.plan_cache.clear()
    monkeypatch.undo()
    bad = list(args)
    bad[3] = args[3].clone()
    bad[3][5] = n + 7                                             # an out-side neighbour that does not exist: the backward refuses it
    o = op.bpt_attention(*bad, *leaves)
    with pytest.raises(ValueError):
        o.sum().backward()
