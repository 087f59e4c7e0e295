"""Which kernel family a call takes is decided on the host from the plan's sizes and the dtype (graphop._tiles,
_tiles_backward, _tile_seg_len, and _tile_seg_without_plan where no plan is needed to decide) and where a plan is built from its size and the caller's preference
(plan._build_on_device, PlanCache.get(prefer_device=...)).  CPU only: the rules are plain functions of sizes."""
import ctypes
from types import SimpleNamespace

import torch

from bpt_amd import _lib, graphop, plan


def fake_plan(n_rows, n_edges):
    return SimpleNamespace(n_rows=n_rows, n_edges=n_edges, n_items=n_rows)


def test_tiles_need_64_columns_and_at_most_16_heads():
    cfg = graphop._SETTINGS
    for dtype in (torch.float32, torch.bfloat16):
        q = torch.empty(4, 8, 64, dtype=dtype)
        assert graphop._tiles(q, 8, 64, fake_plan(10, 100), 0.0, None, cfg)
        assert graphop._tiles(q, 16, 64, fake_plan(10, 100), 0.1, object(), cfg)        # dropout and score term included
        assert not graphop._tiles(q, 8, 32, fake_plan(10, 100), 0.0, None, cfg)
        assert not graphop._tiles(q, 32, 64, fake_plan(10, 100), 0.0, None, cfg)
    assert not graphop._tiles(torch.empty(4, 8, 64, dtype=torch.float64), 8, 64, fake_plan(10, 100), 0.0, None, cfg)
    old = graphop.set_group_rows(8)                                                       # a caller fixing the rows per group
    try:
        assert not graphop._tiles(torch.empty(4, 8, 64), 8, 64, fake_plan(10, 100), 0.0, None, graphop._SETTINGS)
    finally:
        graphop.set_group_rows(old)
    old = graphop.set_tiles(False)
    try:
        assert not graphop._tiles(torch.empty(4, 8, 64), 8, 64, fake_plan(10, 100), 0.0, None, graphop._SETTINGS)
    finally:
        graphop.set_tiles(old)


def test_backward_rule():
    f32, bf16 = torch.float32, torch.bfloat16
    term = torch.empty(1)                                                  # (any tensor: a score term is given)
    for plan in (fake_plan(8191, 98305), fake_plan(65535, 3293955), fake_plan(16383, 430237), fake_plan(33598, 573520)):
        for dtype in (f32, bf16):                                          # wherever the forward runs on tiles
            assert graphop._tiles_backward(plan, dtype) and graphop._tiles_backward(plan, dtype, term)
    old = graphop.TILE_BACKWARD
    try:
        graphop.TILE_BACKWARD = False
        assert not graphop._tiles_backward(fake_plan(10, 10), bf16)
    finally:
        graphop.TILE_BACKWARD = old


def test_segment_length_of_the_tile_plans_follows_the_mean_degree():
    assert graphop._tile_seg_len(fake_plan(16383, 430237)) == 64           # 26 edges per row
    assert graphop._tile_seg_len(fake_plan(65535, 3293955)) == 128         # 50
    assert graphop._tile_seg_len(fake_plan(4097, 524224)) == 256           # 128


def test_segment_length_of_two_node_sets_is_left_to_the_plan():
    """The sizes of a graph of two node sets do not say how many of its rows have edges; both ways of asking agree."""
    two = SimpleNamespace(n_rows=6905, n_index_nodes=6838, n_edges=176728, n_items=6905)
    q, k, units = torch.empty(6905, 8, 64), torch.empty(6838, 8, 64), torch.empty(6900, dtype=torch.int64)
    assert graphop._tile_seg_len(two) == plan.SEG_BY_ROWS
    assert graphop._tile_seg_without_plan(units, 176728, q, k, 8, 64, 0.0, None, graphop._SETTINGS) == plan.SEG_BY_ROWS
    same = SimpleNamespace(n_rows=6905, n_index_nodes=6905, n_edges=176728, n_items=6905)
    assert graphop._tile_seg_len(same) == 64


def test_segment_length_by_the_rows_that_have_edges():
    """Of 1000 rows every second or every one has 20, 40 or 100 edges, in units of up to 32 and as a plain CSR with its empty rows."""
    for edges, step, want in ((20, 1, 64), (20, 2, 64), (40, 1, 128), (40, 2, 128), (100, 1, 256), (100, 2, 256)):
        rows = torch.arange(0, 1000, step)
        ends = torch.arange(32, edges + 32, 32).clamp(max=edges)
        row = rows.repeat_interleave(len(ends))
        indptr = torch.cat([torch.zeros(1, dtype=torch.int64), (torch.arange(len(rows))[:, None] * edges + ends[None]).reshape(-1)])
        plain = torch.zeros(1001, dtype=torch.int64)
        plain[rows + 1] = edges
        for r, ip in ((row, indptr), (torch.arange(1000), plain.cumsum(0))):
            assert plan.rows_with_edges([(r, ip)]) == [len(rows)]
            assert plan.seg_lens_by_rows([(r, ip, len(rows) * edges)] * 2) == [want] * 2
    assert plan.tile_seg_len(176728, 6905) == 64                           # 26 edges a node, but 51 a row with edges
    none = torch.zeros(0, dtype=torch.int64)
    assert plan.seg_lens_by_rows([(none, none.new_zeros(1), 0)] * 2) == [64, 64]
    assert plan.rows_with_edges([(none, none)]) == [0]                     # (refused by the plan's validation, not here)


def test_choice_of_the_tile_kernels_without_a_plan_to_look_at():
    """_tile_seg_without_plan: the same answers as the rules that look at a plan wherever it gives one, None elsewhere."""
    cfg = graphop._SETTINGS
    q = torch.empty(16383, 8, 64)
    units = lambda n: torch.empty(n, dtype=torch.int64)
    seg = lambda un, E, qq=q, p=0.0, bias=None, c=None: graphop._tile_seg_without_plan(units(un), E, qq, qq, qq.size(1), qq.size(2), p, bias,
                                                                                        cfg if c is None else c)
    assert seg(16383, 430237) == graphop._tile_seg_len(fake_plan(16383, 430237)) == 64
    assert seg(65535, 3293955, torch.empty(65535, 16, 64, dtype=torch.bfloat16)) == 128
    assert seg(4097, 524224, torch.empty(4097, 8, 64)) == 256
    assert seg(1535, 28378, torch.empty(1535, 8, 64)) is None              # few rows with edges: the plan's work items decide
    assert seg(1536, 28378, torch.empty(1536, 8, 64)) == 64
    assert seg(100, 1000, torch.empty(100, 8, 64), p=0.1) == 64            # dropout and the score term take groups anyway
    assert seg(100, 1000, torch.empty(100, 8, 64), bias=object()) == 64
    assert seg(16383, 430237, torch.empty(16383, 8, 32)) is None           # no tile kernels for 32 columns per head
    assert seg(16383, 430237, torch.empty(16383, 8, 64, dtype=torch.float64)) is None
    big = SimpleNamespace(size=lambda i: (1 << 22, 16, 64)[i], element_size=lambda: 4, dtype=torch.float32)
    assert graphop._tile_seg_without_plan(units(1 << 22), 1 << 24, big, big, 16, 64, 0.0, None, cfg) is None     # 16 GiB of rows: no 32-bit offsets
    old = graphop.set_group_rows(8)
    try:
        assert seg(16383, 430237, c=graphop._SETTINGS) is None             # a caller fixing the rows per group: no tiles
    finally:
        graphop.set_group_rows(old)
    old = graphop.TILE_SEG_LEN
    try:
        graphop.TILE_SEG_LEN = 96
        assert seg(16383, 430237) == 96
    finally:
        graphop.TILE_SEG_LEN = old


def test_where_a_plan_is_built():
    cpu_eid = torch.zeros(1 << 18, dtype=torch.int64)
    assert not plan._build_on_device(cpu_eid, 1 << 20)                     # host tensors: on the host, whatever the size
    fake = SimpleNamespace(is_cuda=True, numel=lambda: 430237)
    assert not plan._build_on_device(fake, 16383)                          # below 24576 rows, mean degree 26
    assert plan._build_on_device(fake, 24576)
    dense = SimpleNamespace(is_cuda=True, numel=lambda: 524224)
    assert plan._build_on_device(dense, 4097)                              # 2^17 edges and more at a mean degree of 32 and more
    assert not plan._build_on_device(dense, 1000)                          # but not the CSR of a few hundred edge types
    old = plan.set_device_build(True)
    try:
        assert plan._build_on_device(fake, 10)
        plan.set_device_build(False)
        assert not plan._build_on_device(fake, 1 << 20)
    finally:
        plan.set_device_build(old)


def test_padded_shape_of_narrow_heads():
    """Heads of fewer than 64 columns run the fused kernels zero-padded to (h', 64): 6 x 50 and 8 x 40 are the reference's
    other head shapes (configs/imdb-4.yml:10-12, configs/ptb-6.yml:12-14); shapes with kernels of their own are not padded."""
    import torch
    from bpt_amd import graphop
    t = lambda h, d, dt=torch.float32: torch.zeros(3, h, d, dtype=dt)
    assert graphop.attention_padded_shape(t(6, 50)) == (8, 64)
    assert graphop.attention_padded_shape(t(8, 40)) == (8, 64)
    assert graphop.attention_padded_shape(t(8, 40, torch.bfloat16)) == (8, 64)
    assert graphop.attention_padded_shape(t(2, 16, torch.bfloat16)) == (8, 64)      # bfloat16 has no 4-head kernels
    assert graphop.attention_padded_shape(t(3, 24)) == (4, 64)
    assert graphop.attention_padded_shape(t(12, 64)) == (16, 64)
    assert graphop.attention_padded_shape(t(8, 64)) is None and graphop.attention_padded_shape(t(8, 32)) is None      # own kernels
    assert graphop.attention_padded_shape(t(8, 80)) is None and graphop.attention_padded_shape(t(20, 50)) is None   # too wide / too many heads
    assert graphop.attention_padded_shape(t(6, 50, torch.float64)) is None
    assert graphop.attention_padded_shape(torch.zeros(3, 50)) is None              # 2-D (single head) calls take the op chain


def test_order_of_the_source_side_tile_groups():
    """Large sparse graphs keep the locality order of the groups inside an XCD's range on the source side of the backward,
    small or dense ones the order by decreasing work; plan.TILE_ORDER_SRC overrides."""
    from bpt_amd import plan
    assert plan.tile_order_src(16383, 430237) == 0            # L = 8192, k = 4
    assert plan.tile_order_src(65535, 3293955) == 0           # L = 32768, k = 8
    assert plan.tile_order_src(33598, 573520) == 0            # the batch of 32 graphs
    assert plan.tile_order_src(8191, 784687) == 6             # L = 4096, k = 32: dense
    assert plan.tile_order_src(8191, 98305) == 6              # L = 4096, k = 1: small
    assert plan.tile_order_src(1023, 28378) == 6
    old, plan.TILE_ORDER_SRC = plan.TILE_ORDER_SRC, 10
    try:
        assert plan.tile_order_src(16383, 430237) == 10
    finally:
        plan.TILE_ORDER_SRC = old


def test_order_of_the_destination_side_tile_groups():
    """Destination-side tile groups run by decreasing work inside an XCD's range while K and V fit the memory-side cache
    and keep their locality order from 49 152 nodes on; plan.TILE_ORDER_DST overrides; groups of other sizes keep
    GROUP_ORDER; a plan's default is what ensure_groups and linked_to use when no order is named."""
    import numpy as np
    from bpt_amd import graphbuilder as gb, plan
    assert plan.tile_order_dst(16383) == 6                    # L = 8192, k = 4
    assert plan.tile_order_dst(33598) == 6                    # the batch of 32 graphs
    assert plan.tile_order_dst(65535) == 4                    # L = 32768
    assert plan.tile_order_dst(49152) == 4 and plan.tile_order_dst(49151) == 6
    g = gb.BinaryPartition(64, True, 2, 10)
    src, dst, _ = g.get_edges()
    n = g.number_of_nodes
    _, in_csr, _, _, COL, INDPTR_C = gb.get_csrs(src, dst, n)
    p = plan.Plan(COL, INDPTR_C, in_csr[2], in_csr[1], n, n, torch.device("cpu"))
    assert p.default_order(plan.TILE_GROUP_R) == 6 and p.default_order(plan.GROUP_R) == plan.GROUP_ORDER
    old, plan.TILE_ORDER_DST = plan.TILE_ORDER_DST, 4
    try:
        assert plan.tile_order_dst(16383) == 4 and p.default_order(plan.TILE_GROUP_R) == 4
        a = p.ensure_groups(plan.TILE_GROUP_R)                # built in locality order now ...
        assert a is p.ensure_groups(plan.TILE_GROUP_R, 4)     # ... the same groups as when the order is named
    finally:
        plan.TILE_ORDER_DST = old
    assert p.ensure_groups(plan.TILE_GROUP_R) is p.ensure_groups(plan.TILE_GROUP_R, 6)
    assert p.ensure_groups(plan.TILE_GROUP_R) is not a
    chunks = np.asarray(a["host"]["chunks"])
    assert chunks[0] == 0 and chunks[-1] == len(a["host"]["grp_ptr"]) - 1


FWD, DST, SRC, F32, BF16 = 1, 2, 3, 0, 2                                    # bptattn_measure.h, bptattn.h


def test_wavefronts_of_a_row():
    """Kernels that walk single rows: eight, four or one wavefront an item.  Rows of 1024 columns are shared by eight up to
    288 items only (585 items, forward: 22.3 us with eight, 18.7 with one), and a float32 forward with a wavefront for nearly every
    SIMD and many edges an item takes one."""
    lib = _lib.attn_lib()

    def parts(n_items, n_edges, kernel, h, d, dtype):
        p = _lib.PlanStruct()
        p.n_rows, p.n_items, p.n_edges = n_items, n_items, n_edges
        return lib.bpt_wavefronts_per_item(ctypes.byref(p), kernel, h, d, dtype)

    for kernel in (FWD, DST, SRC):
        for dtype in (F32, BF16):
            for h, d, most in ((4, 64, 640), (8, 64, 640), (8, 32, 640), (16, 64, 288)):
                assert [parts(n, 20000, kernel, h, d, dtype) for n in (1, most, most + 1, 801, 1024, 2048, 2049)] == [8, 8, 4, 4, 4, 4, 1]
            for h, d in ((4, 64), (8, 32), (8, 64), (16, 64)):
                want = 1 if kernel == FWD and dtype == F32 and h * d >= 512 else 4
                for n, e in ((801, 25000), (1024, 25000), (1024, 60000)):
                    assert parts(n, e, kernel, h, d, dtype) == want
                for n, e in ((800, 25000), (1025, 25000), (1024, 24999)):
                    assert parts(n, e, kernel, h, d, dtype) == 4
    for bad in ((0, 8, 64, F32), (4, 8, 64, F32), (FWD, 0, 64, F32), (FWD, 8, 0, F32), (FWD, 8, 64, 1), (FWD, 8, 64, 9)):
        assert lib.bpt_wavefronts_per_item(ctypes.byref(_lib.PlanStruct()), *bad) < 0
    assert lib.bpt_wavefronts_per_item(None, FWD, 8, 64, F32) < 0


def test_wavefronts_of_a_tile_and_head():
    """Dense tiles: four, two or one wavefront a tile and head, by the wavefronts of the launch and the blocks each keeps; a float32
    forward stops at 6500 wavefronts (L = 7000, k = 32: 51.7 us with one, 53.9 with two), the backward at 8192."""
    lib = _lib.attn_lib()

    def parts(n_groups, blocks, kernel, h=8, dtype=F32):
        p = _lib.PlanStruct()
        p.n_rows = p.n_items = 16 * n_groups
        p.n_index_nodes = p.n_rows
        p.grp_R, p.n_groups, p.grp_max_chunk, p.n_grp_entries = 16, n_groups, n_groups, 16 * n_groups * blocks
        p.grp_members = p.grp_ptr = p.grp_entries = p.grp_chunks = 16          # (looked at for null only)
        return lib.bpt_wavefronts_per_item(ctypes.byref(p), kernel, h, 64, dtype)

    for kernel in (FWD, DST, SRC):
        # float32: wavefronts 8 n_groups
        assert [parts(n, 1, kernel) for n in (1, 96, 97, 192, 193)] == [4, 4, 2, 2, 1]
        assert [parts(n, 4, kernel) for n in (193, 384, 385)] == [2, 2, 1]
        assert [parts(n, 8, kernel) for n in (192, 193, 384, 385, 812)] == [4, 2, 2, 2, 2]
        assert parts(813, 8, kernel) == parts(1024, 8, kernel) == (1 if kernel == FWD else 2)
        assert parts(1025, 8, kernel) == 1 and parts(812, 7, kernel) == 1
        assert [parts(n, 8, kernel, h=16) for n in (96, 97, 406, 513)] == [4, 2, 2, 1]
        # bfloat16
        assert [parts(n, 1, kernel, dtype=BF16) for n in (75, 76, 150, 151)] == [4, 2, 2, 1]
        assert [parts(n, 8, kernel, dtype=BF16) for n in (150, 151, 288, 289)] == [2, 2, 2, 1]


def test_wavefronts_of_a_tile_and_head_of_the_separate_operators():
    """Heads that access the edge tensor together lose that in parts: they take one where the launch has wavefronts enough without.  The
    others, and smaller launches, follow the attention kernels' rule."""
    lib = _lib.attn_lib()

    def plan_of(n_groups, blocks):
        p = _lib.PlanStruct()
        p.n_rows = p.n_items = p.n_index_nodes = 16 * n_groups
        p.n_edges = 16 * 16 * n_groups * blocks
        p.grp_R, p.n_groups, p.grp_max_chunk, p.n_grp_entries = 16, n_groups, n_groups, 16 * n_groups * blocks
        p.grp_members = p.grp_ptr = p.grp_entries = p.grp_chunks = p.grp_eids = 16          # (looked at for null only)
        return p

    def parts(n_groups, blocks, h, d):
        return lib.bpt_wavefronts_per_product(ctypes.byref(plan_of(n_groups, blocks)), h, d)

    def attention(n_groups, blocks, h):
        return lib.bpt_wavefronts_per_item(ctypes.byref(plan_of(n_groups, blocks)), DST, h, 64, F32)

    for h, d, first in ((4, 64, 850), (8, 64, 425), (6, 50, 567), (8, 40, 425), (2, 64, 1700), (16, 63, 213)):
        for blocks in (3, 9, 20):
            assert [parts(n, blocks, h, d) for n in (first, 2 * first, 9 * first)] == [1, 1, 1]
            assert all(parts(n, blocks, h, d) == attention(n, blocks, h) for n in (1, 60, 100, first // 2, first - 1))
    assert parts(424, 9, 8, 64) == parts(566, 9, 6, 50) == parts(849, 9, 4, 64) == 2
    for blocks in (3, 9, 11):
        assert parts(129, blocks, 16, 64) == 1 and parts(128, blocks, 16, 64) == attention(128, blocks, 16)
    assert parts(128, 9, 16, 64) == 2 and parts(212, 12, 16, 64) == 2 and parts(213, 12, 16, 64) == 1
    for h, d in ((5, 30), (1, 64), (7, 63)):
        for n, blocks in ((1, 9), (200, 9), (800, 4), (1000, 9), (5000, 9)):
            assert parts(n, blocks, h, d) == attention(n, blocks, h)
    assert parts(8, 4, 17, 64) == parts(8, 4, 8, 65) == parts(8, 4, 8, 3) == 0
    assert lib.bpt_wavefronts_per_product(ctypes.byref(_lib.PlanStruct()), 8, 64) == 0
    assert lib.bpt_wavefronts_per_product(ctypes.byref(_lib.PlanStruct()), 0, 64) < 0 and lib.bpt_wavefronts_per_product(None, 8, 64) < 0
