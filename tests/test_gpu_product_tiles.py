"""The separate operators on tiles: SpMM and SDDMM of float32 rows of 4 to 64 columns a head, against float64, over graphs whose tiles are
walked by four, two and one wavefronts a head (tile_parts), with duplicate edges, rows without edges and split rows; edge tensors that
start on four bytes only; rows that are not finite, which may reach the rows that have an edge from them and no others.

Bounds: a float32 sum of n products is off by at most n 2^-24 times the sum of their absolute values (stated with a factor 2)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def bpt(L, k, triu=True):
    from bpt_amd import graphbuilder as gb
    g = gb.BinaryPartition(L, triu, k, 10)
    src, dst, _ = g.get_edges()
    return np.asarray(src), np.asarray(dst), g.number_of_nodes


def window(L, w):
    from bpt_amd import graphbuilder as gb
    g = gb.FullyConnected(L, True, w)
    src, dst, _ = g.get_edges()
    return np.asarray(src), np.asarray(dst), g.number_of_nodes


def multigraph(n=97, E=3000):
    rng = np.random.default_rng(1)
    src, dst = rng.integers(1, n, E), rng.integers(1, n, E)
    dst[:1000], src[1000:1500] = 1, 2                             # heavy rows on both sides
    src[-40:], dst[-40:] = src[-80:-40], dst[-80:-40]              # edges twice
    return src.astype(np.int64), dst.astype(np.int64), n


GRAPHS = {"bpt512": lambda: bpt(512, 4, False), "bpt2000": lambda: bpt(2000, 1), "bpt9000": lambda: bpt(9000, 1), "window": lambda: window(2000, 100), "multigraph": multigraph,
          "one token": lambda: bpt(1, 1)}
SHAPES = [(8, 64), (4, 64), (16, 64), (6, 50), (8, 40), (5, 30), (3, 4), (1, 64), (7, 63)]


class Sides:
    def __init__(self, name):
        from bpt_amd import graphbuilder as gb
        src, dst, self.n = GRAPHS[name]()
        self.E = len(src)
        out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, self.n)
        self.out = tuple(t.to(DEV) for t in (ROW, IR, out_csr[2], out_csr[1]))
        self.inn = tuple(t.to(DEV) for t in (COL, IC, in_csr[2], in_csr[1]))
        self.src, self.dst = (torch.from_numpy(x).to(DEV) for x in (src, dst))


_sides = {}


def sides(name):
    if name not in _sides:
        _sides[name] = Sides(name)
    return _sides[name]


def rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def product_ok(y, a, b):                                          # y (E, h) of gathered rows a, b (E, h, d)
    a, b = a.double(), b.double()
    return ((y.double() - (a * b).sum(-1)).abs() <= 2 * a.size(-1) * 2.0 ** -24 * (a * b).abs().sum(-1) + 1e-37).all()


def sum_ok(y, to, w, x, n):                                       # y (n, h, d) of rows x (E, h, d) weighted with w (E, h)
    terms = w.double().unsqueeze(-1) * x.double()
    zero = torch.zeros(y.shape, dtype=torch.float64, device=y.device)
    want, size = zero.index_add(0, to, terms), zero.index_add(0, to, terms.abs())
    count = torch.zeros(n, dtype=torch.float64, device=y.device).index_add_(0, to, torch.ones_like(to, dtype=torch.float64))
    return ((y.double() - want).abs() <= 2 * count[:, None, None].clamp(min=1) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("h,d", SHAPES)
@pytest.mark.parametrize("name", list(GRAPHS))
def test_products_and_sums_match_float64(name, h, d):
    from bpt_amd import graphop as G
    s = sides(name)
    A, B = rand((s.n, h, d), 1), rand((s.n, h, d), 2)
    held = rand((s.E * h + 1,), 3)
    for W in (held[:-1].view(s.E, h), held[1:].view(s.E, h)):
        for side, frm, to in ((s.out, s.dst, s.src), (s.inn, s.src, s.dst)):
            y = G.vector_spmm_forward(*side, W, A)
            assert sum_ok(y, to, W, A[frm], s.n)
            assert torch.equal(y, G.vector_spmm_forward(*side, W, A))
            assert product_ok(G.maskedmm_csr_forward(*side, A, B), A[to], B[frm])
        dA, dB = G.maskedmm_csr_backward(*s.out, *s.inn, A, B, W)
        assert sum_ok(dA, s.src, W, B[s.dst], s.n) and sum_ok(dB, s.dst, W, A[s.src], s.n)
        dW, dx = G.vector_spmm_backward(*s.inn, *s.out, W, B, A)
        assert product_ok(dW, B[s.dst], A[s.src]) and sum_ok(dx, s.src, W, B[s.dst], s.n)


@pytest.mark.parametrize("h,d", [(8, 64), (6, 50), (5, 30)])
@pytest.mark.parametrize("name", ["bpt512", "bpt9000", "multigraph"])
def test_rows_that_are_not_finite_stay_with_their_neighbours(name, h, d):
    from bpt_amd import graphop as G
    s = sides(name)
    A, W = rand((s.n, h, d), 1), rand((s.E, h), 3)
    A[5], A[6, :, 3] = float("nan"), float("inf")
    for side, frm, to in ((s.out, s.dst, s.src), (s.inn, s.src, s.dst)):
        y = G.vector_spmm_forward(*side, W, A)
        bad = torch.zeros(s.n, dtype=torch.bool, device=DEV).index_fill_(0, to[(frm == 5) | (frm == 6)], True)
        assert torch.isfinite(y[~bad]).all() and not torch.isfinite(y[bad][..., 3]).any()
        keep = ~bad[to]
        assert sum_ok(y[~bad], (torch.cumsum(~bad, 0) - 1)[to[keep]], W[keep], A[frm[keep]], int((~bad).sum()))
        e = G.maskedmm_csr_forward(*side, rand((s.n, h, d), 4), A)
        assert torch.equal(~torch.isfinite(e).all(1), (frm == 5) | (frm == 6))


@pytest.mark.parametrize("h", [4, 8, 16])
@pytest.mark.parametrize("name", ["bpt512", "bpt2000", "bpt9000", "multigraph"])
def test_node_tensors_that_start_on_four_bytes(name, h):
    """64 columns a head, which take the kernels of narrow heads then, on tiles in four, two and one parts, and split rows."""
    from bpt_amd import graphop as G
    s = sides(name)
    off = lambda x: torch.cat([x.new_zeros(1), x.flatten()])[1:].view(x.shape)
    A, B, W = off(rand((s.n, h, 64), 1)), off(rand((s.n, h, 64), 2)), rand((s.E, h), 3)
    assert A.data_ptr() % 16 == B.data_ptr() % 16 == 4
    for W in (W, off(W)):
        for side, frm, to in ((s.out, s.dst, s.src), (s.inn, s.src, s.dst)):
            assert sum_ok(G.vector_spmm_forward(*side, W, A), to, W, A[frm], s.n)
            assert product_ok(G.maskedmm_csr_forward(*side, A, B), A[to], B[frm])
        dA, dB = G.maskedmm_csr_backward(*s.out, *s.inn, A, B, W)
        assert sum_ok(dA, s.src, W, B[s.dst], s.n) and sum_ok(dB, s.dst, W, A[s.src], s.n)
        dW, dx = G.vector_spmm_backward(*s.inn, *s.out, W, B, A)
        assert product_ok(dW, B[s.dst], A[s.src]) and sum_ok(dx, s.src, W, B[s.dst], s.n)


def in_a_window(n, E, width):                                     # sources from the `width` rows around a row
    rng = np.random.default_rng(2)
    dst = np.sort(rng.integers(0, n, E))
    return ((dst + rng.integers(0, width, E)) % n).astype(np.int64), dst.astype(np.int64), n


@pytest.mark.parametrize("graph,h,d,tiles", [((2048, 20000, 2048), 8, 64, False), ((2048, 20000, 2048), 8, 32, False), ((2048, 20000, 2048), 6, 50, True),
                                             ((2048, 20000, 2048), 8, 30, True), ((2048, 40000, 60), 8, 64, True), ((2048, 40000, 60), 8, 32, True),
                                             ((2048, 40000, 130), 8, 64, True), ((2048, 40000, 130), 8, 32, False), ((13000, 107000, 100), 4, 64, True),
                                             ((11000, 90000, 100), 4, 64, False), ((2048, 10000, 2048), 8, 64, True), ((2048, 10001, 2048), 8, 64, False), ((25000, 25000 * 8, 8), 8, 32, False), ((25000, 25000 * 8, 8), 8, 64, True)])
def test_tiles_where_rows_share_their_neighbours(graph, h, d, tiles):
    """Shapes with row-group kernels of their own take those where the tiles' rows have few neighbours in common, and 8 x 32 on large
    graphs; the others always take tiles."""
    from bpt_amd import graphbuilder as gb, graphop as G, plan
    src, dst, n = in_a_window(*graph)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs(src, dst, n)
    out, inn = (tuple(t.to(DEV) for t in side) for side in ((ROW, IR, out_csr[2], out_csr[1]), (COL, IC, in_csr[2], in_csr[1])))
    src, dst = torch.from_numpy(src).to(DEV), torch.from_numpy(dst).to(DEV)
    A, B, W = rand((n, h, d), 1), rand((n, h, d), 2), rand((len(src), h), 3)
    plan.plan_cache.clear()
    for side, frm, to in ((out, dst, src), (inn, src, dst)):
        assert sum_ok(G.vector_spmm_forward(*side, W, A), to, W, A[frm], n)
        assert product_ok(G.maskedmm_csr_forward(*side, A, B), A[to], B[frm])
    dA, dB = G.maskedmm_csr_backward(*out, *inn, A, B, W)
    assert sum_ok(dA, src, W, B[dst], n) and sum_ok(dB, dst, W, A[src], n)
    dW, dx = G.vector_spmm_backward(*inn, *out, W, B, A)
    assert product_ok(dW, B[dst], A[src]) and sum_ok(dx, src, W, B[dst], n)
    grouped = [R for p, _ in plan.plan_cache._d.values() for R, _ in p._groups]
    assert (4 in grouped or 8 in grouped) != tiles
    # bit for bit what the family computes that was chosen
    old = G.set_tiles(tiles)
    try:
        assert torch.equal(dA, G.maskedmm_csr_backward(*out, *inn, A, B, W)[0])
    finally:
        G.set_tiles(old)
