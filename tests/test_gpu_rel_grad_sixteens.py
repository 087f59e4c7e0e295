"""Gradients of the rel_pos score term (graphop.rel_bias_backward) where the kernel's sixteens of slots can go wrong, against float64: rows
of 1 to 17, 63 to 65, 127 to 130 and several hundred slots (segments), whose sixteens hold sixteen types, one type or a mix; more work items than a
wavefront keeps descriptors of; q and dq that start on any element; an infinite value of ds, which reaches its own row and type only; a table row
that is not finite, which reaches the rows that have an edge of its type."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def run(deg, types_of, n_types, h, dtype, seed, offset=0, poison=None, poison_number=None):
    from bpt_amd import graphbuilder as gb, graphop, plan
    plan.plan_cache.clear()
    n, E, d, rng = len(deg), int(sum(deg)), 64, np.random.default_rng(seed)
    dst = np.repeat(np.arange(n), deg).astype(np.int64)
    _, in_csr, _, _, col, ic = gb.get_csrs(rng.integers(0, n, E).astype(np.int64), dst, n)
    et = types_of(rng, deg)
    used_types = np.unique(et).astype(np.int32)
    used = np.full(n_types, -1, dtype=np.int32)
    used[used_types] = np.arange(len(used_types))
    gen = torch.Generator().manual_seed(seed)

    def at_offset(x):                                             # the same values in memory that starts `offset` elements later
        held = torch.empty(x.numel() + offset, dtype=dtype, device=DEV)
        held[offset:] = x.to(DEV).flatten()
        return held[offset:].view(x.shape)

    q, dq0 = (torch.randn(n, h, d, generator=gen).to(dtype) for _ in range(2))
    table, ds = torch.randn(n_types, d, generator=gen).to(dtype), torch.randn(E, h, generator=gen) * 0.1
    if poison is not None:
        ds[poison] = float("inf")
    if poison_number is not None:
        table[used_types[poison_number], 9], table[used_types[poison_number], 50] = float("nan"), float("-inf")
    dq = at_offset(dq0)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    dtable = graphop.rel_bias_backward(col.to(DEV), ic.to(DEV), in_csr[2].to(DEV), to(used[et[in_csr[2].numpy()]].astype(np.int64)), to(used),
                                       to(used_types), torch.cat([ds, torch.zeros(1, h)]).to(DEV), at_offset(q), table.to(DEV), dq)
    qd, td, dd = q.double(), table.double(), ds.double()
    rows, ets = torch.from_numpy(dst), torch.from_numpy(et)
    want_dq, size_dq, want_t, size_t = dq0.double(), dq0.double().abs(), torch.zeros(n_types, d, dtype=torch.float64), torch.zeros(n_types, d, dtype=torch.float64)
    for e0 in range(0, E, 4096):                                  # (a few edges at a time: an edge gives h x 64 products)
        r, t, x = rows[e0:e0 + 4096], ets[e0:e0 + 4096], dd[e0:e0 + 4096]
        to_q, to_t = x.unsqueeze(2) * td[t].unsqueeze(1), torch.einsum("eh,ehd->ed", x, qd[r])
        want_dq.index_add_(0, r, to_q)
        size_dq.index_add_(0, r, to_q.abs())
        want_t.index_add_(0, t, to_t)
        size_t.index_add_(0, t, torch.einsum("eh,ehd->ed", x.abs(), qd[r].abs()))
    return dq.cpu().double(), dtable.cpu().double(), want_dq, size_dq, want_t, size_t


def close(got, want, size, dtype, longest):
    """An error of a rounding (2^-24) of the sum of magnitudes per doubling of the number of terms and one more for the products, and the
    rounding of a bfloat16 result (2^-8 of it)."""
    eps = 2.0 ** -24 * (2 + np.log2(longest + 1)) * 4
    assert ((got - want).abs() <= eps * size + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0) + 1e-30).all()


LENGTHS = list(range(0, 18)) + [31, 32, 33, 63, 64, 65, 127, 128, 129, 130, 300, 0, 700]
KINDS = {"different": lambda rng, deg: np.concatenate([(np.arange(k) + rng.integers(0, 40)) % 40 for k in deg]),
         "the same": lambda rng, deg: np.repeat(rng.integers(0, 40, len(deg)), deg),
         "mixed": lambda rng, deg: rng.integers(0, 40, sum(deg)),
         "pairs": lambda rng, deg: np.concatenate([(np.arange(k) // 2) % 40 for k in deg])}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("h,dtype", [(4, torch.float32), (8, torch.float32), (16, torch.float32), (8, torch.bfloat16), (16, torch.bfloat16)])
def test_rows_of_every_length(h, dtype, kind):
    got_q, got_t, want_q, size_q, want_t, size_t = run(LENGTHS, lambda rng, deg: KINDS[kind](rng, deg).astype(np.int64), 50, h, dtype, 3)
    close(got_q, want_q, size_q, dtype, 700)
    close(got_t, want_t, size_t, dtype, sum(LENGTHS) * h)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_more_items_than_a_wavefront_keeps_descriptors_of(dtype):
    """230 types leave a wavefront a workgroup: 36 000 items are 70 for each of 512."""
    got_q, got_t, want_q, size_q, want_t, size_t = run([1, 3] * 18000, lambda rng, deg: rng.integers(0, 230, sum(deg)), 230, 8, dtype, 4)
    close(got_q, want_q, size_q, dtype, 3)
    close(got_t, want_t, size_t, dtype, 72000 * 8)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_that_start_on_any_element(dtype):
    plain = run(LENGTHS, lambda rng, deg: KINDS["mixed"](rng, deg), 50, 8, dtype, 5)
    for offset in (1, 2, 3):
        moved = run(LENGTHS, lambda rng, deg: KINDS["mixed"](rng, deg), 50, 8, dtype, 5, offset)
        assert torch.equal(plain[0], moved[0]) and torch.equal(plain[1], moved[1])


@pytest.mark.parametrize("kind", ["different", "the same", "mixed"])
def test_an_infinite_value_stays_in_its_row_and_type(kind):
    got_q, got_t, want_q, _, want_t, _ = run(LENGTHS, lambda rng, deg: KINDS[kind](rng, deg).astype(np.int64), 50, 8, torch.float32, 6, poison=(1000, 3))
    assert torch.equal(got_q.isfinite(), want_q.isfinite()) and torch.equal(got_t.isfinite(), want_t.isfinite())
    assert not want_q.isfinite().all() and not want_t.isfinite().all()


@pytest.mark.parametrize("kind", ["different", "the same", "mixed"])
@pytest.mark.parametrize("number", [0, 17, -1])
@pytest.mark.parametrize("h,dtype,n_types", [(4, torch.float32, 40), (8, torch.float32, 40), (16, torch.bfloat16, 40), (8, torch.float32, 88),
                                             (16, torch.bfloat16, 150)])
def test_a_table_row_that_is_not_finite_stays_in_its_types_rows(h, dtype, n_types, number, kind):
    """The first, one and the last of the types in use, rows with and without edges of it, of lengths that leave sixteens and chunks of 64
    slots part empty."""
    draw = {"different": lambda rng, k: (np.arange(k) + rng.integers(0, n_types)) % n_types, "the same": lambda rng, k: np.full(k, rng.integers(0, n_types)),
            "mixed": lambda rng, k: rng.integers(0, n_types, k)}[kind]
    lengths = LENGTHS[:-1] + list(range(1, n_types))

    def types_of(rng, deg):
        out = np.concatenate([draw(rng, k) for k in deg])
        out[-n_types:] = np.arange(n_types)                       # (all of them are in use)
        return out.astype(np.int64)
    got_q, got_t, want_q, size_q, want_t, size_t = run(lengths, types_of, n_types, h, dtype, 8, poison_number=number)
    assert torch.equal(got_q.isfinite(), want_q.isfinite()) and not want_q.isfinite().all() and (want_q.isfinite().all(2).all(1)[1:]).any()
    whole = want_q.isfinite()
    close(got_q[whole], want_q[whole], size_q[whole], dtype, max(lengths))
    close(got_t, want_t, size_t, dtype, sum(lengths) * h)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n_types", [66, 88, 150, 238])
@pytest.mark.parametrize("h,dtype", [(4, torch.float32), (8, torch.float32), (16, torch.bfloat16)])
def test_two_wavefronts_share_the_columns(h, dtype, n_types, offset):
    """From 57 types on (65 at 4 heads, 50 at 16): four, two or one table of sums a workgroup; sixteens of different types, of one and of a mix."""
    def types_of(rng, deg):
        draw = (lambda k: (np.arange(k) + rng.integers(0, n_types)) % n_types, lambda k: np.full(k, rng.integers(0, n_types)), lambda k: rng.integers(0, n_types, k))
        out = np.concatenate([draw[i % 3](k) for i, k in enumerate(deg)])
        out[:n_types] = np.arange(n_types)                        # (all of them are in use)
        return out.astype(np.int64)
    got_q, got_t, want_q, size_q, want_t, size_t = run(LENGTHS, types_of, n_types, h, dtype, 6, offset=offset)
    close(got_q, want_q, size_q, dtype, 700)
    close(got_t, want_t, size_t, dtype, sum(LENGTHS) * h)
