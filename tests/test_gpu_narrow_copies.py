"""The copies of q, k, v and of the result that the forward of narrow heads writes for the backward (keep): whole and exact at every
size around the pieces they are copied in, from rows on any four bytes, with different node counts on the two sides, with tiles
in one and in several parts, and for any choice of the four."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def graph(n_q, n_k):
    from bpt_amd import graphbuilder as gb
    rng = np.random.default_rng(n_q)
    deg = rng.integers(0, 9, n_q)
    deg[n_q // 2] = 300                                           # a split row
    dst = np.repeat(np.arange(n_q), deg).astype(np.int64)
    src = rng.integers(0, n_k, len(dst)).astype(np.int64)
    out_csr, in_csr, ROW, IR, COL, IC = gb.get_csrs_bipartite(src, dst, n_k, n_q)
    return tuple(t.to(DEV) for t in (COL, IC, in_csr[2], in_csr[1]))


# rows of 16 bytes: 1024 of them are one piece; of 36 and 12 bytes: ends inside 16 bytes
@pytest.mark.parametrize("heads,d,dtype,n_q,n_k", [(1, 4, torch.float32, 1024, 1024), (1, 4, torch.float32, 1025, 1023), (1, 4, torch.float32, 3, 4097),
                                                   (3, 6, torch.bfloat16, 455, 456), (1, 6, torch.bfloat16, 1365, 1366), (1, 6, torch.bfloat16, 5, 7),
                                                   (6, 50, torch.float32, 1000, 777), (6, 50, torch.bfloat16, 2001, 2001), (8, 40, torch.float32, 4000, 4000)])
def test_copies_are_whole_and_exact(heads, d, dtype, n_q, n_k, monkeypatch):
    from bpt_amd import graphop, plan
    monkeypatch.setattr(graphop, "_MIN_GROUP_ITEMS", 0)
    plan.plan_cache.clear()
    inn = graph(n_q, n_k)
    gen = torch.Generator(device=DEV).manual_seed(1)

    def rows(n, shift):                                           # starts `shift` x 4 bytes behind a 16-byte address
        held = torch.empty(n * heads * d + 16, dtype=dtype, device=DEV)
        at = shift * 4 // held.element_size()
        x = held[at:at + n * heads * d].view(n, heads, d)
        x.copy_(torch.randn(n, heads, d, generator=gen, device=DEV))
        return x

    h = graphop.attention_padded_shape(torch.empty(1, heads, d, dtype=dtype))[0]
    stand_in = [torch.empty(n, h, 64, dtype=dtype, device="meta") for n in (n_q, n_k, n_k)]
    q, k, v = rows(n_q, 0), rows(n_k, 1), rows(n_k, 3)
    for round_ in range(2):                                       # through Python, then from the native table
        for chosen in ((0, 1, 2, 3), (1,), (0, 3), ()):
            # (room behind each copy: nothing may be written there)
            room = [torch.full((x.numel() + 64,), 7.0, dtype=dtype, device=DEV) for x in (q, k, v, q)]
            keep = [r[:x.numel()].view(x.shape) if i in chosen else None for i, (r, x) in enumerate(zip(room, (q, k, v, q)))]
            o, lse = graphop.attention_forward(*inn, *stand_in, d ** -0.5, 0.0, 3, narrow=(q, k, v), keep=keep)
            for i, (copy, x) in enumerate(zip(keep, (q, k, v, o))):
                if copy is not None:
                    assert torch.equal(copy, x), i
                assert (room[i][x.numel() if copy is not None else 0:] == 7.0).all(), i


def test_copies_of_a_layer_on_padded_rows():
    from bpt_amd import graphop, plan
    plan.plan_cache.clear()
    inn = graph(100, 90)                                          # too small for tiles
    q, k, v = (torch.randn(n, 6, 50, device=DEV) for n in (100, 90, 90))
    keep = [torch.empty_like(x) for x in (q, k, v, q)]
    stand_in = [torch.empty(n, 8, 64, device="meta") for n in (100, 90, 90)]
    o, _ = graphop.attention_forward(*inn, *stand_in, 50 ** -0.5, narrow=(q, k, v), keep=keep)
    for copy, x in zip(keep, (q, k, v, o)):
        assert torch.equal(copy, x)
