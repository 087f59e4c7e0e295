"""The rel_pos score term of a graph that has rows and no edges (graphop.rel_bias_forward with the types in use): nothing is read, and all that is
written is the spare row of zeros behind the last edge's."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def arrays(n, h, dtype):
    empty = torch.empty(0, dtype=torch.int64, device=DEV)
    q, table = torch.randn(n, h, 64, device=DEV).to(dtype), torch.randn(5, 64, device=DEV).to(dtype)
    return (empty, torch.zeros(1, dtype=torch.int64, device=DEV), empty, empty, q, table), torch.tensor([0, 2, 4], dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("n", [1, 4, 17, 300])
@pytest.mark.parametrize("h,dtype", [(4, torch.float32), (8, torch.float32), (16, torch.bfloat16)])
def test_rows_and_no_edges(h, dtype, n):
    from bpt_amd import graphop
    args, used_types = arrays(n, h, dtype)
    bias = graphop.rel_bias_forward(*args, used_types=used_types)
    torch.cuda.synchronize()
    assert bias.shape == (1, h) and not bias.any()
    assert graphop.rel_bias_forward(*args, used_types=used_types, by_pair=True).shape == (h, 0)


def test_the_library_by_itself():
    """Two rows behind the spare one stay as they are; a result of no edges may be NULL, in either order, and q and table with it."""
    from bpt_amd import graphop, plan
    args, used_types = arrays(9, 8, torch.float32)
    p = plan.plan_cache.get(*args[:4], 9, 3, prefer_device=True)
    assert p.n_items == 9 and p.n_edges == 0
    held = torch.full((3, 8), 7.0, device=DEV)
    by_pair = ctypes.byref(graphop._by_pair(p.struct))
    for ref, bias in ((p.ref, held.data_ptr()), (p.ref, None), (by_pair, None), (by_pair, held[1:].data_ptr())):
        assert graphop._LIB.bpt_rel_bias_forward(ref, None, None, used_types.data_ptr(), 3, bias, 8, 64, 0, graphop._stream()) == 0
    torch.cuda.synchronize()
    assert held.tolist() == [[0.0] * 8] + [[7.0] * 8] * 2
