"""Index tensors of the relative-position term (op._rel_aux): the types in use, their numbers and every slot's."""
import pytest
import torch

from bpt_amd import op


@pytest.mark.parametrize("n_types,n_edges", [(1000, 500), (1, 3), (7, 200), (240, 5000), (3, 1), (5, 0), (0, 0)])
def test_types_in_use(n_types, n_edges):
    gen = torch.Generator().manual_seed(n_types)
    etype, eid = torch.randint(0, max(n_types, 1), (n_edges,), generator=gen), torch.randperm(n_edges, generator=gen)
    aux = op._rel_aux(etype, torch.arange(1), torch.tensor([0, n_edges]), eid, n_types)
    types = torch.unique(etype)
    used = torch.full((n_types,), -1, dtype=torch.int32)
    used[types] = torch.arange(len(types), dtype=torch.int32)
    assert aux["n_used"] == len(types) and torch.equal(aux["used_types"], types.to(torch.int32)) and aux["used_types"].is_contiguous()
    assert aux["used"].dtype == torch.int32 and torch.equal(aux["used"], used)
    assert torch.equal(aux["etype_slot"], etype[eid]) and torch.equal(aux["number_slot"], used[etype[eid]].to(torch.int64))


@pytest.mark.parametrize("etype", [[0, 5], [-1, 2]])
def test_types_outside_the_table_are_refused(etype):
    with pytest.raises(ValueError, match="out of range"):
        op._rel_aux(torch.tensor(etype), torch.arange(1), torch.tensor([0, 2]), torch.arange(2), 5)
