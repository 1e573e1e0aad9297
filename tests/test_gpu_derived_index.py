"""The inverse index of a table without its first column, derived from that of the whole table."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n,k", [(1, 2), (3, 5), (700, 9), (5000, 17), (4000, 300)])
@pytest.mark.parametrize("empty", [0.0, 0.3, 1.0])
def test_derived_index_lists_the_empty_slots(n, k, empty):
    """the gradient clears the slots without a neighbour through the index: it names every slot once"""
    from hgcalml_amd import ops
    g = torch.Generator().manual_seed(n + k)
    whole = torch.randint(0, n, (n, k), generator=g, dtype=torch.int32)
    whole[torch.rand(n, k, generator=g) < empty] = -1
    whole = whole.to(DEV)
    offsets, slots = ops.inverse_index_without_first_column(ops.inverse_neighbour_index(whole), n, k)
    want_offsets, want_slots = ops.inverse_neighbour_index(whole[:, 1:].contiguous())
    assert torch.equal(offsets, want_offsets) and torch.equal(slots, want_slots)
