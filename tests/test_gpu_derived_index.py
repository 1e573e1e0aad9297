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


def test_gradient_with_an_index_that_is_longer_than_the_table():
    """only the entries that the offsets name count: n (K + 1) of them are not taken for a wider table's index"""
    from hgcalml_amd import ops
    g = torch.Generator().manual_seed(1)
    n, k, f = 50, 7, 16
    idx = torch.randint(0, n, (n, k), generator=g, dtype=torch.int32).to(DEV)
    w, x, up = (torch.rand(n, c, generator=g).to(DEV) for c in (k, f, 2 * f))
    _, arg, slots = torch.ops.hgcalml.accumulate_knn_slots(w, x, idx, 0, True)
    off, inv = ops.inverse_neighbour_index(idx)
    longer = torch.cat([inv, torch.zeros(n, dtype=torch.int32, device=DEV)])
    for a, b in zip(torch.ops.hgcalml.accumulate_knn_grad_slots(up, w, x, idx, arg, slots, off, inv),
                    torch.ops.hgcalml.accumulate_knn_grad_slots(up, w, x, idx, arg, slots, off, longer)):
        assert torch.equal(a, b)


def test_derived_index_of_the_largest_table():
    """2^31 - 256 slots: the last list ends where a wave's step beyond it is no int any more. Row v names v alone, apart
    from its first slot, so that both indices list the slots in order."""
    from hgcalml_amd import ops
    n, k = 8388607, 256
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 64 GB of device memory")
    offsets = (torch.arange(n + 1, device=DEV) * k).to(torch.int32)
    slots = torch.arange(n * k, dtype=torch.int32, device=DEV)
    got_offsets, got_slots = ops.inverse_index_without_first_column((offsets, slots), n, k)
    del slots
    assert torch.equal(got_offsets, (torch.arange(n + 1, device=DEV) * (k - 1)).to(torch.int32))
    total = n * (k - 1)
    for s in range(0, total, 1 << 28):
        e = min(total, s + (1 << 28))
        assert torch.equal(got_slots[s:e], torch.arange(s, e, dtype=torch.int32, device=DEV))
    del got_slots
    torch.cuda.empty_cache()
