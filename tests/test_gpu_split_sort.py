"""The two-level key sort behind the inverse neighbour index where its variants and batches end: numbers of tiles around
1536 and 4096 (one counter per wave and tile, two passes of 6 and of 7 bits), stretches of a few items, of exactly one
batch of 12,288 and of one more, tiles beyond the 20,480 items that are held in registers."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n,k,kind", [(1, 5, "random"), (63, 65, "random"), (64, 64, "random"), (4096, 1, "random"), (4097, 1, "random"),
                                      (12288, 1, "random"), (49152, 64, "random"), (49153, 64, "random"), (1572863, 1, "random"),
                                      (1572864, 2, "random"), (4194303, 1, "random"), (4194304, 1, "random"), (60000, 40, "few"),
                                      (2000000, 3, "sorted"),
                                      # one tile: held in registers up to 20,480 slots, staged in LDS up to 32,768
                                      (16, 1280, "random"), (1, 20481, "random"), (16, 2048, "random"), (1, 32769, "random"),
                                      (31, 8200, "random"), (3, 512, "random"), (3, 513, "random")])
def test_inverse_index_at_the_ends_of_batches_and_tiles(n, k, kind):
    from hgcalml_amd import ops
    rng = np.random.default_rng(n + 7 * k)
    idx = rng.integers(0, n, (n, k)).astype(np.int32)
    if kind == "few":       # tiles of a hundred thousand items next to empty ones
        idx = (idx % 900).astype(np.int32)
    if kind == "sorted":
        idx = np.repeat(np.arange(n, dtype=np.int32)[:, None], k, 1)
    idx[rng.random((n, k)) < 0.03] = -1
    off, slots = ops.inverse_neighbour_index(torch.from_numpy(idx).to(DEV))
    flat = torch.from_numpy(idx.reshape(-1)).to(DEV).to(torch.int64)
    key = torch.where(flat < 0, torch.full_like(flat, n), flat)
    order = torch.sort(key, stable=True).indices
    assert torch.equal(slots[:n * k].to(torch.int64), order)
    assert torch.equal(off.to(torch.int64), torch.searchsorted(key[order], torch.arange(n + 1, device=DEV)))


@pytest.mark.parametrize("n,k", [(8388607, 256), (1000, 2147483)])
def test_inverse_index_of_the_largest_tables(n, k):
    """2^31 - 256 and 2^31 - 648 slots: the walks look ahead beyond the largest int"""
    from hgcalml_amd import ops
    total = n * k
    assert 2 ** 31 - 12288 < total < 2 ** 31
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 64 GB of device memory")
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n)
    idx = torch.randint(-1, n, (n, k), dtype=torch.int32, device=DEV, generator=gen)
    off, slots = ops.inverse_neighbour_index(idx)
    flat = idx.view(-1)
    # the first position of every key, with that of the slots without a neighbour and the end behind them
    begin = torch.cat([off.to(torch.int64), torch.tensor([total], device=DEV)])
    assert int(begin[0]) == 0 and bool((begin.diff() >= 0).all())
    last_key, last_slot = -1, -1
    for s in range(0, total, 1 << 27):
        part = slots[s:min(total, s + (1 << 27))].to(torch.int64)
        assert int(part.min()) >= 0 and int(part.max()) < total
        key = flat[part].to(torch.int64)
        key[key < 0] = n
        at = torch.arange(s, s + len(part), device=DEV)
        assert bool((begin[key] <= at).all()) and bool((at < begin[key + 1]).all())
        step, same = part.diff(), key.diff() == 0
        assert bool((key.diff() >= 0).all()) and bool((step[same] > 0).all())     # sorted, and stable: no slot twice
        assert int(key[0]) > last_key or (int(key[0]) == last_key and int(part[0]) > last_slot)
        last_key, last_slot = int(key[-1]), int(part[-1])
    del idx, flat, off, slots, part, key, at, step, same
    torch.cuda.empty_cache()
