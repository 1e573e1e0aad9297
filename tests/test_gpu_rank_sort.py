"""Sorting of distinct keys by counting the smaller ones, at the ends of its workgroups of 64 keys and of its range;
equal keys keep their order there."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 1000, 1025, 4999, 16383, 16384, 16385])
@pytest.mark.parametrize("equal", [False, True])
def test_rank_sort(n, equal):
    from hgcalml_amd import ops
    rng = np.random.default_rng(n)
    value = rng.permutation(n).astype(np.uint64)
    high = rng.integers(0, 1 << 43, n, dtype=np.uint64)
    high[rng.random(n) < 0.5] = 77
    keys = (high << np.uint64(20)) | value
    if equal and n > 1:
        keys = keys[rng.integers(0, n, n)]
        if n > 16384:
            keys = np.unique(keys)  # beyond the range equal keys come out in any order
    got = ops.sort_distinct_keys(torch.from_numpy(keys.view(np.int64)).to("cuda:0"), 20).cpu().numpy()
    assert (got == (np.sort(keys) & np.uint64((1 << 20) - 1)).astype(np.int32)).all()
