"""Candidate records of the condensates where their waves and workgroups end (63 to 65, 255 to 257 candidates), for each
length of a record (up to 4, 8 and 16 coordinates) and rows that are no multiple of 16 bytes, against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dims", [1, 3, 4, 7, 8, 13])
@pytest.mark.parametrize("high", [1, 63, 64, 65, 255, 256, 257])
def test_ends_of_waves_and_workgroups(oracle, high, dims):
    from hgcalml_amd import BuildAndAssignCondensatesBinned
    rng = np.random.default_rng(100 * high + dims)
    n = high + 40
    beta = np.where(np.arange(n) < high, 0.2 + 0.7 * rng.random(n), 0.05).astype(np.float32)[rng.permutation(n), None]
    coords = rng.random((n, dims), dtype=np.float32)
    dist = (0.1 + 0.3 * rng.random((n, 1))).astype(np.float32)
    mask = (rng.random((n, 1)) < 0.1).astype(np.int32)
    rs = np.array([0, n // 3, n], np.int32)
    for by_max_beta in (True, False):
        for m in (None, mask):
            want = oracle.BuildAndAssignCondensatesBinned(coords, beta, dist, rs, 0.1, no_condensation_mask=m,
                                                          assign_by_max_beta=by_max_beta)
            got = BuildAndAssignCondensatesBinned(
                *(torch.from_numpy(a).to(DEV) for a in (coords, beta, dist, rs)), 0.1,
                no_condensation_mask=None if m is None else torch.from_numpy(m).to(DEV), assign_by_max_beta=by_max_beta)
            for g, w in zip(got, want):
                assert (g.cpu().numpy() == w).all()
