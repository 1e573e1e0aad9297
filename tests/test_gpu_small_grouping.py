"""The grouping of a few thousand points by one workgroup: neighbours and distances bit for bit those of the oracle, at the
ends of its threads and its range, on single and nested grids, for one and many events, with directions and with all
points in one place."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n,events,dims,K", [
    (1, 1, 3, 4), (2, 1, 2, 4), (63, 2, 3, 8), (1023, 1, 4, 50), (1024, 3, 3, 16), (1025, 5, 2, 16), (2049, 40, 3, 52),
    (2047, 1, 4, 64), (2047, 13, 3, 16), (2048, 1, 3, 64), (2048, 2, 5, 12), (2049, 1, 3, 48), (2050, 7, 4, 16),
    (3000, 1, 6, 10), (700, 1, 3, 16)])
@pytest.mark.parametrize("space", ["clusters", "one place"])
def test_small_grouping(oracle, n, events, dims, K, space):
    from hgcalml_amd import BinnedSelectKnn
    rng = np.random.default_rng(n + dims)
    x = rng.standard_normal((n, dims)).astype(np.float32) * rng.choice([0.02, 1.0], (n, 1)).astype(np.float32)
    if space == "one place":
        x[:min(3 * n // 4, 900)] = 0.25
    cuts = np.sort(rng.integers(0, n + 1, events - 1))
    rs = np.concatenate([[0], cuts, [n]]).astype(np.int32)
    for direction in (None, rng.integers(0, 4, n).astype(np.int32)):
        want_i, want_d = oracle.canonical_knn(*oracle.BinnedSelectKnn(K, x, rs, direction=direction, n_bins=6))
        td = None if direction is None else torch.from_numpy(direction).to(DEV)
        got_i, got_d = BinnedSelectKnn(K, torch.from_numpy(x).to(DEV), torch.from_numpy(rs).to(DEV), direction=td)
        got_i, got_d = got_i.cpu().numpy(), got_d.cpu().numpy()
        assert (got_d.view(np.int32) == want_d.view(np.int32)).all()
        # exact ties of the distance at the K-th place may keep another of the tied points
        differ = (got_i != want_i).any(1)
        for v in np.flatnonzero(differ):
            last = want_d[v][want_i[v] >= 0].max()
            assert set(got_i[v][got_d[v] < last]) == set(want_i[v][want_d[v] < last])
