"""The distances' gradient with more than eight coordinates: rows and lists around the eight slots that are requested
together, vertices that nobody names and one that everybody names, empty slots. Bit for bit against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n,K,C", [(1, 1, 9), (9, 7, 9), (40, 8, 9), (300, 9, 12), (257, 16, 17), (1000, 33, 10), (64, 17, 70)])
def test_distance_gradient_beyond_eight_coordinates(oracle, n, K, C):
    from hgcalml_amd import ops  # noqa: F401
    rng = np.random.default_rng(n + 100 * K + C)
    idx = rng.integers(0, n, (n, K)).astype(np.int32)
    idx[:, 0] = 0
    idx[rng.random((n, K)) < 0.2] = -1
    idx[n // 2, :] = -1
    x, g = (rng.standard_normal(s).astype(np.float32) for s in ((n, C), (n, K)))
    got, order = [], torch.from_numpy(rng.permutation(n).astype(np.int32)).to(DEV)
    for use_order in (False, True):
        ti = torch.from_numpy(idx).to(DEV)
        if use_order:
            ops.set_vertex_order(ti, order)
        tg, tx = torch.from_numpy(g).to(DEV), torch.from_numpy(x).to(DEV)
        got.append(torch.ops.hgcalml.select_knn_grad(tg, ti, torch.zeros_like(tg), tx).cpu().numpy())
    ref = oracle.select_knn_grad_kernel(g, idx, x)
    assert all((a.view(np.int32) == ref.view(np.int32)).all() or np.array_equal(a, ref) for a in got)
