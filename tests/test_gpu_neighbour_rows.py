"""PushKnn's gradient and the neighbour moments at the sizes where their kernels' tiles end: columns around the multiples of
16 and 64, slots around the multiples of 4 and 16, single vertices, padded rows, with and without a processing order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def table(rng, n, K):
    idx = rng.integers(-1, n, (n, K)).astype(np.int32)
    idx[rng.random(n) < 0.2, K // 2:] = -1
    return idx


@pytest.mark.parametrize("n,K,F", [(1, 1, 1), (3, 2, 15), (17, 15, 16), (16, 16, 17), (33, 17, 48), (40, 31, 63), (50, 24, 64),
                                   (31, 33, 65), (29, 5, 96), (65, 64, 127), (66, 20, 128), (64, 7, 129), (35, 16, 192),
                                   (35, 18, 193), (70, 40, 255), (40, 70, 256), (40, 12, 257)])
def test_push_gradient(n, K, F):
    from hgcalml_amd import ops
    rng = np.random.default_rng(n + 100 * K + 10000 * F)
    idx = table(rng, n, K)
    g, x = rng.standard_normal((2, n, F)).astype(np.float32)
    w = rng.standard_normal((n, K)).astype(np.float32)
    rows = np.where((idx < 0)[..., None], 0, g[np.maximum(idx, 0)]).astype(np.float64)   # [n, K, F]
    want_w = (rows * x[:, None, :]).sum(-1)
    want_x = np.zeros((n, F), np.float32)
    for k in range(K):  # slot order, every product and sum rounded
        has = idx[:, k] >= 0
        want_x[has] = want_x[has] + g[idx[has, k]] * w[has, k, None]
    # F products and sums in float32, each off by 2^-24 of a partial sum that the absolute terms bound
    bound = (F + 8) * 2.0 ** -24 * (np.abs(rows) * np.abs(x)[:, None, :]).sum(-1)
    for order in (None, rng.permutation(n).astype(np.int32)):
        ti = torch.from_numpy(idx).to(DEV)
        if order is not None:
            ops.set_vertex_order(ti, torch.from_numpy(order).to(DEV))
        gw, gx = torch.ops.hgcalml.push_knn_grad(torch.from_numpy(g).to(DEV), torch.from_numpy(w).to(DEV),
                                                 torch.from_numpy(x).to(DEV), ti)
        assert (gx.cpu().numpy().view(np.int32) == want_x.view(np.int32)).all()
        assert (np.abs(gw.cpu().numpy() - want_w) <= bound).all()
        assert (gw.cpu().numpy()[idx < 0] == 0).all()


@pytest.mark.parametrize("n,K,F,C", [(1, 1, 1, 1), (5, 3, 2, 2), (40, 4, 8, 4), (33, 5, 7, 3), (70, 9, 16, 4), (50, 32, 4, 6),
                                     (129, 31, 3, 5)])
def test_neighbour_moments(n, K, F, C):
    from hgcalml_amd import NeighbourCovariance, ops
    rng = np.random.default_rng(n + K + F + C)
    idx = table(rng, n, K)
    x, feat = rng.standard_normal((n, C)).astype(np.float32), rng.standard_normal((n, F)).astype(np.float32)
    d = rng.random((n, K), dtype=np.float32)
    a = 1.0 / (1.0 + np.exp(-feat.astype(np.float64))) + 1e-3
    safe = np.maximum(idx, 0)
    wa = np.where((idx < 0)[..., None], 0, np.exp(-d.astype(np.float64))[..., None] * a[safe])         # [n, K, F]
    total = wa.sum(1) + 1e-3
    mean = np.einsum("nkf,nkc->nfc", wa, x[safe].astype(np.float64)) / total[..., None]
    cen = x[safe][:, :, None, :].astype(np.float64) - mean[safe]                                       # [n, K, F, C]
    cov = np.einsum("nkf,nkfc,nkfd->nfcd", wa, cen, cen) / total[..., None, None]
    for order in (None, rng.permutation(n).astype(np.int32)):
        ti = torch.from_numpy(idx).to(DEV)
        if order is not None:
            ops.set_vertex_order(ti, torch.from_numpy(order).to(DEV))
        got_cov, got_mean = NeighbourCovariance(torch.from_numpy(x).to(DEV), torch.from_numpy(d).to(DEV),
                                                torch.from_numpy(feat).to(DEV), ti)
        # sums of K products of numbers below 4 (differences below 8): (K + 16) roundings of 2^-24 of at most 64 each
        bound = (K + 16) * 64 * 2.0 ** -24
        assert np.abs(got_mean.cpu().numpy() - mean).max() <= bound
        assert np.abs(got_cov.cpu().numpy().reshape(n, F, C, C) - cov).max() <= bound
