"""Infinities and NaN where a kernel reads more than a result is made of: slots without a neighbour and lanes beyond the
end of a row contribute nothing, whatever they read. The oracle adds up the same terms and no others."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def same(a, b):
    """the same values, NaN for NaN"""
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("F", [256, 16384, 16400, 40001])
def test_empty_slots_of_wide_rows(oracle, F):
    """columns from 16384 on lie more than 2^16 bytes into the row"""
    from hgcalml_amd import ops  # noqa: F401  (registers torch.ops.hgcalml.*)
    rng = np.random.default_rng(F)
    n, K = 6, 4
    idx = np.array([[0, 1, 2, -1], [1, -1, 2, 3], [-1, 2, 3, -1], [3, 4, 5, 1], [-1, -1, -1, -1], [5, -1, -1, 2]], np.int32)
    x = rng.standard_normal((n, F)).astype(np.float32)
    x[0] = np.where(np.arange(F) % 2 == 0, np.inf, np.nan)
    w = rng.random((n, K), dtype=np.float32)
    for mm in (True, False):
        with np.errstate(invalid="ignore"):
            ref, rarg = oracle.AccumulateLinKnn(w, x, idx, mm)
        out, arg, _ = torch.ops.hgcalml.accumulate_knn_slots(t(w), t(x), t(idx), 0, mm)
        assert np.isfinite(ref[1:]).all() and same(out.cpu().numpy(), ref)
        if mm:
            assert (arg.cpu().numpy() == rarg).all()


def named_once(rng, n, K):
    """K different neighbours a row, the vertex itself not among them"""
    return np.stack([rng.permutation(np.delete(np.arange(n), v))[:K] for v in range(n)]).astype(np.int32)


def close(got, ref, bound):
    """non-finite values alike, finite ones within the bound"""
    finite = np.isfinite(ref)
    return same(got[~finite], ref[~finite]) and (np.abs(got[finite] - ref[finite]) <= bound[finite]).all()


@pytest.mark.parametrize("F", [16, 17, 18, 22, 31, 33, 45, 50, 65, 66, 100, 127, 128])
@pytest.mark.parametrize("mean_and_max", [True, False])
def test_infinite_gradient_in_the_last_columns(oracle, F, mean_and_max):
    """lanes beyond the end of a row hold the last columns again: what is infinite there counts once, and not times 0"""
    from hgcalml_amd import ops  # noqa: F401
    rng = np.random.default_rng(F)
    n, K = 40, 7
    idx = named_once(rng, n, K)
    x = (rng.random((n, F)) + 0.5).astype(np.float32)
    w = (rng.random((n, K)) + 0.5).astype(np.float32)
    g = (rng.random((n, 2 * F if mean_and_max else F)) + 0.5).astype(np.float32)
    g[::3, F - 1] = np.inf
    other = np.arange(1, n, 3)
    g[other, F - 2 - np.arange(len(other)) % 3] = -np.inf
    if mean_and_max:
        g[::4, 2 * F - 1] = np.inf
        g[other, 2 * F - 1] = 1
    _, arg = oracle.AccumulateLinKnn(w, x, idx, mean_and_max)
    rgw, rgx = oracle.accumulate_knn_grad_kernel(g, w, x, idx, arg)
    assert np.isinf(rgw).any() and not np.isnan(rgw).any()
    tw, tx, ti = t(w).requires_grad_(True), t(x).requires_grad_(True), t(idx)
    from hgcalml_amd import AccumulateLinKnn
    gw, gx = torch.autograd.grad(AccumulateLinKnn(tw, tx, ti, mean_and_max)[0], [tw, tx], t(g))
    # up to 2 F products below 2.25 and their sums in float32, in another order
    bound = np.full(rgw.shape, (2 * F + 8) * 2.0 ** -24 * 4.5 * F)
    assert close(gw.cpu().numpy(), rgw, bound)
    assert same(gx.cpu().numpy(), rgx)


@pytest.mark.parametrize("F", [1, 5, 16, 17, 22, 31, 48, 50, 64, 65, 100, 127, 129, 150, 193, 255, 256])
def test_infinite_push_gradient_in_the_last_columns(F):
    from hgcalml_amd import ops  # noqa: F401
    rng = np.random.default_rng(200 + F)
    n, K = 40, 7
    idx = named_once(rng, n, K)
    idx[5, 2:] = -1
    x = (rng.random((n, F)) + 0.5).astype(np.float32)
    w = (rng.random((n, K)) + 0.5).astype(np.float32)
    g = (rng.random((n, F)) + 0.5).astype(np.float32)
    g[::3, F - 1] = np.inf
    other = np.arange(1, n, 3)
    g[other, np.maximum(F - 2 - np.arange(len(other)) % 3, 0)] = -np.inf
    rows = np.where((idx < 0)[..., None], 0, g[idx]).astype(np.float64)
    want_w = (rows * x[:, None, :]).sum(-1)
    with np.errstate(invalid="ignore"):
        want_x = (rows * w[..., None]).sum(1)
    assert np.isinf(want_w).any() and not np.isnan(want_w).any()
    gw, gx = torch.ops.hgcalml.push_knn_grad(t(g), t(w), t(x), t(idx))
    # sums of F (K) products below 2.25
    assert close(gw.cpu().numpy(), want_w, np.full(want_w.shape, (F + 8) * 2.0 ** -24 * 2.25 * F))
    assert close(gx.cpu().numpy(), want_x, np.full(want_x.shape, (K + 8) * 2.0 ** -24 * 2.25 * K))


@pytest.mark.parametrize("F", [16, 22, 64, 100])
def test_infinite_gradient_of_a_maximum_at_repeated_self_references(oracle, F):
    """rows padded with the vertex itself: the max part of the feature gradient counts once, the weight gradient of every one
    of these slots has it"""
    from hgcalml_amd import AccumulateLinKnn
    rng = np.random.default_rng(100 + F)
    n, K = 40, 37
    idx = named_once(rng, n, K)
    idx[:, 3:6] = np.arange(n)[:, None]
    idx[::2, 20:] = np.arange(n)[::2, None]   # over the borders of 16 entries
    x = (rng.random((n, F)) + 0.5).astype(np.float32)
    w = (rng.random((n, K)) + 0.5).astype(np.float32)
    w[:, 3:6] = 3.0
    w[::2, 20:] = 3.0
    g = (rng.random((n, 2 * F)) + 0.5).astype(np.float32)
    g[::3, F:] = np.inf
    _, arg = oracle.AccumulateLinKnn(w, x, idx, True)
    assert (arg == np.arange(n)[:, None]).mean() > 0.1
    rgw, rgx = oracle.accumulate_knn_grad_kernel(g, w, x, idx, arg)
    assert np.isinf(rgx).any() and not np.isnan(rgx).any() and not np.isnan(rgw).any()
    tw, tx = t(w).requires_grad_(True), t(x).requires_grad_(True)
    gw, gx = torch.autograd.grad(AccumulateLinKnn(tw, tx, t(idx), True)[0], [tw, tx], t(g))
    assert close(gw.cpu().numpy(), rgw, np.full(rgw.shape, (2 * F + 8) * 2.0 ** -24 * 4.5 * F))
    assert same(gx.cpu().numpy(), rgx)


@pytest.mark.parametrize("C", [1, 2, 3, 4, 5, 8, 9, 12])
def test_distance_gradient_of_vertices_that_lie_nowhere(oracle, C):
    """slots without a neighbour and the places behind a row or list count nothing, also where the vertex's own coordinates are
    infinite or NaN"""
    from hgcalml_amd import ops  # noqa: F401
    rng = np.random.default_rng(300 + C)
    n, K = 50, 19
    idx = named_once(rng, n, K)
    idx[idx >= 45] = -1        # nobody names the last five vertices
    idx[45:] = -1              # and they name nobody
    x = rng.standard_normal((n, C)).astype(np.float32)
    x[45], x[46], x[47, C - 1] = np.inf, np.nan, -np.inf
    g = rng.standard_normal((n, K)).astype(np.float32)
    ref = oracle.select_knn_grad_kernel(g, idx, x)
    assert np.isfinite(ref).all() and not ref[45:].any()
    got = torch.ops.hgcalml.select_knn_grad(t(g), t(idx), t(np.zeros_like(g)), t(x))
    assert same(got.cpu().numpy(), ref)


@pytest.mark.parametrize("C", [1, 3, 4, 7, 9])
def test_distance_gradient_of_the_largest_gradients(oracle, C):
    """twice such a gradient is beyond the largest float, times the difference of two coordinates it is not"""
    from hgcalml_amd import ops  # noqa: F401
    rng = np.random.default_rng(400 + C)
    n, K = 60, 5
    idx = named_once(rng, n, K)
    x = (rng.random((n, C)) * 1e-3).astype(np.float32)
    x[1] = x[0]
    idx[0, 1] = 1              # a difference of 0
    g = (rng.choice([-1, 1], (n, K)) * np.float32(3e38)).astype(np.float32)
    ref = oracle.select_knn_grad_kernel(g, idx, x)
    assert np.isfinite(ref).all() and np.abs(ref).max() > 1e34
    got = torch.ops.hgcalml.select_knn_grad(t(g), t(idx), t(np.zeros_like(g)), t(x))
    assert same(got.cpu().numpy(), ref)
