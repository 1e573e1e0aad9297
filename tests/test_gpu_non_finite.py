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
