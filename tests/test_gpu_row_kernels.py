"""The accumulation kernels that give a vertex 16 lanes, at the sizes where their tiles end: columns around
the multiples of 16 and 64, rows around the multiples of 4 and 16 slots, a last wave with one to three vertices,
padded rows and a processing order. Bit for bit against the oracle (forward, feature gradient)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def bits(a):
    return np.ascontiguousarray(a).view(np.int32)


def table(rng, n, K):
    """others in random order, self in slot 0; some rows with a padded tail, an empty slot 0, repeated self, nothing"""
    idx = rng.integers(0, n, (n, K)).astype(np.int32)
    for v in range(n):
        others = np.delete(np.arange(n), v)
        row = rng.permutation(others)[:K - 1]
        idx[v, :1 + len(row)] = np.concatenate([[v], row])
        idx[v, 1 + len(row):] = -1
    kind = rng.integers(0, 8, n)
    for v in range(n):
        if kind[v] == 0:
            idx[v, K - rng.integers(0, K):] = -1
        elif kind[v] == 1:
            idx[v, 0] = -1
        elif kind[v] == 2:
            idx[v, K // 2:] = v
        elif kind[v] == 3 and rng.random() < 0.3:
            idx[v] = -1
    return idx


SHAPES = [(1, 1, 16), (2, 3, 17), (3, 4, 31), (5, 5, 32), (17, 15, 33), (66, 16, 47), (67, 17, 48), (65, 20, 49), (80, 33, 63),
          (90, 64, 64), (79, 65, 65), (70, 14, 96), (70, 24, 97), (81, 31, 127), (83, 48, 128), (71, 12, 129), (50, 40, 200),
          (40, 7, 260), (33, 80, 22)]


@pytest.mark.parametrize("n,K,F", SHAPES)
def test_forward_at_the_ends_of_tiles(oracle, n, K, F):
    from hgcalml_amd import ops
    rng = np.random.default_rng(n + 100 * K + 10000 * F)
    idx = table(rng, n, K)
    x = rng.standard_normal((n, F)).astype(np.float32)
    x[rng.random((n, F)) < 0.1] = 0
    w = rng.random((n, K), dtype=np.float32)
    for mm in (True, False):
        ref, rarg = oracle.AccumulateLinKnn(w, x, idx, mm)
        for order in (None, rng.permutation(n).astype(np.int32)):
            ti = t(idx)
            if order is not None:
                ops.set_vertex_order(ti, t(order))
            out, arg, slots = torch.ops.hgcalml.accumulate_knn_slots(t(w), t(x), ti, 0, mm)
            assert (bits(out.cpu().numpy()) == bits(ref)).all()
            if mm:
                assert (arg.cpu().numpy() == rarg).all()
                sl = slots.cpu().numpy().astype(int)
                named = np.where(sl < K, np.take_along_axis(idx, np.minimum(sl, K - 1), 1), 0)
                assert (named == rarg).all()
