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


# rows of whole waves of 16-byte loads, which a wave per vertex takes: slots around its eight at a time and the 64 whose
# weights it forms itself
WAVE_SHAPES = [(1, 1, 256), (5, 4, 256), (33, 7, 256), (40, 8, 256), (41, 9, 512), (50, 13, 256), (30, 16, 768), (40, 31, 256),
               (50, 32, 256), (47, 37, 256), (60, 43, 256), (81, 64, 256), (83, 65, 256), (90, 66, 512)]


@pytest.mark.parametrize("n,K,F", SHAPES + WAVE_SHAPES)
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


@pytest.mark.parametrize("n,K,F", WAVE_SHAPES)
@pytest.mark.parametrize("mm", [True, False])
def test_forward_of_whole_waves_against_sixteen_lanes(n, K, F, mm):
    """bit for bit what 16 lanes per vertex give, which take the same rows from a matrix that is not on a 16-byte
    boundary; infinities and NaN among the features, exp(-d) inside and outside"""
    rng = np.random.default_rng(n + K + F)
    idx = table(rng, n, K)
    x = rng.standard_normal((n, F)).astype(np.float32)
    x[rng.random((n, F)) < 0.05] = np.inf
    x[rng.random((n, F)) < 0.05] = -np.inf
    x[rng.random((n, F)) < 0.02] = np.nan
    x[0] = np.nan
    d, ti = t(rng.random((n, K), dtype=np.float32)), t(idx)
    shifted = torch.empty(n * F + 1, device=DEV)[1:].view(n, F)
    shifted.copy_(t(x))
    for op in (torch.ops.hgcalml.accumulate_knn_slots, torch.ops.hgcalml.accumulate_knn_exp_slots):
        for a, b in zip(op(d, t(x), ti, 0, mm), op(d, shifted, ti, 0, mm)):
            if a.dtype == torch.float32:
                assert torch.equal(torch.isnan(a), torch.isnan(b))
                a, b = torch.nan_to_num(a, nan=0.5), torch.nan_to_num(b, nan=0.5)
            assert torch.equal(a, b)


@pytest.mark.parametrize("n,K,F", SHAPES)
def test_gradient_at_the_ends_of_tiles(oracle, n, K, F):
    """both gradients with and without the quotients' scratch memory, w.r.t. weights and (weights_are_exp) distances;
    lists of very different length in one workgroup"""
    from hgcalml_amd import ops
    from hgcalml_amd._lib import check, lib, p, stream
    rng = np.random.default_rng(n + 200 * K + 20000 * F)
    idx = table(rng, n, K)
    hub = rng.integers(0, min(n, 5), n)  # many rows name the same few vertices
    for v in range(0, n, 3):
        if K > 1 and hub[v] not in idx[v]:
            idx[v, K - 1] = hub[v]
    x = rng.standard_normal((n, F)).astype(np.float32)
    w = rng.random((n, K), dtype=np.float32)
    ti, tw, tx = t(idx), t(w), t(x)
    inv = ops.inverse_neighbour_index(ti)
    for mm in (True, False):
        g = rng.standard_normal((n, 2 * F if mm else F)).astype(np.float32)
        _, rarg = oracle.AccumulateLinKnn(w, x, idx, mm)
        rgw, rgx = oracle.accumulate_knn_grad_kernel(g, w, x, idx, rarg)
        _, arg, slots = torch.ops.hgcalml.accumulate_knn_slots(tw, tx, ti, 0, mm)
        need = lib.hgc_accumulate_knn_grad_scratch_bytes(n, K, F, int(mm))
        # 1e-5 of the sum of the absolute terms of a dot product of F (2 F) float32 products
        absx = np.abs(x[np.maximum(idx, 0)])
        tol = 1e-5 * (absx * (np.abs(g[:, :F]) / K + (np.abs(g[:, F:]) if mm else 0))[:, None, :]).sum(-1) + 1e-30
        order = t(rng.permutation(n).astype(np.int32))
        for with_scratch, exp in ((False, False), (True, False), (True, True)):
            gw, gx = torch.empty_like(tw), torch.empty_like(tx)
            scratch = torch.empty(max(need, 256), dtype=torch.uint8, device=DEV) if with_scratch else None
            check(lib.hgc_accumulate_knn_grad_scratch(p(t(g)), p(tw), p(tx), p(arg), p(slots) if slots.numel() else None, p(ti),
                                                      p(inv[0]), p(inv[1]), p(order) if exp else None, p(gw), p(gx), n, K, F,
                                                      g.shape[1], int(mm), int(exp), p(scratch),
                                                      scratch.numel() if with_scratch else 0, stream()))
            assert (bits(gx.cpu().numpy()) == bits(rgx)).all()
            got, want = gw.cpu().numpy(), -(rgw * w) if exp else rgw
            assert (np.abs(got - want) <= tol).all()
            assert (got[idx < 0] == 0).all()


def test_gradient_of_the_largest_matrix_of_quotients():
    """8,388,480 rows of 64 features, K no power of two: the gradient matrix ends where 32-bit offsets do, that of its quotients
    at half of it; lists of two entries, so that most of the 16 places of a step lie beyond them"""
    from hgcalml_amd import ops
    if torch.cuda.mem_get_info()[0] < 48 << 30:
        pytest.skip("needs 48 GB of device memory")
    n, K, F = 8388480, 3, 64
    gen = torch.Generator(device=DEV)
    gen.manual_seed(7)
    v = torch.arange(n, device=DEV, dtype=torch.int32)
    idx = torch.stack([v, (v + 1) % n, torch.full_like(v, -1)], 1)
    w = torch.rand(n, K, device=DEV, generator=gen)
    x = torch.randn(n, F, device=DEV, generator=gen)
    g = torch.randn(n, 2 * F, device=DEV, generator=gen)
    slots = torch.randint(0, 3, (n, F), device=DEV, generator=gen, dtype=torch.uint8)   # 2: nobody's
    arg = torch.zeros(n, F, device=DEV, dtype=torch.int32)                              # not read where there are slots
    gw, gx = torch.ops.hgcalml.accumulate_knn_grad_slots(g, w, x, idx, arg, slots, *ops.inverse_neighbour_index(idx))
    del arg

    divisor = torch.full((F,), float(K), device=DEV)   # (torch multiplies by the reciprocal of a number)

    def part(rows, slot):
        up, ww = g[rows], w[rows, slot, None]
        return up[:, :F] / divisor * ww + torch.where(slots[rows] == slot, up[:, F:], torch.zeros_like(up[:, F:])) * ww
    for s in range(0, n, 1 << 20):
        rows = torch.arange(s, min(n, s + (1 << 20)), device=DEV)
        own, named = part(rows, 0), part((rows - 1) % n, 1)
        assert torch.equal(gx[rows], torch.where((rows == 0)[:, None], own + named, named + own))   # ascending (vertex, slot)
        for slot in (0, 1):
            xx, up = x[(rows + slot) % n].double(), g[rows].double()
            terms = up[:, :F] * xx / K + torch.where(slots[rows] == slot, up[:, F:] * xx, torch.zeros_like(xx))
            # at most 2 F products, sums and one quotient, each rounded once
            assert bool(((gw[rows, slot].double() - terms.sum(1)).abs() <=
                         (2 * F + 2) * 2.0 ** -24 * ((up[:, :F] * xx).abs().sum(1) + (up[:, F:] * xx).abs().sum(1))).all())
        assert not gw[rows, 2].any()
    del g, x, w, slots, gw, gx, idx, v
    torch.cuda.empty_cache()
