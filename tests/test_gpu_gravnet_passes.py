"""The memory passes of the GravNet block against the tensor operations they stand for: equal bits where nothing is
summed, at odd widths, single rows and the ends of workgroups; the block with the passes against the block without."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n,k", [(1, 2), (3, 3), (5, 2), (127, 4), (255, 17), (1000, 65), (1025, 41)])
def test_drop_self(n, k):
    from hgcalml_amd import ops
    g = torch.Generator().manual_seed(n * k)
    idx = torch.randint(-1, n, (n, k), generator=g, dtype=torch.int32).to(DEV)
    d = torch.rand(n, k, generator=g).to(DEV)
    got_idx, got = ops.gravnet_drop_self(idx, d)
    assert torch.equal(got_idx, idx[:, 1:]) and torch.equal(got, d[:, 1:])
    narrow, wide = torch.randn(n, k - 1, generator=g).to(DEV), torch.randn(n, k, generator=g).to(DEV)
    padded = torch.nn.functional.pad(narrow, (1, 0))
    assert torch.equal(ops.gravnet_drop_self_grad(narrow, None), padded)
    assert torch.equal(ops.gravnet_drop_self_grad(narrow, wide), wide + padded)
    assert torch.equal(ops.gravnet_drop_self_grad(narrow, wide.t().contiguous().t()), wide + padded)
    odd = torch.randn(n * k + 1, generator=g).to(DEV)[1:].view(n, k)  # not on a 16-byte boundary
    assert torch.equal(ops.gravnet_drop_self_grad(narrow, odd), odd + padded)


@pytest.mark.parametrize("n,f,w", [(1, 1, 1), (7, 3, 5), (64, 16, 4), (333, 22, 29), (100, 64, 64), (257, 32, 48),
                                   (3, 300, 700), (2, 4, 4), (1000, 5, 8)])
def test_join(n, f, w):
    from hgcalml_amd import ops
    g = torch.Generator().manual_seed(n + f + w)
    acc, p, x = (torch.randn(n, c, generator=g).to(DEV) for c in (2 * f, f, w))
    assert torch.equal(ops.gravnet_join(acc, p, x), torch.cat([acc - p.repeat(1, 2), x], dim=1))
    grad = torch.randn(n, 2 * f + w, generator=g).to(DEV)
    for wanted in ((True, True, True), (False, True, False), (True, False, False), (False, False, True)):
        got = ops.gravnet_join_grad(grad, f, *wanted)
        for a, b, want in zip(got, (grad[:, :2 * f], -grad[:, :f] - grad[:, f:2 * f], grad[:, 2 * f:]), wanted):
            assert torch.equal(a, b) if want else a.numel() == 0


def additions(n, c, vec):
    """the longest chain of float32 additions a column goes through: the rows of a thread one after the other, the workgroup's
    groups of threads one after the other, and both again over the slabs' sums (the split column_sums takes)"""
    cols = c // vec
    tile = min(32, cols)
    slab = max(16 * (256 // tile), -(-n // max(1, 512 // -(-cols // tile))))
    slabs = -(-n // slab)
    chain = -(-min(slab, n) // (256 // tile)) + 256 // tile
    narrowest = min(tile, cols % tile or tile)   # a narrow last tile has the more groups, none has longer chains of rows
    chain = max(chain, -(-min(slab, n) // (256 // narrowest)) + 256 // narrowest)
    if slabs > 1:
        last = min(8, cols)
        narrowest = min(last, cols % last or last)
        chain += max(-(-slabs // (256 // w)) + 256 // w for w in (last, narrowest))
    return chain


@pytest.mark.parametrize("n,c", [(1, 1), (1, 130), (255, 7), (256, 48), (513, 1), (2477, 48), (64, 24576), (64, 4099),
                                 (150000, 128), (70001, 33), (8192, 4), (9000, 516)])
def test_column_sums(n, c):
    """every addition of a chain is off by 2^-24 of a partial sum, which the sum of the absolute values bounds"""
    from hgcalml_amd import ops
    x = torch.randn(n, c, generator=torch.Generator().manual_seed(n + c))
    shifted = torch.randn(n * c + 1, generator=torch.Generator().manual_seed(c)).to(DEV)[1:].view(n, c)
    for on_gpu, vec in ((x.to(DEV), 4 if c % 4 == 0 else 1), (shifted, 1)):
        exact, got = on_gpu.cpu().double(), ops.column_sums(on_gpu).cpu().double()
        bound = additions(n, c, vec) * 2.0 ** -24 * exact.abs().sum(0)
        assert ((got - exact.sum(0)).abs() <= 1.0001 * bound).all()
    # (about a hundred additions for a tall matrix of ordinary width)
    assert additions(150000, 128, 4) == 37 + 8 + 16 + 32


@pytest.mark.parametrize("n", [2**31 - 1, 2**31 - 257, 2**31 + 5])
def test_column_sums_of_the_tallest_matrices(n):
    """the last rows of the last slab, and more rows than the library counts; whole numbers, so that every order is exact"""
    from hgcalml_amd import ops
    from hgcalml_amd.GravNetLayersRagged import _sum_rows
    x = torch.zeros(n, 1, device=DEV)
    marks = [0, 1, n // 2, n - 5000000, n - 300, n - 2, n - 1]
    for i, row in enumerate(marks):
        x[row] = 2.0 ** i
    with torch.no_grad():
        assert _sum_rows(x).tolist() == [2.0 ** len(marks) - 1]
    if n < 2**31:
        assert ops.column_sums(x).tolist() == [2.0 ** len(marks) - 1]


@pytest.mark.parametrize("total,high", [(1, 1.0), (2, 30.0), (1023, 0.01), (4097, 1.0), (3000001, 9.0)])
def test_radius_step(total, high):
    from hgcalml_amd import ops
    d = torch.rand(total, 1, generator=torch.Generator().manual_seed(total)).to(DEV) * high
    radius = torch.tensor(0.7, device=DEV)

    def step(d, radius):
        dist = d.double().sqrt()
        return 0.05 * (torch.maximum((dist.max() * 1.05).clamp(max=2.0), 2.0 * dist.mean()) + 1e-3 - radius.double())
    # a root, three products and a rounded sum in float32, each off by 2^-24 of values below 6
    assert abs(float(ops.gravnet_radius_step(d, radius)) - float(step(d, radius))) <= 6 * 8 * 2.0 ** -24
    d[total // 2] = float("nan")
    assert torch.isnan(ops.gravnet_radius_step(d, radius))


@pytest.mark.parametrize("return_self,sumw", [(True, False), (False, False), (True, True)])
def test_block_with_and_without_the_passes(return_self, sumw, monkeypatch):
    """same operations in the same order but for sums over rows and the order of two gradients added: 1e-5"""
    from hgcalml_amd import GravNetLayersRagged as module
    torch.manual_seed(5)
    layer = module.RaggedGravNet(13, 9, 3, 30, 11, return_self=return_self, sumwnorm=sumw).to(DEV)
    x = torch.randn(901, 13, device=DEV)
    rs = torch.tensor([0, 5, 400, 901], dtype=torch.int32, device=DEV)  # the first event has padded rows

    def once():
        layer.dynamic_radius.fill_(1.0)
        xx = x.clone().requires_grad_(True)
        out, coords, idx, dist = layer(xx, rs)
        loss = (out * out).sum() + (dist * torch.linspace(0, 1, dist.numel(), device=DEV).view(dist.shape)).sum()
        return [out, coords, idx, dist, layer.dynamic_radius.clone()] + list(
            torch.autograd.grad(loss, [xx] + list(layer.parameters())))
    fused = once()
    monkeypatch.setattr(module, "_library_takes", lambda *tensors: False)
    for a, b in zip(fused, once()):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert (a.double() - b.double()).norm() <= 1e-5 * b.double().norm()


@pytest.mark.parametrize("return_self", [True, False])
@pytest.mark.parametrize("passes", [True, False])
def test_returned_distances_may_be_written_to(return_self, passes, monkeypatch):
    """in place, before the gradient is asked for: what it is without writing, times the factor"""
    from hgcalml_amd import GravNetLayersRagged as module
    if not passes:
        monkeypatch.setattr(module, "_library_takes", lambda *tensors: False)
    torch.manual_seed(6)
    layer = module.RaggedGravNet(5, 4, 3, 6, 7, return_self=return_self).to(DEV)
    x = torch.randn(200, 5, device=DEV, requires_grad=True)
    rs = torch.tensor([0, 3, 200], dtype=torch.int32, device=DEV)

    def gradient(in_place):
        _, _, _, dist = layer(x, rs)
        dist = dist.mul_(4.0) if in_place else dist * 4.0
        return dist.detach().clone(), torch.autograd.grad(dist.sum(), x)[0]
    for a, b in zip(gradient(True), gradient(False)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,k,f", [(1, 1, 1), (17, 5, 3), (33, 16, 15), (100, 17, 32), (64, 40, 33), (90, 70, 130)])
def test_weights_sum(n, k, f):
    """against the composition with a column of ones: equal bits forward; backward the order of a sum of 2 f + 1 products and
    the rounding of 1 / norm differ"""
    from hgcalml_amd import AccumulateKnnSumw
    from hgcalml_amd.accknn_op import _AccumulateSumwFn
    g = torch.Generator().manual_seed(n + k + f)
    idx = torch.rand(n, n, generator=g).argsort(1)[:, :k].to(torch.int32)   # different neighbours in each row
    idx[torch.rand(n, generator=g) < 0.2, k // 2:] = -1
    idx[0] = -1                                      # a row without neighbours: 0, and no gradient
    idx = idx.to(DEV)
    d = torch.rand(n, k, generator=g).to(DEV).requires_grad_(True)
    x = torch.randn(n, f, generator=g).to(DEV).requires_grad_(True)
    grad = torch.randn(n, 2 * f, generator=g).to(DEV)
    want = AccumulateKnnSumw(d, x, idx, mean_and_max=True)[0]
    got = _AccumulateSumwFn.apply(d, x, idx)
    assert torch.equal(got, want)
    for a, b in zip(torch.autograd.grad(got, [d, x], grad), torch.autograd.grad(want, [d, x], grad)):
        assert torch.isfinite(a).all()
        assert (a - b).norm() <= 1e-5 * b.norm() + 1e-30
    assert (torch.autograd.grad(_AccumulateSumwFn.apply(d, x, idx), d, grad)[0][idx < 0] == 0).all()
    # the result may be written to in place before its gradient is asked for
    written = _AccumulateSumwFn.apply(d, x, idx)
    written -= x.detach().repeat(1, 2)
    for a, b in zip(torch.autograd.grad(written, [d, x], grad),
                    torch.autograd.grad(_AccumulateSumwFn.apply(d, x, idx), [d, x], grad)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,k,f", [(2, 1, 16), (17, 3, 17), (66, 15, 33), (67, 16, 64), (90, 17, 65), (83, 40, 128), (70, 64, 48),
                                   (40, 5, 130), (40, 5, 8)])
@pytest.mark.parametrize("mean_and_max", [True, False])
def test_gradient_with_the_index_of_the_whole_table(n, k, f, mean_and_max):
    """bit for bit the gradients with the narrow table's own index, for padded rows and whatever column 0 holds; shapes the
    kernel does not cover are given the narrow index"""
    from hgcalml_amd import AccumulateKnn, ops
    g = torch.Generator().manual_seed(n + k + f)
    part = torch.rand(n, n, generator=g).argsort(1)[:, :k].to(torch.int32)
    part[torch.rand(n, generator=g) < 0.3, k // 2:] = -1
    first = torch.where(torch.rand(n, generator=g) < 0.7, torch.arange(n), torch.randint(-1, n, (n,), generator=g))
    whole = torch.cat([first.to(torch.int32)[:, None], part], dim=1).to(DEV)
    d = torch.rand(n, k, generator=g).to(DEV).requires_grad_(True)
    x = torch.randn(n, f, generator=g).to(DEV).requires_grad_(True)
    grad = torch.randn(n, 2 * f if mean_and_max else f, generator=g).to(DEV)
    results = []
    for declared in (False, True):
        table = part.to(DEV)
        if declared:
            ops.declare_without_first_column(table, whole)
            index = ops.accumulate_gradient_index(table, f, mean_and_max)
            assert index[1].numel() == n * (k + 1 if 16 <= f <= 128 else k)
        out = AccumulateKnn(d, x, table, mean_and_max=mean_and_max)[0]
        results.append(torch.autograd.grad(out, [d, x], grad))
    for a, b in zip(*results):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
