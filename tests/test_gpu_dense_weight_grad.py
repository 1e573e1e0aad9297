"""`hgc_dense_weight_grad` (weight and bias gradient of a dense layer over many rows) against the products in 64 bits, at
the widths where its blocks and loads change and the row counts where its slabs, batches and steps end."""
import pytest
import torch

from hgcalml_amd import ops
from hgcalml_amd.GravNetLayersRagged import TallLinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def check(g, x):
    weight, bias = ops.dense_weight_grad(g, x)
    g64, x64 = g.cpu().double(), x.cpu().double()
    # A term takes part in at most as many additions as a wave's slab has rows (256 parts of the rows, 128 or more where the
    # result takes two workgroups, rounded up to a batch of 32), the four rows of a step and the slabs of a workgroup
    # (16) and the parts (32 by one thread, 8 threads) add theirs, and it is rounded once itself: each addition is off by
    # 2^-24 of the sum of the terms' sizes at most.
    n = len(g)
    bound = (min(n, n // 128 + 32) + 4 + 16 + 32 + 8 + 1) * 2.0 ** -24
    assert ((weight.cpu() - g64.t() @ x64).abs() <= bound * (g64.abs().t() @ x64.abs())).all()
    assert ((bias.cpu() - g64.sum(0)).abs() <= bound * g64.abs().sum(0)).all()


# widths: 1 to 4 tiles of 16 columns, a block of 64 and one more column, three blocks, and remainders of every load width
@pytest.mark.parametrize("n_out,n_in", [(1, 1), (3, 64), (4, 29), (16, 17), (22, 29), (31, 33), (48, 73), (49, 50), (64, 65),
                                        (63, 130), (96, 112), (129, 193), (128, 192), (160, 352)])
# rows: none of a step's four, one more and less than a step, a batch, a wave's least rows, a slab, many parts
@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 65, 1027, 2477, 70003])
def test_against_64_bits(n, n_out, n_in):
    gen = torch.Generator().manual_seed(n * 1000 + n_out + n_in)
    check(torch.randn(n, n_out, generator=gen).to(DEV), torch.randn(n, n_in, generator=gen).to(DEV))


def test_every_row_counts_once_and_rows_off_a_16_byte_boundary():
    n, n_out, n_in = 40013, 23, 37
    g = torch.zeros(n * n_out + 1, device=DEV)[1:].view(n, n_out)
    x = torch.zeros(n * n_in + 3, device=DEV)[3:].view(n, n_in)
    g[:] = 1.0
    x[:] = torch.arange(n_in, device=DEV, dtype=torch.float32) % 5  # whole numbers, sums below 2^24: exact
    weight, bias = ops.dense_weight_grad(g, x)
    assert torch.equal(weight, (n * (torch.arange(n_in, device=DEV) % 5).float()).expand(n_out, n_in))
    assert torch.equal(bias, torch.full((n_out,), float(n), device=DEV))


@pytest.mark.parametrize("n_out,n_in", [(1, 1), (3, 64), (4, 29), (16, 17), (22, 29), (31, 33), (48, 73), (49, 50), (64, 65),
                                        (63, 130), (96, 112), (129, 193), (128, 192), (160, 352)])
# from no batch to many in a slab, odd and even numbers of them, one part of the result to 256
@pytest.mark.parametrize("n", [1, 15, 33, 64, 96, 100, 131, 1027, 2477, 8192, 40013, 70003, 150000])
def test_every_row_counts_once_at_all_widths(n, n_out, n_in):
    """whole numbers whose sums stay below 2^24 are exact in any order: no row, batch, slab or part lost or counted twice"""
    row = torch.arange(n, device=DEV)[:, None]
    g = ((row * 5 + torch.arange(n_out, device=DEV) * 3) % 7 - 2).float()   # -2 .. 4
    x = ((row // 3 + torch.arange(n_in, device=DEV)) % 11 - 4).float()      # -4 .. 6
    weight, bias = ops.dense_weight_grad(g, x)
    assert torch.equal(weight.double(), g.double().t() @ x.double())
    assert torch.equal(bias.double(), g.double().sum(0))


def test_values_that_are_no_numbers_stay_in_their_columns():
    n, n_out, n_in = 1030, 30, 45
    gen = torch.Generator().manual_seed(5)
    g, x = torch.randn(n, n_out, generator=gen).to(DEV), torch.randn(n, n_in, generator=gen).to(DEV)
    g[n - 1, 7] = float("inf")
    x[n - 1, 44] = float("nan")
    weight, bias = ops.dense_weight_grad(g, x)
    bad = torch.zeros(n_out, n_in, dtype=torch.bool, device=DEV)
    bad[7, :] = True
    bad[:, 44] = True
    assert torch.equal(~torch.isfinite(weight), bad)
    assert torch.isinf(bias[7]) and torch.isfinite(bias).sum() == n_out - 1


@pytest.fixture
def passes(monkeypatch):
    """the shapes that reach the one pass"""
    seen, real = [], ops.dense_weight_grad

    def spy(grad, x):
        seen.append((tuple(grad.shape), tuple(x.shape)))
        return real(grad, x)
    monkeypatch.setattr(ops, "dense_weight_grad", spy)
    return seen


# up to 2^15 weights over any rows, up to 2^16 over 2^16 rows
@pytest.mark.parametrize("n,n_in,n_out,taken", [(70000, 256, 128, True), (70000, 257, 128, False), (65536, 256, 256, True),
                                                (65537, 256, 256, False), (300, 257, 256, False), (65537, 100, 70, True)])
def test_which_layers_take_the_one_pass(n, n_in, n_out, taken, passes):
    torch.manual_seed(1)
    layer = TallLinear(n_in, n_out).to(DEV)
    x = torch.randn(n, n_in, device=DEV)
    g = torch.randn(n, n_out, device=DEV)
    weight, bias = torch.autograd.grad(layer(x), [layer.weight, layer.bias], g)
    assert passes == ([((n, n_out), (n, n_in))] if taken else [])
    want = g.double().t() @ x.double()
    # sums of n terms of either sign, in parts of n / 64 rows at the most: as in check()
    bound = (n / 64 + 100) * 2.0 ** -24
    assert ((weight.double() - want).abs() <= bound * (g.abs().double().t() @ x.abs().double())).all()
    assert ((bias.double() - g.double().sum(0)).abs() <= bound * g.abs().double().sum(0)).all()


@pytest.mark.parametrize("n", [1, 700, 5000])
def test_layer_gradients(n, passes):
    """the layer's gradients with and without a second derivative asked for, and through a captured graph"""
    torch.manual_seed(n)
    layer = TallLinear(45, 30).to(DEV)
    x = torch.randn(n, 45, device=DEV, requires_grad=True)
    g = torch.randn(n, 30, device=DEV)
    one = torch.autograd.grad(layer(x), [x, layer.weight, layer.bias], g)
    assert passes == [((n, 30), (n, 45))]
    two = torch.autograd.grad(layer(x), [x, layer.weight, layer.bias], g, create_graph=True)
    assert len(passes) == 1  # a second derivative is left to the tensor operations
    for a, b in zip(one, two):
        assert (a - b).abs().max() <= 1e-5 * (b.abs().max() + 1)
    static = torch.empty_like(g)
    static.copy_(g)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.dense_weight_grad(static, x.detach())
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = ops.dense_weight_grad(static, x.detach())
    for scale in (1.0, 2.0, -3.0):
        static.copy_(scale * g)
        graph.replay()
        torch.cuda.synchronize()
        eager = ops.dense_weight_grad(scale * g, x.detach())
        assert all(torch.equal(a, b) for a, b in zip(captured, eager))
