"""The gradients of the GravNet block's dense layers as passes of the library against the products in 64 bits, and which blocks take
them."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def check(got, terms, addend=None):
    """`terms`: (matrix, weight [out, in]) pairs whose products are added up. Every product and every addition is off by 2^-24
    of a partial sum at the most, and the absolute values bound those."""
    want = sum(a.double() @ w.double().t() for a, w in terms)
    size = sum(a.double().abs() @ w.double().abs().t() for a, w in terms)
    depth = sum(a.shape[1] for a, _ in terms)
    if addend is not None:
        want, size = want + addend.double(), size + addend.double().abs()
    assert ((got.double() - want).abs() <= (depth + 2) * 2.0 ** -24 * size + 1e-37).all()
    return want


# tiles of 16 columns and rows, widths of 4 up, remainders of both, several workgroups along the columns, the widest layers, every
# number of tiles a workgroup takes (output's gradient 4, 6, 8, 10, 12, input's 1 to 6, 8, 10, 12); with 150,011 rows a wave takes several tasks
@pytest.mark.parametrize("n", [1, 16, 17, 2061, 150011])
@pytest.mark.parametrize("x_width,f,c,o", [(4, 4, 1, 4), (5, 7, 2, 6), (16, 16, 4, 16), (17, 31, 3, 33), (64, 64, 4, 128),
                                           (96, 128, 4, 160), (13, 129, 3, 100), (256, 128, 4, 256), (412, 50, 2, 255),
                                           (48, 32, 3, 96), (70, 16, 4, 160), (180, 20, 4, 40), (500, 5, 1, 9)])
def test_passes(n, x_width, f, c, o):
    from hgcalml_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(n + f)

    def normal(*shape):
        return torch.randn(*shape, device=DEV, generator=gen)
    # x starts four bytes into its memory
    x = normal(n * x_width + 1)[1:].view(n, x_width)
    w_feat, bias, w_coords = normal(f, x_width), normal(f), normal(c, x_width)
    feat = torch.relu(torch.nn.functional.linear(x, w_feat, bias))
    acc, w, b = normal(n, 2 * f), normal(o, 2 * f + x_width), normal(o)
    out = torch.relu(torch.nn.functional.linear(ops.gravnet_join(acc, feat, x), w, b))
    g = normal(n, o)
    g_acc, g_feat, g_x, masked = ops.gravnet_output_layer_grad(g, out, w, f)
    assert torch.equal(masked, torch.where(out > 0, g, torch.zeros_like(g)))
    check(g_acc, [(masked, w[:, :2 * f].t())])
    check(g_x, [(masked, w[:, 2 * f:].t())])
    assert torch.equal(g_feat, -g_acc[:, :f] - g_acc[:, f:])

    feat = torch.relu(normal(n, f))
    for g2, g_c, g_x2, relu in ((normal(n, f), normal(n, c), g_x, True), (None, None, None, True), (None, normal(n, c), None, False)):
        g_in, masked = ops.gravnet_input_layers_grad(g_feat, g2, feat, g_c, g_x2, w_feat, w_coords, relu)
        total = g_feat if g2 is None else g_feat + g2
        assert torch.equal(masked, torch.where(feat > 0, total, torch.zeros_like(total)) if relu else total)
        check(g_in, [(masked, w_feat.t())] + ([] if g_c is None else [(g_c, w_coords.t())]), g_x2)


def test_non_finite_values_stay_in_their_rows():
    from hgcalml_amd import ops
    torch.manual_seed(3)
    x = torch.randn(37, 13, device=DEV)
    x[5, 12], x[20, 0] = float("nan"), float("inf")
    acc, feat = torch.randn(37, 20, device=DEV), torch.randn(37, 10, device=DEV)
    acc[20, 3], feat[5, 9] = float("-inf"), float("nan")
    w, b = torch.randn(18, 33, device=DEV), torch.randn(18, device=DEV)
    out = torch.relu(torch.nn.functional.linear(ops.gravnet_join(acc, feat, x), w, b))
    assert torch.isnan(out).any()
    # a result that is not a number passes its gradient on, as torch's relu does
    g = torch.randn(37, 18, device=DEV)
    g[30, 17], g[31, 0] = float("nan"), float("-inf")
    *grads, masked = ops.gravnet_output_layer_grad(g, out, w, 10)
    want = torch.ops.aten.threshold_backward(g, out, 0)
    assert torch.equal(masked.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))
    for grad, part in zip(grads, (w[:, :20], w[:, :10] + w[:, 10:20], w[:, 20:])):
        assert torch.equal(torch.isfinite(grad), torch.isfinite(want @ part))


@pytest.fixture
def layers_taken(monkeypatch):
    from hgcalml_amd import GravNetLayersRagged as module
    seen, real = [], module._InputLayersFn
    monkeypatch.setattr(module, "_InputLayersFn", types.SimpleNamespace(apply=lambda *args: seen.append(1) or real.apply(*args)))
    return seen


def block(sizes=(13, 9, 3, 30, 11), **kwargs):
    """inputs, neighbours, coordinates, outputs, features"""
    from hgcalml_amd import RaggedGravNet
    torch.manual_seed(8)
    return RaggedGravNet(*sizes, **kwargs).to(DEV)


X = dict(row_splits=[0, 5, 400, 700])


def step(layer, x, create_graph=False, second=False):
    rs = torch.tensor(X["row_splits"], dtype=torch.int32, device=DEV)
    layer.dynamic_radius.fill_(1.0)
    out, coords, idx, dist = layer(x, rs)
    wanted = [t for t in [x] + list(layer.parameters()) if t.requires_grad]
    loss = (out * out).sum() + (coords * coords).sum()
    if not second:
        loss = loss + (dist * torch.linspace(0, 1, dist.numel(), device=DEV).view(dist.shape)).sum()
    grads = torch.autograd.grad(loss, wanted, create_graph=create_graph)
    if second:  # the last layer's weight gradient once more, with respect to that weight and its bias and what is in front of them
        last, first = layer.output_feature_transform, layer.input_feature_transform
        at = [i for i, t in enumerate(wanted) if t is last.weight][0]
        grads = torch.autograd.grad((grads[at] * grads[at]).sum(), [last.weight, last.bias, first.weight, first.bias, x])
    return [out.detach()] + [g.detach() for g in grads]


def agree(a, b):
    for s, t in zip(a, b):
        assert (s.double() - t.double()).norm() <= 1e-5 * t.double().norm() + 1e-30


@pytest.mark.parametrize("frozen", [(), ("input_feature_transform.weight",), ("output_feature_transform.weight",),
                                    ("input_feature_transform.weight", "input_feature_transform.bias", "input_spatial_transform.weight")])
@pytest.mark.parametrize("x_grad", [True, False])
def test_block_with_parts_frozen(frozen, x_grad, layers_taken, monkeypatch):
    """the same operations as the layers one by one but for the order of their sums: 1e-5"""
    layer = block()
    for name, weight in layer.named_parameters():
        weight.requires_grad_(name not in frozen)
    x = torch.randn(700, 13, device=DEV, requires_grad=x_grad)
    got = step(layer, x)
    assert layers_taken == [1]
    monkeypatch.setattr(type(layer), "_layers_in_one_pass", lambda self, x: False)
    agree(got, step(layer, x))
    assert layers_taken == [1]


@pytest.mark.parametrize("activation", ["relu", "linear"])
def test_results_are_those_of_the_layers_one_by_one(activation, layers_taken, monkeypatch):
    """Bit for bit: every activation then lets the same gradients pass, and those differ by the order of their sums alone, 400 terms
    of float32 at the most in a row (400 * 2^-24 = 2.4e-5 of the terms' sizes, which a sum of the largest row's size is made of)."""
    from hgcalml_amd import RaggedGravNet
    torch.manual_seed(5)
    layer = RaggedGravNet(64, 16, 3, 128, 64, feature_activation=activation).to(DEV)
    x = torch.randn(60000, 64, device=DEV, requires_grad=True)
    rs = torch.tensor([0, 60000], dtype=torch.int32, device=DEV)
    weight = torch.randn(60000, 128, device=DEV)

    def once():
        layer.dynamic_radius.fill_(1.0)
        results = layer(x, rs)
        return results, torch.autograd.grad((results[0] * weight).sum(), [x] + list(layer.parameters()))
    (results, grads), taken = once(), list(layers_taken)
    monkeypatch.setattr(type(layer), "_layers_in_one_pass", lambda self, x: False)
    one_by_one, want = once()
    assert taken == layers_taken == [1]
    assert all(torch.equal(a, b) for a, b in zip(results, one_by_one))
    for a, b in zip(grads, want):
        assert (a - b).abs().max() <= 2.4e-5 * b.abs().max()


@pytest.mark.parametrize("frozen", [(), ("input_spatial_transform.weight",), ("input_feature_transform.weight", "input_feature_transform.bias"),
                                    ("input_feature_transform.weight", "input_feature_transform.bias", "input_spatial_transform.weight")])
@pytest.mark.parametrize("x_grad", [True, False])
@pytest.mark.parametrize("return_self", [True, False])
def test_frozen_parts_ask_for_no_gradient(frozen, x_grad, return_self, layers_taken, monkeypatch):
    """which results carry a gradient, and which gradients of search and accumulation a step forms: those of the layers one by one"""
    from hgcalml_amd import ops
    layer = block(return_self=return_self)
    for name, weight in layer.named_parameters():
        weight.requires_grad_(name not in frozen)
    x = torch.randn(700, 13, device=DEV, requires_grad=x_grad)
    rs = torch.tensor(X["row_splits"], dtype=torch.int32, device=DEV)
    calls = []
    for name in ("gravnet_drop_self_grad", "accumulate_gradient_index"):
        monkeypatch.setattr(ops, name, lambda *args, name=name, real=getattr(ops, name): calls.append(name) or real(*args))

    def once():
        calls.clear()
        results = layer(x, rs)
        results[0].sum().backward()
        return [t.requires_grad for t in results], list(calls)
    got, taken = once(), list(layers_taken)
    monkeypatch.setattr(type(layer), "_layers_in_one_pass", lambda self, x: False)
    assert got == once() and taken == layers_taken == [1]
    assert got[0][0] and got[0][1] == (x_grad or "input_spatial_transform.weight" not in frozen)


@pytest.mark.parametrize("frozen", [False, True])
def test_what_is_kept_for_the_gradient(frozen, layers_taken):
    """of the last layer its result and, for the weight's gradient, the joined rows; not what those were joined from"""
    layer = block()
    layer.output_feature_transform.weight.requires_grad_(not frozen)
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
        layer(torch.randn(700, 13, device=DEV), torch.tensor(X["row_splits"], dtype=torch.int32, device=DEV))
    assert layers_taken == [1]
    assert kept.count((700, 22)) == 0 and kept.count((700, 35)) == int(not frozen) and kept.count((700, 30)) == 1


@pytest.mark.parametrize("second", [False, True])
def test_derivative_of_the_derivative(second, layers_taken, monkeypatch):
    layer = block()
    x = torch.randn(700, 13, device=DEV, requires_grad=True)
    got = step(layer, x, create_graph=True, second=second)
    assert layers_taken == [1]
    monkeypatch.setattr(type(layer), "_layers_in_one_pass", lambda self, x: False)
    agree(got, step(layer, x, create_graph=True, second=second))


def test_blocks_that_are_left_alone(layers_taken):
    """hooks, replaced layers and methods, other activations, autocast, widths and strides that the passes do not take"""
    x = torch.randn(700, 13, device=DEV, requires_grad=True)
    calls = []
    layer = block()
    layer.output_feature_transform.register_forward_hook(lambda *args: calls.append(1))
    step(layer, x)
    assert calls == [1]
    layer = block()
    layer.input_feature_transform = torch.nn.Linear(13, 11).to(DEV)
    step(layer, x)
    layer = block()
    torch.nn.utils.parametrizations.weight_norm(layer.output_feature_transform)
    step(layer, x)
    layer = block()
    layer.update_dynamic_radius = lambda dist: calls.append(2)
    step(layer, x)
    step(block(feature_activation="tanh"), x)
    layer = block()
    step(layer, x.detach().t().contiguous().t().requires_grad_(True))
    for widths in ((13, 9, 5, 30, 11), (13, 9, 3, 30, 3), (13, 9, 3, 257, 11), (13, 9, 3, 30, 250), (13, 9, 3, 3, 11)):
        step(block(widths), x)
    step(block((3, 9, 3, 30, 11)), x.detach()[:, :3].contiguous().requires_grad_(True))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        layer(x, torch.tensor(X["row_splits"], dtype=torch.int32, device=DEV))
    assert layers_taken == [] and calls == [1, 2]
    with torch.no_grad():
        layer(x, torch.tensor(X["row_splits"], dtype=torch.int32, device=DEV))
    assert layers_taken == [1]


@pytest.mark.parametrize("n,k", [(1, 2), (700, 10), (333, 65)])
def test_scaled_distances_without_the_self_column(n, k):
    """the bits of the product by itself, both ways"""
    from hgcalml_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(n)
    dist, narrow, wide = (torch.randn(n, c, device=DEV, generator=gen) for c in (k, k - 1, k))
    idx = torch.randint(-1, n, (n, k), device=DEV, generator=gen, dtype=torch.int32)
    out_idx, out = ops.gravnet_drop_self(idx, dist, 10.0)
    assert torch.equal(out_idx, idx[:, 1:]) and torch.equal(out, 10.0 * dist[:, 1:])
    moved = torch.nn.functional.pad(10.0 * narrow, (1, 0))
    assert torch.equal(ops.gravnet_drop_self_grad(narrow, wide, 10.0), wide + moved)
    assert torch.equal(ops.gravnet_drop_self_grad(narrow, None, 10.0), moved)
