"""`RaggedGravNet` — the GravNet block that sits directly on top of the custom-op
path (modules/GravNetLayersRagged.py:3095-3283 of the reference), as a
``torch.nn.Module``: learned coordinates -> BinnedSelectKnn -> AccumulateKnn of
the propagated features with weights exp(-10 d^2) -> output transform.

Only the exact kNN is built (the reference asserts the same,
GravNetLayersRagged.py:3135). Gradients flow through the accumulated features
(AccumulateKnnGrad), through the distances into the coordinates (SelectKnnGrad)
and through the dense layers (torch).
"""
import torch
from torch import nn
from torch.nn.modules.module import _has_any_global_hook

from . import globals as gl
from . import ops
from .accknn_op import AccumulateKnn, AccumulateKnnSumw, _AccumulateSumwFn
from .binned_select_knn_op import BinnedSelectKnn


def eye_init_(weight, mean=0.0, stddev=0.1, eye_scaling=1.0):
    """identity + normal noise (modules/Initializers.py:4-26); `weight` is
    [out, in] as torch stores it, the identity is laid on the [in, out] view"""
    with torch.no_grad():
        weight.normal_(mean, stddev)
        n_out, n_in = weight.shape
        weight += torch.eye(n_in, n_out, dtype=weight.dtype, device=weight.device).t() * eye_scaling
    return weight


def _library_takes(*tensors):
    """whether the library's passes stand for the tensor operations: float32 on one GPU, at least one row, no
    derivative of the derivative asked for, and neither switch that asks for differentiable compositions"""
    if gl.knn_ops_use_tf_gradients or gl.acc_ops_use_tf_gradients:
        return False
    return all(t.is_cuda and t.dtype == torch.float32 and t.numel() > 0 and t.device == tensors[0].device
               for t in tensors)


def _sum_rows(t):
    """t.sum(0)"""
    if torch.is_grad_enabled() or not _library_takes(t) or t.shape[0] >= 1 << 31 or t[0].numel() > 1 << 20:
        return t.sum(0)
    return ops.column_sums(t.reshape(t.shape[0], -1)).view(t.shape[1:])


def _weight_grad_in_one_pass(g, x):
    """Whether weight and bias gradient of a dense layer come from the library's one pass over g and x. Wide layers over
    many rows are the batched product's (us with the bias' sums, one pass / batched: 240,000 rows, 160 x 352 371 / 300;
    150,000, 160 x 256 139 / 141, 128 x 256 93 / 112; 65,536, 256 x 256 90 / 88; 60,000, 160 x 352 98 / 122; 20,000 43 / 85)."""
    widths = g.shape[1] * x.shape[1]
    return (not torch.is_grad_enabled() and _library_takes(g, x) and
            (widths <= 1 << 15 or (widths <= 1 << 16 and x.shape[0] <= 1 << 16)))


class _DropSelfFn(torch.autograd.Function):
    """table and distances (times `scale`) without the self column, and the distances themselves: the gradients of both come
    back in one pass. The distances leave as a tensor of their own on the same memory, which may be written to (an input handed
    back would be a view that refuses it): the block reads them no more, and neither does the search's gradient."""

    @staticmethod
    def forward(ctx, idx, dist, scale):
        ctx.set_materialize_grads(False)
        ctx.scale = scale
        nidx, ndist = ops.gravnet_drop_self(idx, dist, scale)
        ctx.mark_non_differentiable(nidx)
        return nidx, ndist, dist.data

    @staticmethod
    def backward(ctx, _grad_nidx, grad_narrow, grad_wide):
        if grad_narrow is None:
            return None, grad_wide, None
        if torch.is_grad_enabled():
            grad = torch.nn.functional.pad(ctx.scale * grad_narrow, (1, 0))
            return None, grad if grad_wide is None else grad + grad_wide, None
        return None, ops.gravnet_drop_self_grad(grad_narrow, grad_wide, ctx.scale), None


class _JoinFn(torch.autograd.Function):
    """[accumulated - (features | features) | x] and its gradients, one pass each"""

    @staticmethod
    def forward(ctx, accumulated, features, x):
        ctx.n_features = features.shape[1]
        return ops.gravnet_join(accumulated, features, x)

    @staticmethod
    def backward(ctx, grad):
        f = ctx.n_features
        if torch.is_grad_enabled():
            return grad[:, :2 * f], -grad[:, :f] - grad[:, f:2 * f], grad[:, 2 * f:]
        out = ops.gravnet_join_grad(grad, f, *ctx.needs_input_grad)
        return tuple(g if want else None for g, want in zip(out, ctx.needs_input_grad))


def _weight_and_bias_grad(g, x, want_bias):
    """(g^T x, sum over the rows of g): gradients of a dense layer over very many rows. The product reduces over those
    rows into a small matrix; as one GEMM it runs on a handful of workgroups (0.35-0.44 ms for 150k rows of 64-192
    columns). The library's pass forms it together with the bias gradient; where that one is not taken, a batch of 64 row
    slices is added up afterwards."""
    if _weight_grad_in_one_pass(g, x):
        return ops.dense_weight_grad(g, x)
    n, s = x.shape[0], _TallLinearFn.SLICES
    whole = n // s * s
    if whole >= 64 * s:
        grad_w = torch.bmm(g[:whole].view(s, -1, g.shape[1]).transpose(1, 2), x[:whole].view(s, -1, x.shape[1]))
        grad_w = _sum_rows(grad_w)
        if whole < n:
            grad_w = grad_w + g[whole:].t() @ x[whole:]
    else:
        grad_w = g.t() @ x
    return grad_w, _sum_rows(g) if want_bias else None


class _TallLinearFn(torch.autograd.Function):
    """y = x W^T + b for x of very many rows, see _weight_and_bias_grad"""

    SLICES = 64

    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        return torch.nn.functional.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors
        g = g.contiguous()
        grad_x = g @ weight if ctx.needs_input_grad[0] else None
        want_b = ctx.has_bias and ctx.needs_input_grad[2]
        if not ctx.needs_input_grad[1]:
            return grad_x, None, _sum_rows(g) if want_b else None
        grad_w, grad_b = _weight_and_bias_grad(g, x, want_b)
        return grad_x, grad_w, grad_b if want_b else None


class _InputLayersFn(torch.autograd.Function):
    """The block's two layers on x. Features and x leave twice, the second time as tensors of their own on the same
    memory, for the block's last layer: what comes back for them is added in the pass that forms the gradient of x."""

    @staticmethod
    def forward(ctx, x, w_features, bias, w_coords, relu):
        ctx.set_materialize_grads(False)
        # library products: their last bits decide which neighbours are near, largest and passed on at all (dense_rows.hip)
        coords = torch.nn.functional.linear(x, w_coords)
        features = torch.nn.functional.linear(x, w_features, bias)
        if relu:
            features = features.relu_()
        ctx.save_for_backward(x, w_features, w_coords, features)
        ctx.relu = relu
        outputs = features, coords, features.data, x.data
        # an output that depends on nothing that wants a gradient wants none either: what follows is spared its part of it
        want_x, want_wf, want_b, want_wc, _ = ctx.needs_input_grad
        wanted = want_x or want_wf or want_b, want_x or want_wc, want_x or want_wf or want_b, want_x
        ctx.mark_non_differentiable(*(t for t, want in zip(outputs, wanted) if not want))
        return outputs

    @staticmethod
    def backward(ctx, g_features, g_coords, g_features2, g_x):
        x, w_features, w_coords, features = ctx.saved_tensors
        want_x, want_wf, want_b, want_wc, _ = ctx.needs_input_grad
        if g_features is None:
            g_features, g_features2 = g_features2, None
        grad_x = masked = None
        if want_x and g_features is not None and not torch.is_grad_enabled():
            grad_x, masked = ops.gravnet_input_layers_grad(g_features, g_features2, features, g_coords, g_x, w_features, w_coords,
                                                           ctx.relu)
        else:  # as tensor operations: derivatives of the derivative, or no gradient of x
            if g_features is not None:
                masked = g_features if g_features2 is None else g_features + g_features2
                if ctx.relu:
                    masked = torch.ops.aten.threshold_backward(masked, features, 0)
                masked = masked.contiguous()
            if want_x:
                parts = [g_x] + [g @ w for g, w in ((masked, w_features), (g_coords, w_coords)) if g is not None]
                grad_x = sum(part for part in parts if part is not None) if any(part is not None for part in parts) else None
        grad_wf = grad_b = grad_wc = None
        if masked is not None and want_wf:
            grad_wf, grad_b = _weight_and_bias_grad(masked, x, want_b)
        elif masked is not None and want_b:
            grad_b = _sum_rows(masked)
        if g_coords is not None and want_wc:
            grad_wc, _ = _weight_and_bias_grad(g_coords.contiguous(), x, False)
        return grad_x, grad_wf, grad_b if want_b else None, grad_wc, None


class _OutputLayerFn(torch.autograd.Function):
    """relu of the block's last layer on joined = [accumulated - (features | features) | x], and joined itself: the weight
    gradient reads it, and the derivative of that gradient comes back through it"""

    @staticmethod
    def forward(ctx, accumulated, features, x, weight, bias):
        ctx.set_materialize_grads(False)
        joined = ops.gravnet_join(accumulated, features, x)
        # (a library product too: its last bits decide which activations pass their gradient on)
        out = torch.nn.functional.linear(joined, weight, bias).relu_()
        ctx.n_features = features.shape[1]
        ctx.save_for_backward(weight, out, joined if ctx.needs_input_grad[3] else None)
        return out, joined

    @staticmethod
    def backward(ctx, g, g_joined):
        weight, out, joined = ctx.saved_tensors
        f = ctx.n_features
        wanted, (want_w, want_b) = ctx.needs_input_grad[:3], ctx.needs_input_grad[3:]
        grads, masked = (None, None, None), None
        if any(wanted) and g is not None and g_joined is None and not torch.is_grad_enabled():
            *grads, masked = ops.gravnet_output_layer_grad(g, out, weight, f)
        else:  # as tensor operations: derivatives of the derivative, or no gradient of the rows
            if g is not None:
                masked = torch.ops.aten.threshold_backward(g, out, 0).contiguous()
            if any(wanted) and (g is not None or g_joined is not None):
                grad = g_joined if g is None else masked @ weight if g_joined is None else masked @ weight + g_joined
                grads = grad[:, :2 * f], -grad[:, :f] - grad[:, f:2 * f], grad[:, 2 * f:]
        grad_w = grad_b = None
        if masked is not None and want_w:
            grad_w, grad_b = _weight_and_bias_grad(masked, joined, want_b)
        elif masked is not None and want_b:
            grad_b = _sum_rows(masked)
        return (*(t if want else None for t, want in zip(grads, wanted)), grad_w, grad_b if want_b else None)


class TallLinear(nn.Linear):
    """nn.Linear whose weight gradient is formed slice-wise (see _TallLinearFn); same parameters and results
    up to the summation order of that gradient"""

    def forward(self, x):
        if x.dim() == 2 and x.is_contiguous():
            return _TallLinearFn.apply(x, self.weight, self.bias)
        return super().forward(x)


_ACTIVATIONS = {None: nn.Identity, "linear": nn.Identity, "relu": nn.ReLU, "elu": nn.ELU, "tanh": nn.Tanh,
                "sigmoid": nn.Sigmoid, "selu": nn.SELU, "gelu": nn.GELU}


_DISTANCE_SCALE = 10.0  # neighbours are weighted by exp(-10 d^2)
_REPLACEABLE = {"compute_neighbours_and_distancesq", "collect_neighbours", "create_output_features", "update_dynamic_radius"}
# what the layers in one pass stand for: with something else in its place (on the class, too) they run one by one
_OWN_LAYER = {TallLinear: TallLinear.forward}
_OWN_ACTIVATIONS = {cls: cls.forward for cls in (nn.ReLU, nn.Identity)}


class RaggedGravNet(nn.Module):
    """call(x [N, F_in], row_splits [R+1]) -> (features [N, n_filters], coordinates
    [N, n_dimensions], neighbour indices, squared distances); the last two with
    the self entry in slot 0 if return_self (then n_neighbours+1 wide)."""

    def __init__(self, in_features, n_neighbours, n_dimensions, n_filters, n_propagate, return_self=True,
                 sumwnorm=False, feature_activation="relu", coord_initialiser_noise=1e-2, n_knn_bins=None):
        super().__init__()
        assert n_neighbours > 1
        self.n_neighbours = n_neighbours
        self.n_dimensions = n_dimensions
        self.n_filters = n_filters
        self.n_propagate = n_propagate
        self.return_self = return_self
        self.sumwnorm = sumwnorm
        self.n_knn_bins = n_knn_bins
        self.input_feature_transform = TallLinear(in_features, n_propagate)
        self.feature_activation = _ACTIVATIONS[feature_activation]()
        self.input_spatial_transform = TallLinear(in_features, n_dimensions, bias=False)
        eye_init_(self.input_spatial_transform.weight, 0.0, coord_initialiser_noise)
        self.output_feature_transform = TallLinear(2 * n_propagate + in_features, n_filters)
        # bookkeeping of the reference (GravNetLayersRagged.py:3180-3193); the exact kNN does not use it
        self.register_buffer("dynamic_radius", torch.tensor(1.0))

    def update_dynamic_radius(self, dist):
        if not self.training:
            return
        with torch.no_grad():
            if _library_takes(dist, self.dynamic_radius):
                self.dynamic_radius += ops.gravnet_radius_step(dist, self.dynamic_radius)
                return
            lindist = torch.sqrt(dist)
            update = lindist.max() * 1.05
            mean_dist = lindist.mean()
            low_update = torch.clamp(update, max=2.0)
            update = torch.where(low_update > 2.0 * mean_dist, low_update, 2.0 * mean_dist) + 1e-3
            self.dynamic_radius += 0.05 * (update - self.dynamic_radius)

    def compute_neighbours_and_distancesq(self, coordinates, row_splits):
        return self._neighbours(coordinates, row_splits, 1.0)

    def _neighbours(self, coordinates, row_splits, scale):
        idx, dist = BinnedSelectKnn(self.n_neighbours + 1, coordinates, row_splits, max_radius=-1.0,
                                    tf_compatible=False, n_bins=self.n_knn_bins)
        self.update_dynamic_radius(dist.detach())  # missing neighbours have distance 0
        # the table without its self column, as tensors of their own; it lists the
        # same vertices row by row, so the kNN's processing order applies to it too
        if _library_takes(dist):
            nidx, ndist, dist = _DropSelfFn.apply(idx, dist, scale)
        else:
            nidx, ndist = idx[:, 1:].contiguous(), dist[:, 1:].contiguous()
            if scale != 1.0:
                ndist = scale * ndist
            if self.return_self:
                dist = dist.clone()  # may be written to: the search keeps its own
        ops.share_vertex_order(idx, nidx)
        ops.declare_without_first_column(nidx, idx)
        if self.return_self:
            return nidx, ndist, idx, dist
        return nidx, ndist, None, None

    def collect_neighbours(self, features, neighbour_indices, distancesq):
        return self._collect(features, neighbour_indices, _DISTANCE_SCALE * distancesq)

    def _collect(self, features, neighbour_indices, distances):
        if self.sumwnorm and _library_takes(distances, features):
            return _AccumulateSumwFn.apply(distances, features, neighbour_indices)
        acc = AccumulateKnnSumw if self.sumwnorm else AccumulateKnn
        f, _ = acc(distances, features, neighbour_indices, mean_and_max=True)
        return f

    def create_output_features(self, x, neighbour_indices, distancesq):
        features = self.feature_activation(self.input_feature_transform(x))
        prev_feat = features
        features = self.collect_neighbours(features, neighbour_indices, distancesq)
        features = features.reshape(-1, prev_feat.shape[1] * 2)
        if _library_takes(features, prev_feat, x):
            joined = _JoinFn.apply(features, prev_feat, x)
        else:
            joined = torch.cat([features - prev_feat.repeat(1, 2), x], dim=-1)
        return torch.relu(self.output_feature_transform(joined))

    def _layers_in_one_pass(self, x):
        """Whether the dense layers run as the library's passes: the block as it is here, its layers and activation
        without hooks or replacements, so that nobody waits for their calls, and tensors that the passes take."""
        if torch.compiler.is_compiling():  # (asked first: a compiler traces this, but not the looks at hooks and dictionaries)
            return False
        if type(self) is not RaggedGravNet or not self.__dict__.keys().isdisjoint(_REPLACEABLE) or not x.is_contiguous():
            return False
        first, spatial, last = self.input_feature_transform, self.input_spatial_transform, self.output_feature_transform
        if _has_any_global_hook() or any(getattr(RaggedGravNet, name) is not method for name, method in _OWN_METHODS):
            return False
        for module, known in ((first, _OWN_LAYER), (spatial, _OWN_LAYER), (last, _OWN_LAYER), (self.feature_activation, _OWN_ACTIVATIONS)):
            if (known.get(type(module)) is not type(module).forward or "forward" in module.__dict__ or module._forward_hooks or
                    module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks):
                return False
        weights = first.weight, first.bias, spatial.weight, last.weight, last.bias
        if any(w is None for w in weights) or spatial.bias is not None or not _library_takes(x, *weights):
            return False
        if not all(w.is_contiguous() for w in weights):
            return False
        f, i, o, c = first.weight.shape[0], x.shape[1], last.weight.shape[0], spatial.weight.shape[0]
        if first.weight.shape[1] != i or spatial.weight.shape[1] != i or last.weight.shape[1] != 2 * f + i:
            return False  # (the layers themselves say what is wrong)
        return not (torch.is_autocast_enabled("cuda") or x.shape[0] >= 1 << 31) and bool(
            ops.lib.hgc_gravnet_dense_covers(f, i, o, c))

    def forward(self, x, row_splits):
        assert x.dim() == 2 and row_splits.dim() == 1
        if self._layers_in_one_pass(x):
            features, coordinates, features_again, x_again = _InputLayersFn.apply(
                x, self.input_feature_transform.weight, self.input_feature_transform.bias, self.input_spatial_transform.weight,
                type(self.feature_activation) is nn.ReLU)
            # (where the distances without the self column are handed back, they are so without the factor)
            scale = _DISTANCE_SCALE if self.return_self else 1.0
            nidx, ndist, sidx, sdist = self._neighbours(coordinates, row_splits, scale)
            accumulated = self._collect(features, nidx, ndist) if self.return_self else self.collect_neighbours(features, nidx, ndist)
            last = self.output_feature_transform
            outfeats, _ = _OutputLayerFn.apply(accumulated, features_again, x_again, last.weight, last.bias)
            return (outfeats, coordinates, sidx, sdist) if self.return_self else (outfeats, coordinates, nidx, ndist)
        coordinates = self.input_spatial_transform(x)
        neighbour_indices, distancesq, sidx, sdist = self.compute_neighbours_and_distancesq(coordinates, row_splits)
        outfeats = self.create_output_features(x, neighbour_indices, distancesq)
        if self.return_self:
            neighbour_indices, distancesq = sidx, sdist
        return outfeats, coordinates, neighbour_indices, distancesq


_OWN_METHODS = [(name, getattr(RaggedGravNet, name)) for name in sorted(_REPLACEABLE)]
