"""The work a user has this package do, as timed cases: neighbour search, neighbour accumulation
(forward and gradient), the GravNet layer that joins them, condensate assignment and the smaller
ops beside them, from single small events to batches of a million hits.

``listed()`` names the standing cases, ``draw(rng)`` gives another one of the same ranges,
``prepare`` makes a case's inputs on the GPU and ``run`` makes one pass through the public API.
"""
import math
import random

import torch

from hgcalml_amd import (AccumulateKnn, BinnedSelectKnn, BuildAndAssignCondensatesBinned, NeighbourCovariance, PushKnn,
                         RaggedGravNet)

DEVICE = "cuda:0"


# ------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # one small event of an inference server: the time is launches and host work
        dict(name="knn_small_event", kind="knn", points=700, events=1, dims=3, space="clusters", K=16, radius=0.0),
        # a batch as it comes from the detector: 16 uneven events, radius cut, rows with padding
        dict(name="knn_ragged_batch", kind="knn", points=1140000, events=16, dims=3, space="clusters", K=32, radius=0.1),
        # search + weighted mean and max, forward only (inference): a plain uniform event ...
        dict(name="forward_20k", kind="forward", points=20000, events=1, dims=3, space="uniform", K=16, features=32),
        # ... and a full HGCal-like event, the package's headline workload
        dict(name="forward_150k", kind="forward", points=150000, events=1, dims=4, space="clusters", K=64, features=64),
        # training step of the layer: a few small odd-sized events
        dict(name="gravnet_small", kind="gravnet", points=2477, events=3, dims=3, inputs=29, K=14, features=22, filters=48,
             sumw=False),
        # training step of the layer on one full event
        dict(name="gravnet_150k", kind="gravnet", points=150000, events=1, dims=4, inputs=64, K=64, features=64, filters=128,
             sumw=False),
        # training step of the layer on a ragged batch, mean normalised by the weights' sum
        dict(name="gravnet_ragged", kind="gravnet", points=240011, events=6, dims=3, inputs=48, K=40, features=32, filters=96,
             sumw=True),
        # accumulation over a given banded neighbour table, forward and gradient: the widest case
        dict(name="accumulate_1m", kind="accumulate", points=1000000, K=64, features=128, window=2000),
        # condensate assignment of one small event, the nearest point takes a hit, noise kept
        dict(name="condensates_small", kind="condensates", points=4999, events=1, dims=3, max_beta=False, keep_noise=True),
        # condensate assignment of a batch of uneven events
        dict(name="condensates_500k", kind="condensates", points=500000, events=8, dims=4, max_beta=True, keep_noise=False),
        # hits push weighted features to the neighbours a search has found, forward and gradient
        dict(name="push_60k", kind="push", points=60000, events=2, dims=3, space="clusters", K=24, features=48),
        # shape of the neighbourhood, an input feature of later layers
        dict(name="covariance_40k", kind="covariance", points=40000, events=1, dims=4, space="clusters", K=32, features=8),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["knn", "knn", "forward", "forward", "gravnet", "gravnet", "gravnet", "accumulate", "condensates",
                       "condensates", "push", "covariance"])
    dims = rng.choice([2, 3, 3, 3, 4, 4, 4, 5, 6])
    space = rng.choice(["clusters", "clusters", "clusters", "uniform", "normal"])
    K = _log_int(rng, 8, 96)
    features = rng.randint(8, 128)
    case = dict(kind=kind)
    if kind == "knn":
        radius = rng.choice([0.0, 0.0, 0.1, 0.3])
        case.update(points=_log_int(rng, 500, 1140000 if K <= 40 and dims <= 4 else 300000), dims=dims, space=space, K=K, radius=radius)
    elif kind == "forward":
        case.update(points=_log_int(rng, 500, 300000), dims=dims, space=space, K=K, features=features)
    elif kind == "gravnet":
        dims = min(dims, 4)
        case.update(points=_log_int(rng, 700, 240000), dims=dims, inputs=rng.randint(16, 96), K=min(K, 72), features=features,
                    filters=rng.randint(32, 160), sumw=rng.random() < 0.25)
    elif kind == "accumulate":
        K = min(K, 64)
        case.update(points=_log_int(rng, 20000, 1000000), K=K, features=features, window=rng.choice([300, 2000]))
    elif kind == "condensates":
        case.update(points=_log_int(rng, 1000, 500000), dims=min(dims, 4), max_beta=rng.random() < 0.5,
                    keep_noise=rng.random() < 0.5)
    elif kind == "push":
        case.update(points=_log_int(rng, 2000, 200000), dims=min(dims, 4), space=space, K=min(K, 64), features=min(features, 96))
    else:
        case.update(points=_log_int(rng, 2000, 150000), dims=max(2, min(dims, 4)), space=space, K=min(K, 64),
                    features=rng.randint(4, 16))
    if kind != "accumulate":
        most = max(1, min(16, case["points"] // 300))
        case["events"] = rng.choice([1, rng.randint(1, most), most])
    return case


# ------------------------------------------------------------------------------------------ inputs

def event_sizes(points, events):
    """uneven event sizes, the largest up to six times the smallest; the same for every seed"""
    rng = random.Random(events)
    share = [rng.uniform(20, 120) for _ in range(events)]
    sizes = [int(points * s / sum(share)) for s in share]
    sizes[0] += points - sum(sizes)
    return sizes


def row_splits_of(sizes):
    splits = [0]
    for s in sizes:
        splits.append(splits[-1] + s)
    return torch.tensor(splits, dtype=torch.int32, device=DEVICE)


def clusters(n, dims, gen):
    """showers and noise of one event: 60 % of the hits in Gaussian clusters of log-normal size, the others
    uniform in [-1, 1]^dims, shuffled; also the distance to the own cluster's centre in sigmas"""
    count = min(300, max(4, n // 100))
    weight = torch.exp(5 + torch.randn(count, device=DEVICE, generator=gen))
    centre = torch.rand(count, dims, device=DEVICE, generator=gen) * 2 - 1
    sigma = 0.02 + 0.08 * torch.rand(count, device=DEVICE, generator=gen)
    own = torch.multinomial(weight, n, replacement=True, generator=gen)
    off = torch.randn(n, dims, device=DEVICE, generator=gen)
    noise = torch.rand(n, dims, device=DEVICE, generator=gen) * 2 - 1
    is_noise = torch.rand(n, device=DEVICE, generator=gen) < 0.4
    hits = torch.where(is_noise[:, None], noise, centre[own] + off * sigma[own, None])
    rel = torch.where(is_noise, torch.full_like(sigma[own], math.inf), off.norm(dim=1))
    return hits, rel


def hits_of(sizes, dims, space, gen):
    if space == "uniform":
        return torch.rand(sum(sizes), dims, device=DEVICE, generator=gen)
    if space == "normal":
        return torch.randn(sum(sizes), dims, device=DEVICE, generator=gen)
    return torch.cat([clusters(s, dims, gen)[0] for s in sizes])


def banded_table(n, K, window, gen):
    """slot 0 = the point itself, K - 1 different others from its window in random order"""
    window = min(window, (n - 1) // 3)
    stratum = 2 * window // (K - 1)
    table = torch.empty(n, K, dtype=torch.int32, device=DEVICE)
    for s in range(0, n, 1 << 17):
        own = torch.arange(s, min(n, s + (1 << 17)), device=DEVICE)[:, None]
        off = torch.arange(K - 1, device=DEVICE) * stratum + 1 + \
            torch.randint(0, stratum, (len(own), K - 1), device=DEVICE, generator=gen)
        off = off.gather(1, torch.rand(len(own), K - 1, device=DEVICE, generator=gen).argsort(dim=1))
        off = torch.where(off > window, window - off, off)
        other = own + off
        other = torch.where(other < 0, own + window - off, other)      # mirrored beyond the window: still different
        other = torch.where(other >= n, own - window - off, other)
        table[s:s + len(own), :1] = own.to(torch.int32)
        table[s:s + len(own), 1:] = other.to(torch.int32)
    return table


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    kind, n = case["kind"], case["points"]

    def normal(*shape):
        return torch.randn(*shape, device=DEVICE, generator=gen)

    if kind == "accumulate":
        K, f = case["K"], case["features"]
        dist = torch.rand(n, K, device=DEVICE, generator=gen) * 0.5
        dist[:, 0] = 0
        return dict(case=case, table=banded_table(n, K, case["window"], gen), dist=dist, features=normal(n, f), grad=normal(n, 2 * f))
    sizes = event_sizes(n, case["events"])
    state = dict(case=case, row_splits=row_splits_of(sizes))
    if kind == "gravnet":
        # a hit's position and its other properties
        hits = torch.cat([hits_of(sizes, case["dims"], "clusters", gen), normal(n, case["inputs"] - case["dims"])], dim=1)
        layer = RaggedGravNet(case["inputs"], case["K"], case["dims"], case["filters"], case["features"],
                              sumwnorm=case["sumw"]).to(DEVICE)
        with torch.no_grad():  # fresh weights from the seed, of the size the layer's own initialisation has
            for name, weight in sorted(layer.named_parameters()):
                weight.copy_(normal(*weight.shape) * (0.01 if "spatial" in name else weight.shape[-1] ** -0.5))
                if "spatial" in name:
                    weight += torch.eye(*weight.shape, device=DEVICE)
        state.update(hits=hits.requires_grad_(True), layer=layer, grad=normal(n, case["filters"]),
                     dist_grad=normal(n, case["K"] + 1))
        return state
    if kind == "condensates":
        parts = [clusters(s, case["dims"], gen) for s in sizes]
        rel = torch.cat([p[1] for p in parts])
        # beta of the network: Beta(1/2, 2), raised in the cores of the clusters
        u = torch.rand(2, n, device=DEVICE, generator=gen).clamp_min(1e-7)
        half, two = normal(n) ** 2 / 2, -torch.log(u[0]) - torch.log(u[1])
        beta = half / (half + two)
        beta = torch.where(rel < 1, (beta + 0.5).clamp_max(0.999), beta)
        state.update(hits=torch.cat([p[0] for p in parts]), beta=beta[:, None].contiguous(),
                     radius=torch.full((n, 1), 0.5, device=DEVICE))
        return state
    state["hits"] = hits_of(sizes, case["dims"], case["space"], gen)
    if kind == "knn":
        return state
    state["features"] = normal(n, case["features"])
    if kind == "push":
        state["features"].requires_grad_(True)
        state["weights"] = torch.rand(n, case["K"], device=DEVICE, generator=gen).requires_grad_(True)
        state["grad"] = normal(n, case["features"])
    return state


# ------------------------------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "accumulate":
        dist, features = state["dist"].detach().requires_grad_(True), state["features"].detach().requires_grad_(True)
        table = state["table"].clone()  # every training step comes with a table of its own
        out, arg = AccumulateKnn(dist, features, table)
        return (out, arg) + torch.autograd.grad(out, [dist, features], state["grad"])
    if kind == "gravnet":
        layer, hits = state["layer"], state["hits"]
        out, coords, idx, dist = layer(hits, state["row_splits"])
        wanted = [hits] + list(layer.parameters())
        return (out, coords, idx, dist) + torch.autograd.grad([out, dist], wanted, [state["grad"], state["dist_grad"]])
    if kind == "condensates":
        assignment, asso, alpha, is_cond, count = BuildAndAssignCondensatesBinned(
            state["hits"], state["beta"], state["radius"], state["row_splits"], 0.1,
            assign_by_max_beta=case["max_beta"], keep_noise=case["keep_noise"])
        # the list of condensation points in a buffer that fits every event
        return assignment, asso, torch.nn.functional.pad(alpha, (0, case["points"] - len(alpha)), value=-1), is_cond, count
    if kind == "knn":
        return BinnedSelectKnn(case["K"], state["hits"], state["row_splits"], max_radius=case["radius"] or None)
    idx, dist = BinnedSelectKnn(case["K"], state["hits"], state["row_splits"])
    if kind == "forward":
        out, arg = AccumulateKnn(10.0 * dist, state["features"], idx)
        return idx, dist, out, arg
    if kind == "push":
        out = PushKnn(state["weights"], state["features"], idx)
        return (idx, out) + torch.autograd.grad(out, [state["weights"], state["features"]], state["grad"])
    cov, mean = NeighbourCovariance(state["hits"], 10.0 * dist, state["features"], idx)
    return idx, dist, cov, mean


# ------------------------------------------------------------------------------------------ what a pass cannot do without

def work(case):
    """bytes: every input once and every output once; flops: the sums over the neighbours that the results are made of"""
    kind, n = case["kind"], case["points"]
    K, f, c = case.get("K", 0), case.get("features", 0), case.get("dims", 0)
    search_bytes, search_flops = 4 * n * (c + 2 * K), 3 * n * K * c
    if kind == "knn":
        return dict(bytes=search_bytes, flops=search_flops)
    if kind == "forward":  # features in; mean, max and arg-max out
        return dict(bytes=search_bytes + 4 * n * 4 * f, flops=search_flops + 4 * n * K * f)
    if kind == "accumulate":  # distances, table, features, gradient in; outputs and both gradients out
        return dict(bytes=4 * n * (2 * K + f + 2 * f + 3 * f + K + f), flops=n * K * (4 + 4) * f)
    if kind == "gravnet":
        i, o, k = case["inputs"], case["filters"], case["K"] + 1
        dense = i * c + i * f + (2 * f + i) * o
        return dict(bytes=4 * n * (2 * i + o + o + c + 3 * k), flops=n * (6 * dense + 6 * k * c + 8 * k * f))
    if kind == "condensates":
        return dict(bytes=4 * n * (c + 2 + 2) + n, flops=3 * n * c)
    if kind == "push":
        return dict(bytes=search_bytes - 4 * n * K + 4 * n * (2 * K + 4 * f), flops=search_flops + 6 * n * K * f)
    return dict(bytes=search_bytes + 4 * n * (f + f * c * c + f * c), flops=search_flops + n * K * f * (2 * c + 3 * c * c))


def tolerance(case):
    """What another correct implementation in 32 bits may differ by: about four times what the same path differs by
    with its sums in 64 bits."""
    kind = case["kind"]
    if kind in ("knn", "condensates"):
        return "exact"
    if kind == "gravnet":
        # Coordinates in 64 bits, rounded, move one index in 10,000 (neighbours at nearly equal distances); with them,
        # and with activations and maxima that are decided by the last bits, single rows change as a whole: gradients
        # 3e-3. Where no such decision falls differently 1e-6.
        return dict(rel=1.2e-2, max=0.99, differ=5e-4)
    if kind == "covariance":  # products of differences of coordinates: 1.3e-6
        return dict(rel=6e-6, max=6e-5)
    return dict(rel=6e-7, max=2e-5)  # sums over the neighbours and the inverse neighbours: 1.5e-7
