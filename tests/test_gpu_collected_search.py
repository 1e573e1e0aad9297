"""The kNN search that collects candidates and sorts them once (every coordinate binned, up to 129 neighbours), against a
brute force with the same serial float32 sums, and the search by shells on both sides of the rules."""
import numpy as np
import pytest
import torch

from hgcalml_amd import BinnedSelectKnn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def brute_force(x, splits, K, radius, direction):
    """ascending (squared distance, index), the point itself first, -1 / 0 behind the last neighbour"""
    n = len(x)
    idx = torch.full((n, K), -1, dtype=torch.int32)
    dist = torch.zeros(n, K)
    for a, b in zip(splits[:-1], splits[1:]):
        if a == b:
            continue
        y = x[a:b]
        d = torch.zeros(b - a, b - a)
        for c in range(x.shape[1]):
            step = y[:, c, None] - y[None, :, c]
            d = d + step * step
        key = (d.view(torch.int32).to(torch.int64) << 32) | torch.arange(a, b)[None, :]
        none = torch.iinfo(torch.int64).max
        key.fill_diagonal_(none)
        if radius:
            r = np.float32(radius)
            key[d > float(r * r)] = none
        if direction is not None:
            own = direction[a:b]
            key[:, (own == 1) | (own == 2)] = none
            key[(own == 0) | (own == 2), :] = none
        key = key.sort(dim=1).values[:, :K - 1]
        width = key.shape[1]
        there = key != none
        idx[a:b, 0] = torch.arange(a, b, dtype=torch.int32)
        idx[a:b, 1:1 + width] = torch.where(there, key & 0xffffffff, -1).to(torch.int32)
        dist[a:b, 1:1 + width] = torch.where(there, key >> 32, 0).to(torch.int32).view(torch.float32)
    return idx, dist


def points(kind, n, dims, gen):
    if kind == "same":  # more equal keys than the buffer holds
        return torch.full((n, dims), 0.25)
    if kind == "lattice":  # many ties at every distance
        return torch.randint(0, 5, (n, dims), generator=gen).float()
    x = torch.rand(n, dims, generator=gen)
    if kind == "clump":  # crowded bins beside empty space
        x[: n // 2] = 0.5 + 1e-4 * x[: n // 2]
        x[n - 3:] = 40 * x[n - 3:] - 20
    if kind == "line":  # one dimension without extent
        x[:, 0] = 1.0
    return x


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("kind", ["uniform", "clump", "lattice", "same", "line"])
@pytest.mark.parametrize("K,radius,directed", [(2, 0, False), (16, 0, False), (33, 0.3, False), (48, 0, True), (64, 0, False), (65, 1e-3, False),
                                               (66, 0, False), (96, 0.5, True), (129, 0, False), (130, 0, False)])
def test_matches_brute_force(dims, kind, K, radius, directed):
    gen = torch.Generator().manual_seed(100 * dims + K)
    splits = [0, 900, 900, 910, 1500]  # an empty and a tiny event among them
    x = points(kind, splits[-1], dims, gen)
    direction = torch.randint(0, 4, (len(x),), generator=gen, dtype=torch.int32) if directed else None
    got = BinnedSelectKnn(K, x.to(DEV), torch.tensor(splits, dtype=torch.int32, device=DEV), max_radius=radius or None,
                          direction=None if direction is None else direction.to(DEV))
    want = brute_force(x, splits, K, radius, direction)
    assert torch.equal(got[0].cpu(), want[0])
    assert torch.equal(got[1].cpu().view(torch.int32), want[1].view(torch.int32))


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K,radius", [(17, 0.02), (17, 0.2), (40, 0.9), (40, 5.0), (100, 5.0)])
@pytest.mark.parametrize("kind", ["uniform", "clump", "line"])
def test_radius_of_many_bins(dims, K, radius, kind):
    """from a radius inside one bin to one that reaches across the grid while the first bins hold too few points"""
    gen = torch.Generator().manual_seed(dims)
    x = points(kind, 3000, dims, gen) ** 2  # denser towards one corner
    got = BinnedSelectKnn(K, x.to(DEV), torch.tensor([0, 3000], dtype=torch.int32, device=DEV), max_radius=radius)
    want = brute_force(x, [0, 3000], K, radius, None)
    assert torch.equal(got[0].cpu(), want[0])
    assert torch.equal(got[1].cpu().view(torch.int32), want[1].view(torch.int32))


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K", [17, 65, 129])  # a list that fills its registers exactly, and one that does not
def test_first_two_points_share_the_last_distance(dims, K):
    """points 0 and 1 coincide and are the farthest ones of a query that has one neighbour too many"""
    gen = torch.Generator().manual_seed(dims)
    x = torch.rand(K + 1, dims, generator=gen) * 0.3 + 0.7
    x[:2] = 0.0
    idx, dist = BinnedSelectKnn(K, x.to(DEV), torch.tensor([0, K + 1], dtype=torch.int32, device=DEV))
    want = brute_force(x, [0, K + 1], K, 0, None)
    assert (want[0][2:, K - 1] == 0).all()
    assert torch.equal(idx.cpu(), want[0])
    assert torch.equal(dist.cpu().view(torch.int32), want[1].view(torch.int32))


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan")])
def test_unbounded_coordinates_end(dims, bad):
    """one such coordinate leaves bin widths without a meaning: the search ends and the finite points keep each other"""
    gen = torch.Generator().manual_seed(dims)
    x = torch.rand(700, dims, generator=gen)
    clean = brute_force(x[1:], [0, 699], 9, 0, None)
    x[0, dims - 1] = bad
    idx, dist = BinnedSelectKnn(9, x.to(DEV), torch.tensor([0, 700], dtype=torch.int32, device=DEV))
    assert torch.equal(idx[1:].cpu(), clean[0] + 1)
    assert torch.equal(dist[1:].cpu(), clean[1])


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("scale", [1e-23, 1e-20, 1e-18, 1e16, 1e18, 1e20])
def test_squares_at_the_ends_of_the_range(dims, scale):
    """squared distances that are denormal, zero or infinite, and bin widths whose squares are"""
    gen = torch.Generator().manual_seed(dims)
    x = torch.rand(800, dims, generator=gen) * scale
    x[400:500] = x[:100]
    idx, dist = BinnedSelectKnn(12, x.to(DEV), torch.tensor([0, 800], dtype=torch.int32, device=DEV))
    want = brute_force(x, [0, 800], 12, 0, None)
    assert torch.equal(idx.cpu(), want[0])
    assert torch.equal(dist.cpu().view(torch.int32), want[1].view(torch.int32))


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K", [2, 17, 49, 65, 129])
@pytest.mark.parametrize("kind", ["one place", "half in one place", "few sites", "two sites"])
def test_many_points_at_the_last_distance(dims, K, kind):
    """far more points at the Kn-th distance than the buffer holds, met in any order of their indices"""
    gen = torch.Generator().manual_seed(10 * dims + K)
    n = 3001
    x = torch.rand(n, dims, generator=gen)
    if kind == "one place":
        x[:] = 0.25
    elif kind == "half in one place":
        x[torch.rand(n, generator=gen) < 0.5] = 0.5
    elif kind == "few sites":
        x = torch.randint(0, 3, (n, dims), generator=gen).float()
    else:  # the last neighbours of most queries are at the other site
        x = torch.zeros(n, dims)
        x[40:] = 1.0
        x = x[torch.randperm(n, generator=gen)]
    got = BinnedSelectKnn(K, x.to(DEV), torch.tensor([0, n], dtype=torch.int32, device=DEV))
    want = brute_force(x, [0, n], K, 0, None)
    assert torch.equal(got[0].cpu(), want[0])
    assert torch.equal(got[1].cpu().view(torch.int32), want[1].view(torch.int32))


def test_points_in_one_place_cost_no_more_than_others():
    """the buffer is not cut again for every candidate at the Kn-th distance: 163 us against 39 for spread points, 57 where
    candidates beyond the last index stay out, 58 by shells"""
    n, K = 4000, 17
    splits = torch.tensor([0, n], dtype=torch.int32, device=DEV)

    def best(x):
        times = []
        for _ in range(30):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                BinnedSelectKnn(K, x, splits)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    gen = torch.Generator(device=DEV).manual_seed(1)
    spread = best(torch.rand(n, 3, device=DEV, generator=gen))
    assert best(torch.full((n, 3), 0.25, device=DEV)) < 2.5 * spread
