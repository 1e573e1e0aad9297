"""The search on grids with so many bins along one dimension that a place in the grid, in bins, is no longer good to a
thousandth: the bounds that leave bins out have to allow for that."""
import pytest
import torch

from test_data_errors import _status_after
from test_gpu_collected_search import brute_force

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n_bins", [(3, 1 << 13), (3, 1 << 16), (3, 1 << 18), (2, 3, 1 << 18), (2, 2, 2, 1 << 17), (2, 2, 2, 2, 1 << 16),
                                    (5, 1 << 20), (2, 1 << 22)])
@pytest.mark.parametrize("K", [2, 9, 140])  # collected (up to four dimensions), and by shells
@pytest.mark.parametrize("width", [0.001237, 0.73])
def test_neighbours_across_bin_edges(n_bins, K, width):
    from hgcalml_amd._lib import check, lib, p, stream
    gen = torch.Generator().manual_seed(len(n_bins) * 1000 + K)
    dims, n, far = len(n_bins), 3000, 1000  # the last bins of the long dimension, where the rounding is largest
    bins = torch.tensor(n_bins, dtype=torch.float64)
    place = torch.rand(n, dims, generator=gen, dtype=torch.float64) * bins
    place[:, -1] = n_bins[-1] - far * torch.rand(n, generator=gen, dtype=torch.float64) - 1
    x = (place * width).float()
    on_gpu, gbins = x.to(DEV), torch.tensor(n_bins, dtype=torch.int32, device=DEV)
    gwidth, shift = torch.tensor([width], device=DEV), torch.zeros(dims, device=DEV)
    total = int(gbins.long().prod())
    rows, flat, count = torch.ops.hgcalml.bin_by_coordinates(on_gpu, torch.tensor([0, n], dtype=torch.int32, device=DEV), gwidth,
                                                             gbins, total, True)
    order = torch.argsort(flat.long() * n + torch.arange(n, device=DEV))
    table = torch.zeros(total + 1, dtype=torch.int32, device=DEV)
    table[1:] = torch.cumsum(count, 0, dtype=torch.int32)
    idx = torch.empty((n, K), dtype=torch.int32, device=DEV)
    dist = torch.empty((n, K), dtype=torch.float32, device=DEV)
    a = [on_gpu[order].contiguous(), flat[order].contiguous(), rows[order].contiguous()]
    sorting = order.to(torch.int32)
    assert 0 == _status_after(lambda: check(lib.hgc_binned_select_knn_fused(
        p(a[0]), p(a[1]), None, p(a[2]), p(table), p(gbins), p(gwidth), p(sorting), p(shift), -1.0, p(idx), p(dist), n, K, dims,
        dims, len(table), 0, 0, stream())))
    want = brute_force(x, [0, n], K, 0.0, None)
    assert torch.equal(dist.cpu().view(torch.int32), want[1].view(torch.int32))
    assert torch.equal(idx.cpu(), want[0])


@pytest.mark.parametrize("n_bins", [1100, 8000, 9000, 12000])
@pytest.mark.parametrize("K,radius", [(9, 0.0), (9, 0.01), (140, 0.0)])
def test_a_callers_grid_of_many_bins_in_two_dimensions(n_bins, K, radius):
    """the rows of bins are fewer than 2^22, which is what the pipeline accepts"""
    from hgcalml_amd import BinnedSelectKnn
    from hgcalml_amd import globals as gl
    gen = torch.Generator().manual_seed(n_bins)
    x = torch.rand(1500, 2, generator=gen) * torch.tensor([1.0, 0.02])
    gl.knn_callers_grid = True
    try:
        idx, dist = BinnedSelectKnn(K, x.to(DEV), torch.tensor([0, 1500], dtype=torch.int32, device=DEV), n_bins=n_bins,
                                    max_radius=radius or None)
    finally:
        gl.knn_callers_grid = False
    want = brute_force(x, [0, 1500], K, radius, None)
    assert torch.equal(idx.cpu(), want[0])
    assert torch.equal(dist.cpu().view(torch.int32), want[1].view(torch.int32))
