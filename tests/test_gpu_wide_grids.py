"""The search on grids with many bins along one dimension."""
import pytest
import torch

from test_gpu_collected_search import brute_force

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


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
