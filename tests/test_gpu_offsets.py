"""instantiate on both sides of the cell count that divides the two ways of
making bin_offsets (a search per cell; chunks of cells under the permutation),
few and many particles for the cells, in one cell and spread, against the
oracle: whole numbers, exact."""
import numpy as np
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu

GRIDS = [(3, 161, "grid"), (3, 162, "grid"), (2, 2047, "grid"), (2, 2048, "grid"), (3, 128, "particle"),
         (3, 256, "particle")]


@pytest.mark.parametrize("dim,gs,mode", GRIDS)
@pytest.mark.parametrize("N,sigma", [(3, 1.0), (5000, 0.01), (90001, 1.0)])
def test_offsets_match_oracle(dim, gs, mode, N, sigma):
    import npa_amd.sphops as sp
    c = H.random_case("o", 1, N, 1, dim, gs, 2.0 / gs, False, mode, sigma=sigma, seed=gs)
    grid = sp.HashGrid(dim=dim, boundary=c.boundary, mode=mode, grid_size=[gs] * dim, eps=c.eps, num_particles=N,
                       batch_size=1, max_particles_per_block=c.maxp)
    ref = H.oracle_binning(c)
    snap = grid.instantiate(torch.from_numpy(c.x).cuda())
    assert np.array_equal(snap.permutation.cpu().numpy(), ref["permutation"])
    assert np.array_equal(snap.bin_offsets.cpu().numpy(), ref["bin_offsets"])
    if mode == "grid":
        total = int(snap.total_blocks)
        assert total == ref["total_blocks"]
        assert np.array_equal(snap.block_info[:total].cpu().numpy(), ref["block_info"][:total])
