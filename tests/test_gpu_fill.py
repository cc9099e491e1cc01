"""The neighbour list's periodic short cut (candidates that cannot wrap) and the
grouped neighbour count against the oracle's pair test, which wraps every pair:
grids of three to many cells an axis, positions on the box's faces and outside
it, few and many particles a cell.  Whole numbers: exact."""
import numpy as np
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu

CASES = [(3, 5, 1500, 1.0, "grid"), (3, 8, 6001, 1.0, "particle"), (3, 4, 300, 1.0, "grid"), (3, 3, 90, 1.0, "grid"),
         (2, 8, 900, 1.0, "particle"), (2, 40, 20011, 1.0, "grid"), (3, 6, 1200, 2.6, "grid"), (2, 9, 70, 9.5, "grid")]
# about one and about two particles a cell: many alone in theirs, on both sides
# of the rule that adds their candidates up first
CASES += [(3, 8, 500, 1.0, "grid"), (3, 8, 1100, 1.0, "particle"), (2, 32, 1000, 1.0, "grid"), (2, 32, 2100, 1.0, "grid")]


@pytest.mark.parametrize("dim,gs,N,spread,mode", CASES)
@pytest.mark.parametrize("periodic", [True, False])
def test_list_and_count(dim, gs, N, spread, mode, periodic):
    import npa_amd.sphops as sp
    from npa_amd.sphops.sph import _plan
    half = 0.5
    c = H.random_case("f", 2, N, 4, dim, gs, 2 * half / gs, periodic, mode, sigma=half * spread, seed=gs + N)
    c.x[0, : N // 4, :dim] = np.round(c.x[0, : N // 4, :dim] * 2) / 2  # the box's centre, faces and corners
    grid = sp.HashGrid(dim=dim, boundary=c.boundary, mode=mode, grid_size=[gs] * dim, eps=c.eps, num_particles=N,
                       batch_size=2, max_particles_per_block=c.maxp)
    x, s = torch.from_numpy(c.x).cuda(), torch.from_numpy(c.s).cuda()
    snap = grid.instantiate(x)
    xb, _ = sp.bin_particles(x, s, snap)
    ctx = H.oracle_context(c, xb.cpu().numpy(), snap.bin_offsets.cpu().numpy())
    want = np.bincount(ctx.p.i, minlength=2 * N)
    for _ in range(2):  # the first list's buffer is an estimate; the second holds every row
        snap.plan = None
        nbr = _plan(snap, xb)
        got = sp.count(xb, snap).cpu().numpy().ravel()
        assert np.array_equal(got, want)
        torch.cuda.synchronize()
        start, count, index = (t.cpu().numpy() for t in nbr[:3])
        stored = count >= 0
        assert np.array_equal(count[stored], want[stored])
        rows = np.split(ctx.p.j, ctx.p.starts[1:])
        for i in np.flatnonzero(stored):
            assert np.array_equal(np.sort(index[start[i]: start[i] + count[i]]), np.sort(rows[i])), i
        grid.instantiate(x)
