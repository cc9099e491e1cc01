"""npa_amd.perceive's one-call path (Perceive) against the operators called one
by one, over dimensions, boundaries, modes, channel counts, the stop-gradient
and normalisation flags, the inputs that require a gradient and the outputs
that receive one.  The forward runs the same kernels: bit for bit.  A gradient
is a sum of at most three terms, which the two paths add in another order:
within 2^-22 of the sum of their magnitudes, taken as eight times the larger of
the value and the tensor's root mean square (their scale here)."""
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu

GRIDS = [(2, False, "grid", 16), (2, True, "grid", 12), (3, False, "particle", 5), (3, True, "grid", 20),
         (3, False, "grid", 32)]


def _grid(dim, per, mode, C, B=2, N=301):
    import npa_amd.sphops as sp
    c = H.random_case("p", B, N, C, dim, 8, 0.25, per, mode, seed=dim + C)
    grid = sp.HashGrid(dim=dim, boundary="periodic" if per else "clamped", mode=mode, grid_size=list(c.grid_size),
                       eps=c.eps, num_particles=N, batch_size=B, max_particles_per_block=c.maxp)
    return grid, torch.from_numpy(c.x).cuda(), torch.from_numpy(c.s).cuda()


def _both(monkeypatch, call):
    from npa_amd import perceive as PF
    got = call()
    monkeypatch.setattr(PF, "_native_ok", lambda *a: False)
    call()  # the grid learns the pass pairs: the fused kernels from here on
    ref = call()
    monkeypatch.undo()
    return got, ref


def _close(a, b):
    if b is None:
        assert a is None
        return
    rms = b.double().pow(2).mean().sqrt()
    assert torch.all((a.double() - b.double()).abs() <= 2.0 ** -22 * 8 * (b.double().abs() + rms))


@pytest.mark.parametrize("dim,per,mode,C", GRIDS)
@pytest.mark.parametrize("stop_pos,stop_state", [(True, False), (False, False), (False, True), (True, True)])
def test_perceive_matches_operators(monkeypatch, dim, per, mode, C, stop_pos, stop_state):
    from npa_amd import perceive as PF
    grid, x, s = _grid(dim, per, mode, C)
    g = torch.Generator(device="cuda").manual_seed(1)
    W = PF.feature_width(C, dim, PF.STATE_GRAD | PF.DENSITY_GRAD)
    ups = [torch.randn(2, 301, k, device="cuda", generator=g) for k in (W, x.shape[2], C)]
    for which in ((0, 1, 2), (0,), (1, 2), (2,)):
        for need in ((True, True), (False, True), (True, False)):
            def call():
                xr, sr = (t.clone().requires_grad_(r) for t, r in zip((x, s), need))
                z, xb, sb, snap = PF.perceive(xr, sr, grid, 0.1, log_norm_grad=C != 12, log_norm_density_grad=C != 5,
                                              stopgrad_pos=stop_pos, stopgrad_state=stop_state)
                outs = (z, xb, sb)
                live = [i for i in which if outs[i].requires_grad]
                if live:
                    torch.autograd.backward([outs[i] for i in live], [ups[i] for i in live])
                return [t.detach() for t in outs], [t.requires_grad for t in outs], snap, (xr.grad, sr.grad)
            (fo, fr, fs, fg), (ro, rr, rs, rg) = _both(monkeypatch, call)
            assert fr == rr
            assert all(torch.equal(a, b) for a, b in zip(fo, ro))
            for k in ("permutation", "inverse", "bin_offsets", "block_info", "total_blocks"):
                if k != "block_info" or mode == "grid":
                    assert torch.equal(getattr(fs, k), getattr(rs, k)), k
            for a, b in zip(fg, rg):
                _close(a, b)


def test_snapshot_and_list_serve_later_operators():
    """The returned snapshot's list is reused by the operators; a permutation
    modified in place makes the backward gather by it, as the operators do."""
    import npa_amd.sphops as sp
    from npa_amd import perceive as PF
    grid, x, s = _grid(3, False, "grid", 16)
    with torch.no_grad():
        z, xb, sb, snap = PF.perceive(x, s, grid, 0.1)
        plan = snap.plan[4]
        rho = sp.density(xb, snap)
        assert snap.plan[4] is plan and torch.equal(sb, z[..., :16])
        assert torch.equal(sp.blur(xb, rho, sb, snap), sp.blur(xb, rho, sb, grid.instantiate(x)))
    grads = []
    for touch in (False, True):
        sr = s.clone().requires_grad_(True)
        z, _, _, snap = PF.perceive(x, sr, grid, 0.1)
        if touch:
            snap.permutation.add_(0)
        z.square().sum().backward()
        grads.append(sr.grad)
    assert torch.equal(*grads)


def test_overflowing_list_walks_the_stencil():
    """A list without room for its rows: the same features and gradients to
    rounding (sums of at most 70 terms, in another order)."""
    from npa_amd import perceive as PF
    grid, x, s = _grid(2, False, "grid", 16)
    outs = []
    for cap in (0, 7):
        grid.set_capture_capacity(cap)
        sr = s.clone().requires_grad_(True)
        z, _, _, _ = PF.perceive(x, sr, grid, 0.1)
        z.sum().backward()
        outs.append((z.detach(), sr.grad))
        assert grid.list_overflow() == (cap == 7)
    for a, b in zip(*outs):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4 * b.abs().max().item())


def test_other_grids_keep_their_own_instantiate():
    """A grid that instantiates in its own way, as a subclass, on the instance
    or without a native grid of its own, is asked for its snapshot."""
    import npa_amd.sphops as sp
    from npa_amd import perceive as PF
    grid, x, s = _grid(2, False, "grid", 16)
    with torch.no_grad():
        ref = PF.perceive(x, s, grid, 0.1)
        asked = []

        class Own(sp.HashGrid):
            def instantiate(self, x):
                asked.append("subclass")
                return super().instantiate(x)

        class Wrapped:
            dim, eps = grid.dim, grid.eps

            def instantiate(self, x):
                asked.append("wrapped")
                return grid.instantiate(x)

        own = Own(dim=2, boundary="clamped", mode="grid", grid_size=grid.grid_size, eps=grid.eps, num_particles=301,
                  batch_size=2, max_particles_per_block=grid.max_particles_per_block)
        patched = _grid(2, False, "grid", 16)[0]
        patched.instantiate = lambda x: asked.append("instance") or grid.instantiate(x)
        for other in (own, Wrapped(), patched):
            got = PF.perceive(x, s, other, 0.1)
            assert all(torch.equal(a, b) for a, b in zip(got[1:3], ref[1:3]))
            assert torch.allclose(got[0], ref[0], rtol=1e-4, atol=1e-5)
    assert asked == ["subclass", "wrapped", "instance"]


def test_records_only_for_a_backward(monkeypatch):
    """The (x, weight) records that only the backward reads are kept where one
    can follow: not under no_grad, whatever the inputs require."""
    from npa_amd import perceive as PF
    grid, x, s = _grid(2, False, "grid", 16)
    kept, call = [], PF._lib.sphops_perceive_forward

    def spy(h, a, stream):
        kept.append((bool(a._obj.packed_mass), bool(a._obj.packed_volume)))
        return call(h, a, stream)

    monkeypatch.setattr(PF._lib, "sphops_perceive_forward", spy)
    xr, sr = x.clone().requires_grad_(True), s.clone().requires_grad_(True)
    outs = []
    with torch.no_grad():
        outs.append(PF.perceive(xr, sr, grid, 0.1, stopgrad_pos=False))
    outs.append(PF.perceive(xr, sr, grid, 0.1, stopgrad_pos=False))
    assert kept == [(False, False), (True, True)]
    assert not outs[0][0].requires_grad and all(torch.equal(a, b) for a, b in zip(outs[0][:3], outs[1][:3]))


@pytest.mark.parametrize("dim,per,mode,C", GRIDS[:3])
def test_steps_in_flight_keep_their_own_lists(dim, per, mode, C):
    """Several forwards on one grid before the first backward, the backwards
    in reverse order: each reads its own list and records (another cloud's
    give other values altogether).  Which rows the first lists' estimated
    buffers leave to the stencil, and so the order of their sums, may differ:
    bound as for an overflowing list."""
    from npa_amd import perceive as PF
    grid, x, s = _grid(dim, per, mode, C)
    g = torch.Generator(device="cuda").manual_seed(3)
    clouds = [(x, s), (x.roll(7, 1) * 0.9, s.flip(1)), (x * 0.8, s * 2)]

    def forward(cloud):
        xr, sr = (t.clone().requires_grad_(True) for t in cloud)
        return xr, sr, PF.perceive(xr, sr, grid, 0.1, stopgrad_pos=False)[0]

    W = PF.feature_width(C, dim, PF.STATE_GRAD | PF.DENSITY_GRAD)
    up = torch.randn(2, 301, W, device="cuda", generator=g)
    alone = []
    for cloud in clouds:
        xr, sr, z = forward(cloud)
        z.backward(up)
        alone.append((xr.grad, sr.grad))
    steps = [forward(cloud) for cloud in clouds]
    for (xr, sr, z), ref in zip(steps[::-1], alone[::-1]):
        z.backward(up)
        for a, b in zip((xr.grad, sr.grad), ref):
            assert torch.allclose(a, b, rtol=1e-4, atol=1e-4 * b.abs().max().item())
