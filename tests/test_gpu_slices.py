"""The lane-split pass-B kernels at the channel counts whose rows they read in
dword-aligned slices (8, 12, 20 and 24; 2, 3, 5 or 6 channels a lane), against
the CPU oracle with the bounds of the other parity tests, and from bases that
are only 4-byte aligned, against the same call on aligned copies."""
import pytest
import torch

import helpers as H
import test_gpu_parity as T

pytestmark = pytest.mark.gpu

SLICES = {}
for _C in (8, 12, 20, 24):
    for _D, _per, _mode in ((2, False, "grid"), (2, True, "grid"), (3, False, "particle"), (3, True, "grid")):
        _c = H.random_case(f"slice{_C}-{_D}d-{'per' if _per else 'clamp'}-{_mode}", 2, 257, _C, _D, 8, 0.25, _per, _mode)
        SLICES[_c.name] = _c
T.CASES.update(SLICES)


@pytest.mark.parametrize("name", sorted(SLICES))
def test_slices_match_oracle(name):
    T.test_forward(name)
    T.test_gradient_hybrid(name)
    T.test_backward(name)
    T.test_fused_passes(name)


@pytest.mark.parametrize("C", [8, 12, 20, 24])
def test_unaligned_rows(C):
    """State and upstream tensors one float past a 16-byte boundary."""
    import npa_amd.sphops as sp
    B, N, D = 1, 700, 3
    g = torch.Generator(device="cuda").manual_seed(C)
    x = torch.zeros(B, N, 4, device="cuda")
    x[..., :3] = torch.rand(B, N, 3, device="cuda", generator=g) * 1.6 - 0.8
    grid = sp.HashGrid(dim=D, boundary="clamped", mode="grid", grid_size=[8] * 3, eps=0.25, num_particles=N,
                       batch_size=B, max_particles_per_block=64)
    snap = grid.instantiate(x)
    s = torch.randn(B, N, C, device="cuda", generator=g)
    ups = torch.randn(B, N, C, device="cuda", generator=g), torch.randn(B, N, C, D, device="cuda", generator=g)
    xb, sb = sp.bin_particles(x, s, snap)

    def shifted(t):
        room = torch.empty(t.numel() + 1, device="cuda")
        room[1:] = t.reshape(-1)
        return room[1:].view(t.shape)

    def call(place):
        xr, sr = xb.detach().requires_grad_(True), place(sb).detach().requires_grad_(True)
        rho = sp.density(xr, snap)
        outs = sp.blur(xr, rho, sr, snap), sp.gradient_hybrid(xr, rho, sr, snap), sp.gradient(xr, rho, sr, snap)
        torch.autograd.backward(outs, [place(ups[0]), place(ups[1]), place(ups[1])])
        return [*outs, xr.grad, sr.grad]

    call(lambda t: t.clone())  # the grid learns the pass pair, so that both calls below take the fused kernels
    for a, b in zip(call(lambda t: t.clone()), call(shifted)):
        assert torch.equal(a, b)
