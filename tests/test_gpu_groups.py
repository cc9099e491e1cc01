"""The lane groups of the list kernels at every width that the number of waves
can choose (base, twice, four times; kernels of more than 32 channels join
waves of the wider ones), each operator over the list against the same
operator on the stencil, which knows no groups.

Both are 32-bit sums of one particle's at most n pair terms in other orders:
within 2 (n + 8) 2^-24 of the sum of the terms' magnitudes, for the blur its
value for |s|; for the others, whose terms cancel, that sum is taken as n^(1/2)
times the value and the tensor's root mean square."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _cloud(n, spread, dim=3):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.zeros(1, n, 2 if dim == 2 else 4, device="cuda")
    if spread == "even":
        x[..., :dim] = torch.rand(1, n, dim, device="cuda", generator=g) - 0.5
        h = (24 / (math.pi * n)) ** 0.5 if dim == 2 else (24 / (4.19 * n)) ** (1 / 3)
    else:
        x[..., :dim] = torch.randn(1, n, dim, device="cuda", generator=g) * 0.25
        h = 0.7 * (24 / (4.19 * n)) ** (1 / 3)
    return x, h, int(2 * math.ceil(1.0 / h)) + 2, g


@pytest.mark.parametrize("spread", ["even", "uneven"])
@pytest.mark.parametrize("n", [700, 5003, 9001, 14007, 40009, 70001, 120011, 140009])
def test_groups_match_stencil(n, spread):
    import npa_amd.sphops as sp
    from npa_amd.sphops.sph import _plan
    x, h, G, g = _cloud(n, spread)
    grid = sp.HashGrid(dim=3, boundary="clamped", mode="grid", grid_size=[G] * 3, eps=h, num_particles=n, batch_size=1,
                       max_particles_per_block=64)
    native, mass = grid.hashgrid, torch.rand(1, n, device="cuda", generator=g) + 0.5
    for _ in range(2):  # the first list's buffer is an estimate; the second holds every row
        snap = grid.instantiate(x)
        xb, _ = sp.bin_particles(x, x[..., :1].contiguous(), snap)
        nbr = _plan(snap, xb)
        torch.cuda.synchronize()
    assert not grid.list_overflow()
    top = int(nbr[1].max())

    def close(got, ref, mag):
        assert torch.all((got.double() - ref.double()).abs() <= 2 * (top + 8) * 2.0 ** -24 * mag)

    def scale(ref):
        return top ** 0.5 * (ref.double().abs() + ref.double().pow(2).mean().sqrt())

    tail = (snap.bin_offsets, snap.block_info)
    rho, ref = sp.density(xb, snap, mass), torch.empty(1, n, device="cuda")
    native.density_forward(xb, mass, ref, *tail)
    close(rho, ref, ref)
    for C in (12, 20, 16, 33, 48):
        s = torch.randn(1, n, C, device="cuda", generator=g)
        up, up_g = torch.randn(1, n, C, device="cuda", generator=g), torch.randn(1, n, C, 3, device="cuda", generator=g)
        ref, mag = torch.empty_like(s), torch.empty_like(s)
        native.blur_forward(xb, rho, mass, s, ref, *tail)
        native.blur_forward(xb, rho, mass, s.abs(), mag, *tail)
        xr, sr, rr = (t.detach().clone().requires_grad_(True) for t in (xb, s, rho))
        snap.plan = (xr.detach(), xr.data_ptr(), xr._version, tuple(xr.shape), nbr)
        out = sp.sph.Blur.apply(xr, sr, rr, mass, snap)
        close(out, ref, mag)
        out.backward(up)
        refs = torch.empty_like(xb), torch.empty_like(s), torch.empty_like(rho)
        native.blur_backward(xb, rho, mass, s, up, *refs, *tail)
        for t, b in zip((xr, sr, rr), refs):
            close(t.grad, b, scale(b))
            t.grad = None
        out, ref = sp.gradient(xr, rr, sr, snap, mass), torch.empty_like(up_g)
        native.gradient_forward(xb, rho, mass, s, ref, *tail)
        close(out, ref, scale(ref))
        out.backward(up_g)
        native.gradient_backward(xb, rho, mass, s, up_g, *refs, *tail)
        for t, b in zip((xr, sr, rr), refs):
            close(t.grad, b, scale(b))
