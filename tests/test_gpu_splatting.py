"""Splatting kernels (npa_amd.splatting) against the oracle restatement of
utils/splatting.py (oracle/splatting.py, float64 on the CPU): images and the
gradients with respect to positions and colours, for single images,
batches and ragged sections (with an empty one), normalised or not, y_up,
particles partly outside the image; and run-to-run determinism."""
import math

import numpy as np
import pytest
import torch

from oracle import splatting as S
from test_oracle_splatting import particles

pytestmark = pytest.mark.gpu

CASES = [
    dict(img_size=64, sigma=1.0, pixel_size=2.0 / 32, normalize_color=True, y_up=False),
    dict(img_size=256, sigma=2.0, normalize_color=True, y_up=True),  # the reference's defaults, y flipped: r = 20
    dict(img_size=50, sigma=1.5, normalize_color=False, y_up=False, lo=-1.5, hi=2.0),
    dict(img_size=17, sigma=1.0, pixel_size=2.0 / 8, normalize_color=True, y_up=True),  # tiles cut by the edge
    dict(img_size=32, sigma=0.1, normalize_color=False, y_up=True),  # the smallest patch, r = 1
    dict(img_size=96, sigma=12.0, normalize_color=False, y_up=False),  # r = 60: patches wider than tiles
    dict(img_size=64, sigma=3.0, pixel_size=2.0 / 64, normalize_color=True, y_up=False, lo=-3.0, hi=1.0),
]
PARTICLES = {5: 200}  # fewer particles where the patch is large (the float64 oracle is dense)
# sigma = 0.1 px: the exponent -|offset - frac|^2 / (2 sigma^2) reaches -50 within a
# pixel, so fp32 rounding of the position (about 2e-6 px at 30 px) moves a weight by
# up to 1e-4 of itself, in the reference's fp32 arithmetic as much as here
IMAGE_ATOL = {4: 2e-5}


def _radius(kw):
    span = kw.get("hi", 1.0) - kw.get("lo", -1.0)
    s = kw["sigma"] * kw["img_size"] * kw.get("pixel_size", 2.0 / 128.0) / span if kw["normalize_color"] else \
        kw["sigma"]
    return max(1, math.ceil(5 * s))


def _close(name, got, ref, rtol=2e-5, atol=1e-6):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    scale = float(np.abs(ref).max()) if ref.size else 0.0
    err = np.abs(got - ref)
    bad = err > rtol * np.abs(ref) + atol * (scale + 1e-30)
    assert not bad.any(), f"{name}: {bad.sum()} of {bad.size} off, max err {err.max():.3g} (max |ref| {scale:.3g})"


def _check(images_fn, oracle_images, x, c, seed, image_atol=1e-6):
    xg = x.float().cuda().requires_grad_(True)
    cg = c.float().cuda().requires_grad_(True)
    img = images_fn(xg, cg)
    xr = xg.detach().double().cpu().requires_grad_(True)
    cr = cg.detach().double().cpu().requires_grad_(True)
    ref = oracle_images(xr, cr)
    assert img.shape == ref.shape
    _close("image", img.detach().cpu(), ref.detach(), atol=image_atol)
    up = torch.randn(ref.shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    gx, gc = torch.autograd.grad(img, (xg, cg), up.float().cuda())
    rx, rc = torch.autograd.grad(ref, (xr, cr), up)
    _close("dL/dx", gx.cpu(), rx, rtol=1e-4, atol=1e-5)
    _close("dL/dcolor", gc.cpu(), rc, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("ci", range(len(CASES)))
def test_single_image(ci):
    from npa_amd import splatting as SP
    kw = CASES[ci]
    x, c = particles(PARTICLES.get(ci, 700), kw["img_size"], _radius(kw), kw.get("lo", -1.0), kw.get("hi", 1.0),
                     seed=ci, ncolor=3 + ci % 5)
    _check(lambda a, b: SP.splat_particles(a, b, **kw), lambda a, b: S.splat(a, b, **kw), x, c, ci,
           image_atol=IMAGE_ATOL.get(ci, 1e-6))


def test_batch_and_sections():
    from npa_amd import splatting as SP
    kw = CASES[0]
    r = _radius(kw)
    x, c = particles(3 * 300, kw["img_size"], r, -1.0, 1.0, seed=11, ncolor=3)
    _check(lambda a, b: SP.splat_particles_batch(a.view(3, 300, 2), b.view(3, 300, 3), **kw),
           lambda a, b: torch.stack([S.splat(a[i * 300:(i + 1) * 300], b[i * 300:(i + 1) * 300], **kw)
                                     for i in range(3)]), x, c, 1)
    sections = [250, 0, 650]
    bounds = np.cumsum([0] + sections)
    _check(lambda a, b: SP.splat_particles_sections(a, b, sections, **kw),
           lambda a, b: torch.stack([S.splat(a[bounds[i]:bounds[i + 1]], b[bounds[i]:bounds[i + 1]], **kw)
                                     for i in range(3)]), x, c, 2)
    # one block size, the last block shorter (torch.split semantics)
    _check(lambda a, b: SP.splat_particles_sections(a, b, 400, **kw),
           lambda a, b: torch.stack([S.splat(a[i:i + 400], b[i:i + 400], **kw) for i in (0, 400, 800)]), x, c, 3)


def test_deterministic_and_empty():
    from npa_amd import splatting as SP
    kw = CASES[1]
    x, c = particles(5000, kw["img_size"], _radius(kw), -1.0, 1.0, seed=5)
    xg, cg = x.float().cuda(), c.float().cuda()
    a = SP.splat_particles(xg, cg, **kw)
    b = SP.splat_particles(xg, cg, **kw)
    assert torch.equal(a, b)
    far = torch.full((10, 2), 50.0, device="cuda")  # every patch off the image
    assert torch.count_nonzero(SP.splat_particles(far, cg[:10], **kw)) == 0
    assert torch.count_nonzero(SP.splat_particles(far[:0], cg[:0], **kw)) == 0


@pytest.mark.parametrize("img_size,sigma,B,N,spread", [
    (64, 0.8, 8, 60000, 1.1), (33, 1.0, 2, 140000, 1.3), (256, 4.0, 8, 2500, 0.01), (128, 4.0, 1, 21000, 0.7),
    (250, 6.3, 3, 2700, 1.2)])
@pytest.mark.parametrize("odd", [None, "pixel", "color"])
def test_tiled_backward_matches_patches(monkeypatch, img_size, sigma, B, N, spread, odd):
    # the two routes of the gradient, radii 4 to 32, lists that overflow (2500
    # and more particles in a few tiles) and images cut by their edge; sums of the same
    # terms in another order, at most (2 r + 1)^2 of them, each a product of at
    # most six roundings: within 2^-24 (6 + 66) of the sum of magnitudes, taken
    # as 30 times the gradient's largest element
    from npa_amd import splatting as SP
    lib = SP._lib
    kw = dict(img_size=img_size, sigma=sigma, normalize_color=False)
    g = torch.Generator(device="cuda").manual_seed(N)
    x = (torch.rand(B, N, 2, device="cuda", generator=g) * 2 - 1) * spread
    c = torch.rand(B, N, 5, device="cuda", generator=g)
    up = torch.randn(B, img_size, img_size, 4, device="cuda", generator=g)
    if odd == "pixel":
        up[0, img_size // 2, img_size // 2, 1] = float("inf")
    if odd == "color":
        c[0, N // 2, 3] = float("nan")
    assert lib.sphops_splat_backward_workspace_bytes(B * N, img_size, sigma, -1.0, 1.0, 0, 2.0 / 128) > 0
    res = []
    for tiled in (True, False):
        if not tiled:
            monkeypatch.setattr(lib, "sphops_splat_backward_workspace_bytes", lambda *a: 0)
        xr, cr = x.clone().requires_grad_(True), c.clone().requires_grad_(True)
        res.append(torch.autograd.grad(SP.splat_particles_batch(xr, cr, **kw), (xr, cr), up))
    for a, b in zip(*res):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        ok = torch.isfinite(b)
        assert torch.all((a - b)[ok].abs() <= 72 * 2.0 ** -24 * 30 * (b[ok].abs().max() if ok.any() else 0))


def test_large_pixels_outside_a_patch_add_nothing(monkeypatch):
    """Finite upstreams so large that a column's sum times a colour passes the
    largest float, in the rows but not in the columns of some patches: those
    particles' gradients are the same as on the wave per particle's route,
    which never reads such pixels (bound as above)."""
    from npa_amd import splatting as SP
    lib = SP._lib
    kw = dict(img_size=64, sigma=0.8, normalize_color=False)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = (torch.rand(8, 60000, 2, device="cuda", generator=g) * 2 - 1) * 1.1
    c = torch.rand(8, 60000, 3, device="cuda", generator=g) * 30
    up = torch.randn(8, 64, 64, 4, device="cuda", generator=g)
    up[:, :, 20, 1] = 3e38
    assert lib.sphops_splat_backward_workspace_bytes(480000, 64, 0.8, -1.0, 1.0, 0, 2.0 / 128) > 0
    res = []
    for tiled in (True, False):
        if not tiled:
            monkeypatch.setattr(lib, "sphops_splat_backward_workspace_bytes", lambda *a: 0)
        xr, cr = x.clone().requires_grad_(True), c.clone().requires_grad_(True)
        res.append(torch.autograd.grad(SP.splat_particles_batch(xr, cr, **kw), (xr, cr), up))
    for a, b in zip(*res):
        far = torch.isfinite(b).all(-1) & (b.abs().amax(-1) < 1e30)  # the patch does not reach column 20
        assert 0.5 < far.float().mean() < 1.0 and torch.isfinite(a[far]).all()
        assert torch.all((a - b)[far].abs() <= 72 * 2.0 ** -24 * 30 * b[far].abs().max())


@pytest.mark.parametrize("normalize", [True, False])
@pytest.mark.parametrize("N", [9000, 45000])
def test_crowded_images_beside_even_ones(monkeypatch, normalize, N):
    """Images whose particles lie in few tiles leave the tiles' route by
    themselves, beside even ones, an empty one and ones of one and two
    particles, few and many particles a wave; bound as above."""
    from npa_amd import splatting as SP
    lib = SP._lib
    sizes = [N // 3, 0, 1, N // 3 + 5, 2, N - 2 * (N // 3) - 8]
    # radius 32 and, without normalisation, sigma in pixels
    kw = dict(img_size=256, sigma=6.3, normalize_color=normalize, pixel_size=2.0 / 256)
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.rand(N, 2, device="cuda", generator=g) * 2 - 1
    x[:sizes[0]] *= 0.05  # one tile's worth
    x[-sizes[5]:] = x[-sizes[5]:] * 0.2 + 0.9  # a corner, some patches cut, some outside
    c = torch.rand(N, 4, device="cuda", generator=g)
    up = torch.randn(6, 256, 256, 4, device="cuda", generator=g)
    assert lib.sphops_splat_backward_workspace_bytes(N, 256, 6.3, -1.0, 1.0, int(normalize), 2.0 / 256) > 0
    res = []
    for tiled in (True, True, False):
        if not tiled:
            monkeypatch.setattr(lib, "sphops_splat_backward_workspace_bytes", lambda *a: 0)
        xr, cr = x.clone().requires_grad_(True), c.clone().requires_grad_(True)
        res.append(torch.autograd.grad(SP.splat_particles_sections(xr, cr, sizes, **kw), (xr, cr), up))
    for a, again, b in zip(*res):
        assert torch.equal(a, again)
        assert torch.all((a - b).abs() <= 72 * 2.0 ** -24 * 30 * b.abs().max())
    if not normalize:  # a crowded image's patches are swept in the same order on both routes: the same bits
        assert all(torch.equal(a[:sizes[0]], b[:sizes[0]]) for a, b in zip(res[0], res[2]))
