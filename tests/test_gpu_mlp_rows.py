"""The fused MLP (npa_amd.mlp.MlpRows: Linear, ReLU, Linear with 128 hidden
units) against float64, at the edges of its row tiles (32), chunks (64 rows
and up), input groups of 8 and tiles of 32 columns, and output groups and
tiles; and the shapes and types that keep the layers' own functions.

Bounds: an fp32 sum of n products is within (n + 2) 2^-24 of the sum of their
absolute values; a value that goes through both layers adds the first layer's
error times |W2| (or |W1|).  Rows with a pre-activation within that error of
the ReLU's kink get no upstream."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24
SHAPES = [(83, 19), (66, 18), (50, 14), (130, 34), (163, 35), (4, 4), (8, 8), (13, 33), (32, 32), (33, 5), (96, 64),
          (104, 16), (105, 40), (168, 64)]


def _case(rows, nin, nout, bias2, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    net = torch.nn.Sequential(torch.nn.Linear(nin, 128), torch.nn.ReLU(), torch.nn.Linear(128, nout, bias=bias2)).cuda()
    with torch.no_grad():
        for p in net.parameters():
            p.copy_(torch.randn(p.shape, device="cuda", generator=g) / max(p.shape[-1], 8) ** 0.5)
    z = torch.randn(rows, nin, device="cuda", generator=g)
    return net, z, torch.randn(rows, nout, device="cuda", generator=g)


def _check(name, got, ref, bound):
    err = (got.double() - ref).abs()
    assert torch.all(err <= bound + 1e-30), f"{name}: {(err - bound).max().item():.3g} over its bound"


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("rows", [1, 31, 33, 65, 5000])
def test_mlp_rows_match_float64(shape, rows):
    from npa_amd import mlp as M
    nin, nout = shape
    net, z, up = _case(rows, nin, nout, rows % 2 == 1, rows + nin)
    w1, b1, w2 = (t.detach().double() for t in (net[0].weight, net[0].bias, net[2].weight))
    zd = z.double()
    a = zd @ w1.T + b1
    ea = (nin + 3) * EPS * (zd.abs() @ w1.abs().T + b1.abs())
    up[(a.abs() <= 2 * ea).any(1)] = 0
    zr = z.clone().requires_grad_(True)
    y = M.mlp(net, zr)
    assert type(y.grad_fn).__name__.startswith(("MlpRows", "View", "Reshape"))
    y.backward(up)
    h = a.clamp_min(0)
    yd = h @ w2.T + (net[2].bias.double() if net[2].bias is not None else 0)
    mag = h.abs() @ w2.abs().T + (net[2].bias.double().abs() if net[2].bias is not None else 0)
    _check("y", y, yd, 131 * EPS * mag + ea @ w2.abs().T)
    ud = up.double()
    on = (a > 0).double()
    da, eda = (ud @ w2) * on, (nout + 2) * EPS * (ud.abs() @ w2.abs()) * on
    _check("dz", zr.grad, da @ w1, 130 * EPS * (da.abs() @ w1.abs()) + eda @ w1.abs())
    n = (rows + 2) * EPS
    _check("dW1", net[0].weight.grad, da.T @ zd, n * (da.abs().T @ zd.abs()) + eda.T @ zd.abs())
    _check("db1", net[0].bias.grad, da.sum(0), n * da.abs().sum(0) + eda.sum(0))
    _check("dW2", net[2].weight.grad, ud.T @ h, n * (ud.abs().T @ h) + ud.abs().T @ ea)
    if net[2].bias is not None:
        _check("db2", net[2].bias.grad, ud.sum(0), n * ud.abs().sum(0))


def test_mlp_rows_special_values_stay_in_their_row():
    """NaN and infinities reach their own rows' outputs and input gradients
    only, the relu keeps NaN, and leading dimensions and strides are as the
    module's."""
    from npa_amd import mlp as M
    net, z, up = _case(99, 83, 19, True, 3)
    base = z.clone().requires_grad_(True)
    M.mlp(net, base).backward(up)
    bad = z.clone()
    bad[40, 82], bad[41, 0], bad[98, 5] = float("nan"), float("inf"), float("-inf")
    br = bad.clone().requires_grad_(True)
    y = M.mlp(net, br)
    y.backward(up)
    keep = torch.ones(99, dtype=torch.bool, device="cuda")
    keep[[40, 41, 98]] = False
    ref = net(bad)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(br.grad[keep], base.grad[keep])
    strided = z.t().contiguous().t()
    assert torch.equal(M.mlp(net, strided), M.mlp(net, z))
    assert torch.equal(M.mlp(net, z[:98].reshape(2, 49, 83)).reshape(98, 19), M.mlp(net, z[:98]))
    assert M.mlp(net, z[:0]).shape == (0, 19)


def test_mlp_rows_is_deterministic_and_optional():
    from npa_amd import mlp as M
    net, z, up = _case(70001, 83, 19, False, 5)
    grads = []
    for _ in range(2):
        net.zero_grad()
        zr = z.clone().requires_grad_(True)
        M.mlp(net, zr).backward(up)
        grads.append([zr.grad, *(p.grad.clone() for p in net.parameters())])
    assert all(torch.equal(a, b) for a, b in zip(*grads))
    with torch.no_grad():
        y = M.mlp(net, z)
    assert not y.requires_grad and torch.allclose(y, net(z), rtol=1e-5, atol=1e-5)
    net[0].weight.requires_grad_(False)  # each gradient alone
    net.zero_grad()
    M.mlp(net, z).backward(up)
    assert net[0].weight.grad is None and torch.equal(net[2].weight.grad, grads[0][3])
    for other in (torch.nn.Sequential(torch.nn.Linear(83, 64), torch.nn.ReLU(), torch.nn.Linear(64, 19)),
                  torch.nn.Sequential(torch.nn.Linear(200, 128), torch.nn.ReLU(), torch.nn.Linear(128, 19))):
        other = other.cuda()  # shapes the kernels do not take: the layers' own functions
        v = torch.randn(50, other[0].in_features, device="cuda")
        assert torch.allclose(M.mlp(other, v), other(v), rtol=1e-5, atol=1e-5)


def test_pre_activations_only_for_a_backward(monkeypatch):
    """The 512 bytes a row that only the backward reads are written where one
    can follow: not under no_grad, and not without an input that needs a
    gradient."""
    from npa_amd import mlp as M
    net, z, _ = _case(200, 83, 19, True, 7)
    kept, call = [], M._lib.sphops_mlp_forward
    monkeypatch.setattr(M._lib, "sphops_mlp_forward", lambda *a: kept.append(bool(a[5].value)) or call(*a))
    with torch.no_grad():
        y = M.mlp(net, z)
        M.mlp(net, z.clone().requires_grad_(True))
    ref = M.mlp(net, z)
    for p in net.parameters():
        p.requires_grad_(False)
    M.mlp(net, z)
    assert kept == [False, False, True, False] and torch.equal(y, ref)


@pytest.mark.parametrize("rows,shape", [(300001, (83, 19)), (300001, (100, 16)), (300001, (163, 40)), (32769, (163, 40)),
                                        (32800, (130, 32))])
def test_many_rows_match_float64(rows, shape):
    """Every wave's second and later row tiles, the moves of the second
    layer's sums to LDS, ragged last chunks, and both sides of the forward's
    two workgroup sizes.  The sums' 2-norms are within 4e-6, ten times what
    their roundings measure; a row tile left out or read twice is off by
    (32 / rows)^(1/2), 1e-2."""
    from npa_amd import mlp as M
    nin, nout = shape
    net, z, up = _case(rows, nin, nout, True, nin)
    w1, b1, w2, b2 = (t.detach().double() for t in (net[0].weight, net[0].bias, net[2].weight, net[2].bias))
    zd = z.double()
    a = zd @ w1.T + b1
    up[(a.abs() < 1e-5).any(1)] = 0
    zr = z.clone().requires_grad_(True)
    y = M.mlp(net, zr)
    y.backward(up)
    with torch.no_grad():
        assert torch.equal(M.mlp(net, z), y)
    h, ud = a.clamp_min(0), up.double()
    da = (ud @ w2) * (a > 0)
    for name, got, ref in (("y", y, h @ w2.T + b2), ("dz", zr.grad, da @ w1), ("dW1", net[0].weight.grad, da.T @ zd),
                           ("db1", net[0].bias.grad, da.sum(0)), ("dW2", net[2].weight.grad, ud.T @ h),
                           ("db2", net[2].bias.grad, ud.sum(0))):
        assert ((got.double() - ref).norm() <= 4e-6 * ref.norm()).item(), name
    last = rows - rows % 32  # the ragged last row tile, row by row
    for got, ref in ((y, h @ w2.T + b2), (zr.grad, da @ w1)):
        assert torch.all((got[last - 32:].double() - ref[last - 32:]).abs() <= 1e-5 * ref.abs().max())
