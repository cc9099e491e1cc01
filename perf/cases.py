"""What this framework is timed on: its public calls, as programs make them.

A case is one call sequence of a Neural Particle Automata program, at one size:

* ``step``    one ``step_euler`` (or ``step_euler_trace``) of the model: perception, MLP, Euler
              update; in inference under ``no_grad``, in training with its backward (the gradients of
              positions, states and weights).  The model's defaults: positions are not differentiated
              through perception.
* ``static``  the state-only model's ``step_euler_static`` (point-cloud classification), in training.
* ``ops``     the perception operators as ``NPA.perceive`` calls them, with the full backward (positions
              too): the path of a model without stopped position gradients.
* ``fields``  the single operators a program evaluates fields with: count, density, gradient and moment
              matrix, with their backward.
* ``binning`` instantiate, bin and unbin: sorting a cloud into cells and rows back.
* ``mlp``     the model's MLP over one row per particle, with its backward.
* ``splat``   2D Gaussian splatting of a batch of particle clouds, with its backward.

Clouds: the uniform disk and segments of the 2D growing and classification workloads, the uniform
periodic box of the texture workload, and the Gaussian mixtures of the 3D ones (the mixture is fixed, the
seed draws the points).  Radii keep each workload's mean neighbour count at every size.  A step's particles
come in the order its predecessor leaves them (binned, then moved by a fraction of the radius), as in a
rollout; the other kinds take them in random order, as a data set holds them.
"""
import itertools
import math

import numpy as np
import torch

DEVICE = "cuda"
HIDDEN = 128  # the model's hidden units

# Gaussian mixtures (components, sigma range, log-uniform sigmas) and the radius that gives the reference
# size its mean neighbour count: 30 (growth) and 32 (stress)
MIXTURES = {"growth": (4, 0.05, 0.2, False, 65536, 0.028674138709902763),
            "stress": (8, 0.01, 0.2, True, 1048576, 0.0026222667656838894)}


def listed():
    return [
        # the interactive viewer: one 2D growing cloud stepped forever, latency-bound
        dict(name="step_2d_infer", kind="step", train=False, trace=False, dim=2, cloud="disk", periodic=False,
             mode="grid", B=1, N=4096, C=16, maxp=32, update_prob=1.0),
        # training of the 2D growing model: a batch of clouds, stochastic updates
        dict(name="step_2d_train", kind="step", train=True, trace=False, dim=2, cloud="disk", periodic=False,
             mode="grid", B=8, N=4096, C=16, maxp=32, update_prob=0.5),
        # 2D texture synthesis in the periodic box, differentiated through positions
        dict(name="ops_2d_texture", kind="ops", dim=2, cloud="box", periodic=True, mode="grid", B=4, N=16384, C=12,
             maxp=32),
        # point-cloud classification: many small clouds, the state-only model
        dict(name="static_2d_train", kind="static", dim=2, cloud="segments", periodic=False, mode="grid", B=64, N=512,
             C=32, maxp=64, update_prob=0.5),
        # growth of a 3D Gaussian-splat object, wide states
        dict(name="ops_3d_growth", kind="ops", dim=3, cloud="growth", periodic=False, mode="grid", B=1, N=65536, C=32,
             maxp=64),
        # the largest perception call: a million particles of very uneven density
        dict(name="ops_3d_stress", kind="ops", dim=3, cloud="stress", periodic=False, mode="grid", B=1, N=1048576,
             C=16, maxp=64),
        # the largest whole training step
        dict(name="step_3d_train", kind="step", train=True, trace=False, dim=3, cloud="stress", periodic=False,
             mode="grid", B=1, N=1048576, C=16, maxp=64, update_prob=0.5),
        # offline rendering of a 3D model: traced steps (input order) on a Morton grid, an odd particle count
        dict(name="step_3d_trace", kind="step", train=False, trace=True, dim=3, cloud="growth", periodic=False,
             mode="particle", B=1, N=250007, C=16, maxp=64, update_prob=1.0),
        # field evaluation and its adjoint in a small 3D periodic box, a ragged size and an unusual width
        dict(name="fields_3d_periodic", kind="fields", dim=3, cloud="box", periodic=True, mode="grid", B=3, N=20011,
             C=20, maxp=64),
        # sorting a large 3D cloud with wide states and putting the rows back
        dict(name="binning_3d", kind="binning", dim=3, cloud="stress", periodic=False, mode="grid", B=1, N=400003,
             C=32, maxp=64),
        # the MLP of the 3D model over a million particles
        dict(name="mlp_train", kind="mlp", dim=3, rows=1048576, C=16),
        # images of a batch of growing clouds for an image loss
        dict(name="splat_2d_train", kind="splat", B=8, N=4096, C=16, img=256, pixel=2.0 / 64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges; every size is drawn on a log scale."""
    kind = rng.choice(["step2", "step2", "step3", "static", "ops2", "ops3", "ops3", "fields", "binning", "mlp", "splat"])
    maxp = rng.choice([32, 64])
    prob = rng.choice([0.5, 1.0])
    if kind == "step2":
        N = _log(rng, 1000, 40000)
        return dict(kind="step", train=rng.random() < 0.5, trace=False, dim=2, cloud=rng.choice(["disk", "box"]),
                    periodic=False, mode="grid", B=min(8, max(1, 65536 // N)), N=N, C=rng.choice([12, 16, 32]),
                    maxp=maxp, update_prob=prob)
    if kind == "step3":
        train = rng.random() < 0.5
        return dict(kind="step", train=train, trace=not train, dim=3, cloud=rng.choice(["growth", "stress"]),
                    periodic=False, mode="grid", B=1, N=_log(rng, 20000, 700000), C=rng.choice([12, 16]), maxp=maxp,
                    update_prob=prob)
    if kind == "static":
        N = _log(rng, 128, 2048)
        return dict(kind="static", dim=2, cloud="segments", periodic=False, mode="grid", B=max(1, 32768 // N), N=N,
                    C=rng.choice([16, 32]), maxp=64, update_prob=prob)
    if kind == "ops2":
        N = _log(rng, 2000, 60000)
        cloud = rng.choice(["disk", "box"])
        return dict(kind="ops", dim=2, cloud=cloud, periodic=cloud == "box", mode="grid", B=max(1, 65536 // N), N=N,
                    C=rng.choice([12, 16, 20, 32]), maxp=maxp)
    if kind == "ops3":
        cloud = rng.choice(["growth", "stress", "box"])
        return dict(kind="ops", dim=3, cloud=cloud, periodic=cloud == "box", mode="grid", B=1, N=_log(rng, 20000, 900000),
                    C=rng.choice([12, 16]), maxp=maxp)
    if kind == "fields":
        return dict(kind="fields", dim=3, cloud="box", periodic=True, mode="grid", B=rng.choice([1, 3]),
                    N=_log(rng, 5000, 60000), C=rng.choice([8, 16, 20]), maxp=64)
    if kind == "binning":
        return dict(kind="binning", dim=3, cloud=rng.choice(["growth", "stress"]), periodic=False, mode="grid", B=1,
                    N=_log(rng, 30000, 800000), C=rng.choice([16, 32]), maxp=64)
    if kind == "mlp":
        dim = rng.choice([2, 3])
        return dict(kind="mlp", dim=dim, rows=_log(rng, 20000, 1000000), C=rng.choice([12, 16]))
    return dict(kind="splat", B=rng.choice([1, 4, 8]), N=_log(rng, 500, 4096), C=16, img=rng.choice([128, 200, 256]),
                pixel=rng.choice([2.0 / 64, 2.0 / 128]))


# ------------------------------------------------------------------ inputs (from the seed alone)

def _geometry(case):
    """(radius, cells per axis) of a case's cloud: the workload's mean neighbour count at this size."""
    N, D, cloud = case["N"], case["dim"], case["cloud"]
    if cloud == "box":  # unit box centred on the origin, about 24 (2D) or 32 (3D) neighbours, a whole number of cells
        h = math.sqrt(24.0 / (math.pi * N)) if D == 2 else (32.0 / (4.0 / 3.0 * math.pi * N)) ** (1.0 / 3.0)
        G = max(3, round(1.0 / h))
        return float(np.float32(1.0 / G)), (G,) * D
    if cloud == "disk":  # unit disk, about 20 neighbours
        h, ext = math.sqrt(20.0 / N), np.ones(2)
    elif cloud == "segments":
        h, ext = 0.06505652517080307 * math.sqrt(512.0 / N), np.full(2, 1.04)
    else:
        n0, h0 = MIXTURES[cloud][4:]
        h = h0 * (n0 / N) ** (1.0 / 3.0)
        means, sig = _mixture(cloud)
        ext = np.sort(np.abs(means) + 3.0 * sig[:, None], axis=0)[-1] * 0.9
    h = float(np.float32(h))
    G = tuple(int(2 * math.ceil(e / h) + 2) for e in ext)
    if case["mode"] == "particle":  # Morton order: a cubic grid of a power-of-two side
        G = (min(1024, 1 << (max(G) - 1).bit_length()),) * D
    return h, G


def _mixture(cloud):
    k, lo, hi, log_sigma = MIXTURES[cloud][:4]
    rng = np.random.default_rng(42)
    means = rng.uniform(-0.5, 0.5, (k, 3))
    sig = np.exp(rng.uniform(math.log(lo), math.log(hi), k)) if log_sigma else rng.uniform(lo, hi, k)
    return means, sig


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _positions(case, g):
    """(B, N, D) positions of the case's cloud."""
    B, N, D, cloud = case["B"], case["N"], case["dim"], case["cloud"]

    def rand(*shape):
        return torch.rand(*shape, device=DEVICE, generator=g)

    def randn(*shape):
        return torch.randn(*shape, device=DEVICE, generator=g)

    if cloud == "box":
        return rand(B, N, D) - 0.5
    if cloud == "disk":
        r, t = torch.sqrt(rand(B, N)), 2.0 * math.pi * rand(B, N)
        return torch.stack([r * torch.cos(t), r * torch.sin(t)], -1)
    if cloud == "segments":  # 3 to 6 random segments a cloud, points spread evenly over their length
        a, b = rand(B, 6, 2) * 2 - 1, rand(B, 6, 2) * 2 - 1
        used = torch.arange(6, device=DEVICE)[None] < 3 + torch.floor(4 * rand(B, 1))
        edges = torch.cumsum((b - a).norm(dim=-1) * used, 1)
        u = rand(B, N) * edges[:, -1:]
        seg = torch.searchsorted(edges, u).clamp_max(5)
        a, b = (t.gather(1, seg[..., None].expand(-1, -1, 2)) for t in (a, b))
        return a + rand(B, N, 1) * (b - a) + 0.02 * randn(B, N, 2)
    means, sig = (torch.as_tensor(t, dtype=torch.float32, device=DEVICE) for t in _mixture(cloud))
    comp = torch.randint(len(sig), (B, N), device=DEVICE, generator=g)
    return means[comp] + randn(B, N, 3) * sig[comp][..., None]


def _inputs(case, seed):
    """The tensors a program has before the call."""
    g = _generator(seed)

    def randn(*shape):
        return torch.randn(*shape, device=DEVICE, generator=g)

    if case["kind"] == "mlp":
        W, out = _feature_width(case), case["dim"] + case["C"]
        d = dict(z=randn(case["rows"], W), up=randn(case["rows"], out), **_weights(W, out, g))
        d["up"][_at_kink(d["z"].double(), d)] = 0
        return d
    B, N, C = case["B"], case["N"], case["C"]
    if case["kind"] == "splat":
        return dict(x=(torch.rand(B, N, 2, device=DEVICE, generator=g) - 0.5) * 1.6,
                    color=torch.rand(B, N, C, device=DEVICE, generator=g), up=randn(B, case["img"], case["img"], 4))
    D = case["dim"]
    h, _ = _geometry(case)
    pos = _positions(case, g)
    if case["kind"] in ("step", "static"):  # a rollout's particles: last step's binned order, moved since
        order = _order(case, pos)
        pos = pos.gather(1, order[..., None].expand(-1, -1, D)) + 0.1 * h * randn(B, N, D)
    x = torch.zeros(B, N, 2 if D == 2 else 4, device=DEVICE)
    x[..., :D] = pos
    d = dict(x=x, s=randn(B, N, C))
    if case["kind"] == "ops":
        d.update(up_blur=randn(B, N, C), up_grad=randn(B, N, C, D), up_rho=randn(B, N, D))
    elif case["kind"] == "fields":
        d.update(mass=0.5 + torch.rand(B, N, device=DEVICE, generator=g), up_density=randn(B, N),
                 up_grad=randn(B, N, C, D), up_moment=randn(B, N, D, D))
    elif case["kind"] in ("step", "static"):
        out = C if case["kind"] == "static" else D + C
        d.update(up_x=randn(*x.shape), up_s=randn(B, N, C), seed=seed, **_weights(_feature_width(case), out, g))
        if case["kind"] == "static" or case["train"]:
            p = _perception(case, d)
            kink = _at_kink(_features(case, p.forward(), p.s), d).reshape(B, N)
            d["up_x"][kink], d["up_s"][kink] = 0, 0
    return d


def _at_kink(z, d):
    """Rows with a hidden unit so near its ReLU's kink that 32 bits do not decide the side (about one in a
    thousand).  Their gradient is not defined in 32 bits, so they get no upstream, like a particle that the
    update mask leaves out."""
    return ((z @ d["w1"].double().T + d["b1"].double()).abs() < 1e-5).any(1)


def _feature_width(case):
    C, D = case["C"], case["dim"]
    return 2 * C + C * D + D


def _weights(fan_in, out, g):
    def uniform(bound, *shape):
        return (torch.rand(*shape, device=DEVICE, generator=g) * 2 - 1) * bound

    a, b = 1.0 / math.sqrt(fan_in), 1.0 / math.sqrt(HIDDEN)
    return dict(w1=uniform(a, HIDDEN, fan_in), b1=uniform(a, HIDDEN), w2=uniform(b, out, HIDDEN))


class _Model(torch.nn.Module):
    """The attributes of the reference's NPA module that its step reads (models/npa.py:15-63)."""

    def __init__(self, dim, net):
        super().__init__()
        self.spatial_dims = dim
        self.register_buffer("eps0", torch.tensor([0.1]))
        self.register_buffer("alpha", torch.tensor([1.0]))
        self.state_grad = self.density_grad = self.log_norm_grad = self.log_norm_density_grad = True
        self.stopgrad_pos, self.stopgrad_state = True, False
        self.model = net


def _net(d):
    net = torch.nn.Sequential(torch.nn.Linear(d["w1"].shape[1], HIDDEN), torch.nn.ReLU(),
                              torch.nn.Linear(HIDDEN, d["w2"].shape[0], bias=False)).to(DEVICE)
    with torch.no_grad():
        net[0].weight.copy_(d["w1"])
        net[0].bias.copy_(d["b1"])
        net[2].weight.copy_(d["w2"])
    return net


def prepare(case, seed):
    import npa_amd.sphops as sp

    d = _inputs(case, seed)
    state = dict(case=case, **d)
    if "w1" in d:
        net = _net(d)
        state["net"] = net
        if "dim" in case and case["kind"] != "mlp":
            state["model"] = _Model(case["dim"], net).to(DEVICE)
    if "x" in d and case["kind"] != "splat":
        h, G = _geometry(case)
        state["grid"] = sp.HashGrid(dim=case["dim"], boundary="periodic" if case["periodic"] else "clamped",
                                    mode=case["mode"], grid_size=list(G), eps=h, num_particles=case["N"],
                                    batch_size=case["B"], max_particles_per_block=case["maxp"])
    return state


# ------------------------------------------------------------------ one pass

def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


def _leaf(t):
    return t.detach().requires_grad_(True)


def _gradients(net):
    return dict(w1=net[0].weight.grad, b1=net[0].bias.grad, w2=net[2].weight.grad)


def _run_step(st, case):
    from npa_amd import step

    if case["update_prob"] < 1.0:
        torch.cuda.manual_seed(st["seed"])  # a reproducible run
    if not case["train"]:
        with torch.no_grad():
            if case["trace"]:
                x, s, dx, ds = step.step_euler_trace(st["model"], st["x"], st["s"], st["grid"],
                                                     update_prob=case["update_prob"], return_aux=True)
                return dict(x=x, s=s, dx=dx, ds=ds)
            x, s, _ = step.step_euler(st["model"], st["x"], st["s"], st["grid"], update_prob=case["update_prob"])
            return dict(x=x, s=s)
    st["model"].zero_grad(set_to_none=True)
    x0, s0 = _leaf(st["x"]), _leaf(st["s"])
    x, s, _ = step.step_euler(st["model"], x0, s0, st["grid"], update_prob=case["update_prob"])
    torch.autograd.backward([x, s], [st["up_x"], st["up_s"]])
    return dict(x=x.detach(), s=s.detach(), grad_x=x0.grad, grad_s=s0.grad, **_gradients(st["net"]))


def _run_static(st, case):
    from npa_amd import step

    if case["update_prob"] < 1.0:
        torch.cuda.manual_seed(st["seed"])
    st["model"].zero_grad(set_to_none=True)
    s0 = _leaf(st["s"])
    x, s = step.step_euler_static(st["model"], st["x"], s0, st["grid"], update_prob=case["update_prob"])
    s.backward(st["up_s"])
    return dict(x=x.detach(), s=s.detach(), grad_s=s0.grad, **_gradients(st["net"]))


def _run_ops(st, case):
    import npa_amd.sphops as sp

    x0, s0 = _leaf(st["x"]), _leaf(st["s"])
    with torch.no_grad():
        snap = st["grid"].instantiate(x0)
    x, s = sp.bin_particles(x0, s0, snap)
    rho = sp.density(x, snap)
    blur = sp.blur(x, rho, s, snap)
    grad = sp.gradient_hybrid(x, rho, s, snap)
    grad_rho = sp.density_gradient(x, snap)
    torch.autograd.backward([blur, grad, grad_rho], [st["up_blur"], st["up_grad"], st["up_rho"]])
    return dict(permutation=snap.permutation, rho=rho.detach(), blur=blur.detach(), grad=grad.detach(),
                grad_rho=grad_rho.detach(), grad_x=x0.grad, grad_s=s0.grad)


def _run_fields(st, case):
    import npa_amd.sphops as sp

    x0, s0 = _leaf(st["x"]), _leaf(st["s"])
    with torch.no_grad():
        snap = st["grid"].instantiate(x0)
    x, s, m = sp.bin_particles(x0, s0, snap, st["mass"])
    n = sp.count(x, snap)
    rho = sp.density(x, snap, m)
    grad = sp.gradient(x, rho, s, snap, m)
    moment = sp.moment_matrix(x, rho, snap, m)
    torch.autograd.backward([rho, grad, moment], [st["up_density"], st["up_grad"], st["up_moment"]])
    return dict(permutation=snap.permutation, count=n, rho=rho.detach(), grad=grad.detach(), moment=moment.detach(),
                grad_x=x0.grad, grad_s=s0.grad)


def _run_binning(st, case):
    import npa_amd.sphops as sp

    with torch.no_grad():
        snap = st["grid"].instantiate(st["x"])
        x, s = sp.bin_particles(st["x"], st["s"], snap)
        x0, s0 = sp.unbin_particles(x, s, snap)
    return dict(permutation=snap.permutation, bin_offsets=snap.bin_offsets, block_info=snap.block_info,
                total_blocks=snap.total_blocks, x_bin=x, s_bin=s, x=x0, s=s0)


def _run_mlp(st, case):
    from npa_amd import mlp

    st["net"].zero_grad(set_to_none=True)
    z = _leaf(st["z"])
    y = mlp.mlp(st["net"], z)
    y.backward(st["up"])
    return dict(y=y.detach(), grad_z=z.grad, **_gradients(st["net"]))


def _run_splat(st, case):
    from npa_amd import splatting

    x, c = _leaf(st["x"]), _leaf(st["color"])
    img = splatting.splat_particles_batch(x, c, img_size=case["img"], sigma=1.0, y_up=True, pixel_size=case["pixel"])
    img.backward(st["up"])
    return dict(image=img.detach(), grad_x=x.grad, grad_color=c.grad)


_RUN = dict(step=_run_step, static=_run_static, ops=_run_ops, fields=_run_fields, binning=_run_binning, mlp=_run_mlp,
            splat=_run_splat)


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    """Bytes: each input read once and each output written once.  Operations: those of the in-radius pairs
    (the workload's mean neighbour count, self included), of the MLP's products and of the splat's patches."""
    kind, C = case["kind"], case["C"]
    f = 4
    if kind == "mlp":
        W, out, R = _feature_width(case), case["dim"] + C, case["rows"]
        return dict(bytes=f * R * (2 * W + 2 * out) + 2 * f * HIDDEN * (W + out + 1),
                    flops=3 * 2 * R * HIDDEN * (W + out))
    B, N = case["B"], case["N"]
    if kind == "splat":
        r = math.ceil(5 * case["img"] * case["pixel"] / 2)
        pix = f * 4 * B * case["img"] ** 2
        return dict(bytes=2 * pix + 2 * f * B * N * (2 + C), flops=2 * B * N * (2 * r + 1) ** 2 * 12)
    D, P = case["dim"], 2 if case["dim"] == 2 else 4
    n = B * N
    _, G = _geometry(case)
    cells = B * math.prod(G)
    pairs = n * {"disk": 20, "segments": 16, "growth": 30, "stress": 32, "box": 24 if D == 2 else 32}[case["cloud"]]
    if kind == "binning":
        return dict(bytes=f * (n * (3 * P + 3 * C + 2) + 4 * n + cells), flops=n * 4 * D)
    geometry = 3 * D + 10
    forward = geometry + 2 + 2 * D + C * (2 + 2 * D) + D * (D + 1)  # density, its gradient, blur, gradient, moments
    if kind == "ops":
        return dict(bytes=f * (n * (2 * P + 4 * C + 2 * C * D + 2 * D + 2) + cells),
                    flops=pairs * (forward + geometry + C * (6 + 8 * D) + 4 * D * D))
    if kind == "fields":
        return dict(bytes=f * (n * (2 * P + 2 * C + 2 * C * D + 2 * D * D + 5) + cells),
                    flops=pairs * (2 * geometry + C * (10 * D + 2) + 4 * D * D))
    W, out = _feature_width(case), (C if kind == "static" else D + C)
    train = kind == "static" or case["train"]
    weights = HIDDEN * (W + out + 1)
    row = 2 * P + 2 * C
    if train:
        row += P + 2 * C + (P if kind == "step" else 0)
    elif case["trace"]:
        row += P + C
    return dict(bytes=f * (n * row + cells + weights * (2 if train else 1)),
                flops=pairs * (forward + (geometry + C * (2 + 4 * D) if train else 0))
                + 2 * n * HIDDEN * (W + out) * (3 if train else 1))


def tolerance(case):
    """About four times the error of this framework's 32-bit results against ``exact``, over the listed and
    a hundred drawn cases.  Sums of a few dozen pair terms are within 5e-7.  What divides by small numbers is
    further off: the corrected state gradient by nearly singular moment matrices (3e-6, single values 2e-4),
    and the position gradient by the distance of the closest pairs, which a periodic box's wrapped
    displacements round once more (5e-4, single values 2e-2)."""
    kind = case["kind"]
    if kind == "binning":
        return "exact"
    if kind == "ops":
        return {"rel": 2e-3, "max": 7e-2} if case["periodic"] else {"rel": 1.2e-5, "max": 8e-4}
    if kind == "fields":
        return {"rel": 8e-6, "max": 8e-4}
    if kind == "splat":
        return {"rel": 1.7e-5, "max": 2e-4}
    return {"rel": 2e-6, "max": 2e-4}


# ------------------------------------------------------------------ the same results in 64 bits

def exact(case, seed):
    """What ``run`` returns, from plain torch in float64 (pair sums by a cell list of its own, gradients by
    autograd over the pairs)."""
    d = _inputs(case, seed)
    return _EXACT[case["kind"]](case, d)


def _cells(case, pos):
    """Cell key of every position (B, N), as the grid defines it: floor(x / h) in 32 bits from the middle of
    the grid, clamped or wrapped, row-major or bit-interleaved."""
    h, G = _geometry(case)
    inv = np.float32(1.0) / np.float32(h)
    c = [torch.floor(pos[..., d] * torch.tensor(inv, device=pos.device)).long() + G[d] // 2 for d in range(case["dim"])]
    c = [t.remainder(g) if case["periodic"] else t.clamp(0, g - 1) for t, g in zip(c, G)]
    if case["mode"] == "particle":
        key = torch.zeros_like(c[0])
        for bit in range(10):
            for d, t in enumerate(c):
                key |= ((t >> bit) & 1) << (bit * len(c) + d)
        return key
    key = c[-1]
    for d in reversed(range(case["dim"] - 1)):
        key = key * G[d] + c[d]
    return key


def _order(case, pos):
    """Source row of every binned slot (B, N): by cell, then by input order."""
    return torch.argsort(_cells(case, pos), dim=1, stable=True)


def _slots(order):
    """Destination slot of every row: the inverse of ``order``."""
    slots = torch.empty_like(order)
    return slots.scatter_(1, order, torch.arange(order.shape[1], device=order.device).expand_as(order))


def _take(t, order):
    return t.gather(1, order.reshape(order.shape + (1,) * (t.dim() - 2)).expand(t.shape))


class _Pairs:
    """In-radius pairs (i, j) of flat float64 positions, found by sorting into cells of side h, visited in
    chunks of whole cells."""

    def __init__(self, case, x):
        self.h, G = _geometry(case)
        B, N, D = case["B"], case["N"], case["dim"]
        self.D, self.n = D, B * N
        self.x = x.reshape(B * N, -1)[:, :D]
        self.box = None
        cell = torch.floor(self.x / self.h).long()
        if case["periodic"]:
            side = torch.tensor([float(np.float32(np.float32(g) * np.float32(self.h))) for g in G], dtype=torch.float64,
                                device=x.device)
            self.box, size = side, torch.tensor(G, device=x.device)
            cell = cell.remainder(size)
        else:
            cell = cell - cell.amin(0) + 1
            size = cell.amax(0) + 2
        self.size, self.cell = size, cell
        self.cloud = torch.arange(B, device=x.device).repeat_interleave(N)
        self.key, self.rank = torch.sort(self._key(cell))

    def _key(self, cell):
        k = self.cloud
        for d in range(self.D):
            k = k * self.size[d] + cell[:, d]
        return k

    def chunks(self, budget=1 << 21):
        """Yields (i, j): all pairs of a run of particles, about ``budget`` candidates at a time."""
        spans = []
        for off in itertools.product((-1, 0, 1), repeat=self.D):
            c = self.cell + torch.tensor(off, device=self.cell.device)
            if self.box is not None:
                c = c.remainder(self.size)
            k = self._key(c)
            lo = torch.searchsorted(self.key, k)
            spans.append((lo, torch.searchsorted(self.key, k, right=True) - lo))
        total = torch.cumsum(sum(n for _, n in spans), 0)
        cuts = torch.searchsorted(total, torch.arange(budget, int(total[-1]) + budget, budget, device=total.device))
        a = 0
        for b in [min(int(c) + 1, self.n) for c in cuts]:
            if b <= a:
                continue
            ii, jj = [], []
            for lo, n in spans:
                m = n[a:b]
                i = torch.repeat_interleave(torch.arange(a, b, device=m.device), m)
                first = torch.cumsum(m, 0) - m
                j = self.rank[lo[i] + torch.arange(i.numel(), device=m.device) - first[i - a]]
                keep = self.squared(self.displacement(self.x, i, j)) < self.h * self.h
                ii.append(i[keep])
                jj.append(j[keep])
            yield torch.cat(ii), torch.cat(jj)
            a = b

    def displacement(self, x, i, j):
        r = x.index_select(0, j)[:, :self.D] - x.index_select(0, i)[:, :self.D]
        if self.box is not None:
            r = r - self.box * torch.floor(r.detach() / self.box + 0.5)
        return r

    @staticmethod
    def squared(r):
        return (r * r).sum(-1)

    def kernels(self, r, i, j):
        """poly6 W and spiky gradient K of a pair (K = 0 for a particle with itself)."""
        h, D = self.h, self.D
        c6, cs = ((4 / math.pi / h ** 8, 10 / math.pi / h ** 5) if D == 2
                  else (315 / (64 * math.pi) / h ** 9, 15 / math.pi / h ** 6))
        d2 = self.squared(r)
        W = c6 * (h * h - d2).clamp_min(0) ** 3
        other = i != j
        dist = torch.sqrt(torch.where(other, d2, torch.ones_like(d2)))
        K = torch.where(other, cs * 3 * (h - dist).clamp_min(0) ** 2 / dist, torch.zeros_like(d2))[:, None] * r
        return W, K


def _sum(n, i, t):
    return torch.zeros((n,) + t.shape[1:], dtype=t.dtype, device=t.device).index_add(0, i, t)


class _Perception:
    """The perception sums over a cloud's pairs, and their gradients by autograd chunk by chunk."""

    def __init__(self, case, x, s, mass=None):
        self.p = _Pairs(case, x)
        self.n, self.D = self.p.n, case["dim"]
        self.x = x.reshape(self.n, -1)
        self.s = s.reshape(self.n, -1)
        self.m = torch.ones(self.n, dtype=x.dtype, device=x.device) if mass is None else mass.reshape(-1)
        self.pairs = list(self.p.chunks())

    def first(self, x, i, j):
        """Count, density and its gradient."""
        W, K = self.p.kernels(self.p.displacement(x, i, j), i, j)
        m = self.m[j]
        return m * W, m[:, None] * K

    def second(self, x, s, rho, i, j):
        """Blur, state gradient and moment matrix."""
        r = self.p.displacement(x, i, j)
        W, K = self.p.kernels(r, i, j)
        v = self.m[j] / rho.index_select(0, j)
        sj = s.index_select(0, j)
        ds = sj - s.index_select(0, i)
        return ((v * W)[:, None] * sj, v[:, None, None] * ds[:, :, None] * K[:, None, :],
                v[:, None, None] * r[:, :, None] * K[:, None, :])

    def forward(self):
        def zeros(*shape):
            return torch.zeros(self.n, *shape, dtype=torch.float64, device=self.x.device)

        C, D = self.s.shape[1], self.D
        o = dict(count=zeros(), rho=zeros(), grad_rho=zeros(D), blur=zeros(C), grad=zeros(C, D), moment=zeros(D, D))
        for i, j in self.pairs:
            w, k = self.first(self.x, i, j)
            o["count"].index_add_(0, i, torch.ones_like(w))
            o["rho"].index_add_(0, i, w)
            o["grad_rho"].index_add_(0, i, k)
        for i, j in self.pairs:
            for name, t in zip(("blur", "grad", "moment"), self.second(self.x, self.s, o["rho"], i, j)):
                o[name].index_add_(0, i, t)
        det = torch.linalg.det(o["moment"])
        solve = torch.where((det.abs() < 1e-3)[:, None, None], torch.eye(D, dtype=det.dtype, device=det.device),
                            o["moment"])
        o["hybrid"] = o["grad"] @ torch.linalg.inv(solve)
        return o

    def backward(self, rho, positions=True, up_rho=None, up_grad_rho=None, up_blur=None, up_grad=None, up_moment=None):
        """Gradients of x and s (the state gradient's stands for the hybrid's: its correction is a constant)."""
        x, s, r = (t.detach().clone().requires_grad_(True) for t in (self.x, self.s, rho))
        for i, j in self.pairs:
            terms = self.second(x if positions else self.x, s, r if positions else rho, i, j)
            ups = (up_blur, up_grad, up_moment)
            some = [(t, u.index_select(0, i)) for t, u in zip(terms, ups) if u is not None]
            torch.autograd.backward([t for t, _ in some], [u for _, u in some])
        if positions:
            g = r.grad if up_rho is None else r.grad + up_rho
            for i, j in self.pairs:
                w, k = self.first(x, i, j)
                some = [(w, g.index_select(0, i))]
                if up_grad_rho is not None:
                    some.append((k, up_grad_rho.index_select(0, i)))
                torch.autograd.backward([t for t, _ in some], [u for _, u in some])
        return x.grad, s.grad


def _perception(case, d):
    order = _order(case, d["x"])
    return _Perception(case, *(_take(d[k], order).double() for k in ("x", "s", "mass") if k in d))


def _exact_ops(case, d):
    B, N, C, D = case["B"], case["N"], case["C"], case["dim"]
    fields = case["kind"] == "fields"
    p = _perception(case, d)
    slots = _slots(_order(case, d["x"]))
    o = p.forward()
    out = dict(permutation=slots.int())
    if fields:
        names = dict(count="count", rho="rho", grad="grad", moment="moment")
        ups = dict(up_rho=d["up_density"], up_grad=d["up_grad"], up_moment=d["up_moment"])
    else:
        names = dict(rho="rho", blur="blur", grad="hybrid", grad_rho="grad_rho")
        ups = dict(up_blur=d["up_blur"], up_grad=d["up_grad"], up_grad_rho=d["up_rho"])
    for k, v in names.items():
        # (the counts have no 64-bit value: whether a pair at the radius counts is decided in 32 bits)
        out[k] = None if k == "count" else o[v].reshape((B, N) + o[v].shape[1:])
    gx, gs = p.backward(o["rho"], **{k: u.double().flatten(0, 1) for k, u in ups.items()})
    out["grad_x"], out["grad_s"] = (_take(t.reshape(B, N, -1), slots) for t in (gx, gs))
    return out


def _features(case, o, s):
    """The model's perception features: [s, blur, normalised state gradient, normalised density gradient]."""
    h, _ = _geometry(case)
    coef = h / float(np.float32(0.1))

    def normalise(v):
        return torch.log1p(v.norm(dim=-1, keepdim=True)) * torch.nn.functional.normalize(v, dim=-1)

    return torch.cat([s, o["blur"], normalise(o["hybrid"] * coef).flatten(1),
                      normalise(o["grad_rho"] * coef ** (1 + case["dim"]) / case["N"])], dim=1)


def _exact_step(case, d):
    B, N, C, D = case["B"], case["N"], case["C"], case["dim"]
    static, train = case["kind"] == "static", case["kind"] == "static" or case["train"]
    p = _perception(case, d)
    x, s, slots = p.x, p.s, _slots(_order(case, d["x"]))
    o = p.forward()
    names = ("blur", "hybrid", "grad_rho")
    leaves = {k: (o[k].requires_grad_(True) if k != "grad_rho" else o[k]) for k in names}
    s = s.requires_grad_(True)
    w1, b1, w2 = (d[k].double().requires_grad_(True) for k in ("w1", "b1", "w2"))
    mask = 1.0
    if case["update_prob"] < 1.0:
        torch.cuda.manual_seed(d["seed"])
        mask = (torch.rand(B, N, 1, device=DEVICE) < case["update_prob"]).double().flatten(0, 1)
    with torch.set_grad_enabled(train):
        y = torch.relu(_features(case, leaves, s) @ w1.T + b1) @ w2.T
        a, ds = (None, y) if static else (y[:, :D], y[:, D:])
        s_new, x_new = s + ds * mask, x
        if not static:
            dx = a * float(np.float32(_geometry(case)[0])) / (1 + a.norm(dim=1, keepdim=True))
            dx = torch.nn.functional.pad(dx, (0, x.shape[1] - D))
            x_new = x + dx * mask

    def rows(t, by=None):
        t = t.detach().reshape(B, N, -1)
        return t if by is None else _take(t, by)

    if not train:
        by = slots if case["trace"] else None
        out = dict(x=rows(x_new, by), s=rows(s_new, by))
        if case["trace"]:
            out.update(dx=rows(dx, by), ds=rows(ds, by))
        return out
    ends = [(s_new, d["up_s"].double().flatten(0, 1))]
    if not static:
        ends.append((x_new, d["up_x"].double().flatten(0, 1)))
    torch.autograd.backward([t for t, _ in ends], [u for _, u in ends])
    _, gs = p.backward(o["rho"], positions=False, up_blur=leaves["blur"].grad, up_grad=leaves["hybrid"].grad)
    out = dict(x=rows(x_new), s=rows(s_new))
    if not static:
        out["grad_x"] = _take(d["up_x"].double(), slots)
    out["grad_s"] = _take((s.grad + gs).reshape(B, N, C), slots)
    return dict(out, w1=w1.grad, b1=b1.grad, w2=w2.grad)


def _exact_mlp(case, d):
    z, w1, b1, w2 = (d[k].double().requires_grad_(True) for k in ("z", "w1", "b1", "w2"))
    y = torch.relu(z @ w1.T + b1) @ w2.T
    y.backward(d["up"].double())
    return dict(y=y.detach(), grad_z=z.grad, w1=w1.grad, b1=b1.grad, w2=w2.grad)


def _exact_splat(case, d):
    S, C, N = case["img"], case["C"], case["N"]
    scale = (S * case["pixel"] / 2.0) ** 2
    sigma = S * case["pixel"] / 2.0
    r = math.ceil(5 * sigma)
    off = torch.arange(-r, r + 1, device=DEVICE)
    images, gx, gc = [], [], []
    for b in range(case["B"]):
        x, c = (d[k][b].double().requires_grad_(True) for k in ("x", "color"))
        pos = (x + 1.0) / 2.0 * (S - 1)
        pos = torch.stack([pos[:, 0], (S - 1) - pos[:, 1]], dim=1)
        base = torch.floor(pos.detach())
        wx, wy = (torch.exp(-(off[None] - (pos - base)[:, k:k + 1]) ** 2 / (2 * sigma * sigma)) for k in (0, 1))
        w = wy[:, :, None] * wx[:, None, :]
        w = w / (1e-8 + w.sum((1, 2), keepdim=True)) * scale
        ix, iy = (base[:, k].long()[:, None] + off[None] for k in (0, 1))
        inside = ((iy >= 0) & (iy < S))[:, :, None] & ((ix >= 0) & (ix < S))[:, None, :]
        flat = (iy[:, :, None] * S + ix[:, None, :])[inside]
        row = torch.arange(N, device=DEVICE)[:, None, None].expand_as(inside)[inside]
        w = w[inside]
        val = torch.cat([w[:, None] * c[:, -3:].index_select(0, row), w[:, None]], 1)
        img = _sum(S * S, flat, val).reshape(S, S, 4)
        img.backward(d["up"][b].double())
        images.append(img.detach())
        gx.append(x.grad)
        gc.append(c.grad)
    return dict(image=torch.stack(images), grad_x=torch.stack(gx), grad_color=torch.stack(gc))


def _exact_binning(case, d):
    _, G = _geometry(case)
    B, N, cells = case["B"], case["N"], math.prod(G)
    order = _order(case, d["x"])
    slots = _slots(order)
    key = (_take(_cells(case, d["x"]), order) + cells * torch.arange(B, device=DEVICE)[:, None]).flatten()
    counts = torch.bincount(key, minlength=B * cells)
    offsets = torch.zeros(B * cells + 1, dtype=torch.int64, device=DEVICE)
    offsets[1:] = torch.cumsum(counts, 0)
    used = torch.nonzero(counts)[:, 0]
    blocks = (counts[used] + case["maxp"] - 1) // case["maxp"]
    cell = torch.repeat_interleave(used, blocks)
    nth = torch.arange(cell.numel(), device=DEVICE) - torch.repeat_interleave(torch.cumsum(blocks, 0) - blocks, blocks)
    info = torch.zeros(B * min(N, cells + (N + case["maxp"] - 1) // case["maxp"]), 4, dtype=torch.int32, device=DEVICE)
    info[:cell.numel()] = torch.stack([cell, nth * case["maxp"],
                                       torch.minimum(counts[cell] - nth * case["maxp"],
                                                     torch.full_like(cell, case["maxp"])), cell // cells], 1).int()
    return dict(permutation=slots.int(), bin_offsets=offsets.int(), block_info=info,
                total_blocks=torch.tensor([cell.numel()], dtype=torch.int32, device=DEVICE),
                x_bin=_take(d["x"], order), s_bin=_take(d["s"], order), x=d["x"], s=d["s"])


_EXACT = dict(step=_exact_step, static=_exact_step, ops=_exact_ops, fields=_exact_ops, mlp=_exact_mlp,
              splat=_exact_splat, binning=_exact_binning)
