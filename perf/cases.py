"""The work that programs have jaxpm_amd do, as cases that can be timed and compared.

Every case names a ``kind`` (what is called), a mesh and the options of the
call.  ``listed`` holds one case of each kind and size that matters, ``draw``
makes others of the same ranges, ``prepare`` builds what a program holds
before the call, ``run`` makes the call, ``work`` counts the bytes and
operations it cannot do without and ``exact`` repeats it in 64 bits with
plain torch and numpy.
"""
import math

import numpy as np
import torch

from jaxpm_amd import config, cosmology, diffsim, integrate, lensing, painting, pm, utils

OMEGA_C, OMEGA_B = 0.25, 0.05   # flat LCDM of the differentiable-simulation configuration
A_START = 0.1                   # a node of the tabulated growth functions


def listed():
    return [
        # the density of particles in no spatial order (a catalogue, a shuffled snapshot)
        dict(name="paint_random_256", kind="paint", nx=256, ny=256, nz=256, n=256 ** 3, order="random",
             weighted=False),
        # a field sampled at evolved particles, and its gradients, on a mesh of no convenient size
        dict(name="read_grad_ragged", kind="read", nx=250, ny=201, nz=180, n=250 * 201 * 180, order="lattice",
             grad=True),
        # one force evaluation of an ODE solver on displacements (paint_absolute_pos=False)
        dict(name="forces_relative_192", kind="forces", nx=192, ny=192, nz=192, absolute=False, grad=False,
             r_split=0.0, f64=False),
        # a force and its gradient with the long-range split, mesh axes of 5-smooth and odd lengths
        dict(name="forces_grad_odd", kind="forces", nx=100, ny=125, nz=90, absolute=True, grad=True, r_split=1.25,
             f64=False),
        # the float64 switch (jax_enable_x64) of the equivalence tests
        dict(name="forces_f64_128", kind="forces", nx=128, ny=128, nz=128, absolute=True, grad=False, r_split=0.0,
             f64=True),
        # initial conditions: Gaussian field and second-order LPT onto the lattice
        dict(name="lpt2_256", kind="lpt", nx=256, ny=256, nz=256, order=2, absolute=False),
        # the smallest simulation: 32^3, 10 leapfrog steps, no gradient
        dict(name="leapfrog_32", kind="leapfrog", nx=32, ny=32, nz=32, steps=10, absolute=True, grad=False,
             checkpoint=0),
        # the headline: 256^3 leapfrog, the final density and its adjoint, checkpoints every 5 steps
        dict(name="leapfrog_grad_256", kind="leapfrog", nx=256, ny=256, nz=256, steps=10, absolute=True, grad=True,
             checkpoint=5),
        # a differentiable simulation: noise and cosmology to the final density and back, 2LPT + leapfrog
        dict(name="model_grad_64", kind="model", nx=64, ny=64, nz=64, steps=10, order=2, absolute=True,
             checkpoint=4),
        # many simulations of three mesh sizes stepped together, forward and adjoint
        dict(name="batch_64_96_128", kind="batch", sizes="64x4 96x4 128x4", steps=20, checkpoint=5),
        # power spectrum multipoles of a density
        dict(name="spectrum_256", kind="spectrum", nx=256, ny=256, nz=256, multipoles="0 2 4", cross=False),
        # a smoothed lens plane of a slab of an evolved box, and its gradient
        dict(name="plane_grad_256", kind="plane", nx=256, ny=256, nz=256, res=1024, order="lattice", sigma=2.0,
             grad=True),
    ]


def _side(rng, side):
    """An axis length near ``side``: a power of two, 3 * 2^k, a 5-smooth or any length."""
    style = rng.randrange(4)
    if style == 0:
        return 2 ** max(3, round(math.log2(side)))
    if style == 1:
        return 3 * 2 ** max(1, round(math.log2(side / 3)))
    if style == 2:
        return 10 * max(1, round(side / 10))
    return max(9, round(side)) | 1


def _mesh(rng, lo, hi):
    """Mesh axes whose cells spread evenly in logarithm between about lo^3 and at most hi^3."""
    while True:
        side = lo * (hi / lo) ** rng.random()
        if rng.random() < 0.5:
            a = _side(rng, side)
            dims = (a, a, a)
        else:
            dims = tuple(_side(rng, side * rng.uniform(0.7, 1.4)) for _ in range(3))
        if dims[0] * dims[1] * dims[2] <= hi ** 3 and max(dims) <= 2 * hi:
            return dict(nx=dims[0], ny=dims[1], nz=dims[2])


def draw(rng):
    kind = rng.choice(["paint", "read", "forces", "forces", "lpt", "leapfrog", "leapfrog", "model", "batch",
                       "spectrum", "plane"])
    if kind in ("paint", "read"):
        m = _mesh(rng, 16, 250)
        cells = m["nx"] * m["ny"] * m["nz"]
        n = min(16_000_000, int(cells * rng.choice([0.5, 1.0, 1.7])))
        order = rng.choice(["random", "lattice"])
        c = dict(kind=kind, **m, n=cells if order == "lattice" else n, order=order)
        c.update({"weighted": rng.random() < 0.5} if kind == "paint" else {"grad": rng.random() < 0.5})
        return c
    if kind == "forces":
        f64 = rng.random() < 0.2
        return dict(kind=kind, **_mesh(rng, 16, 128 if f64 else 224), absolute=rng.random() < 0.5,
                    grad=not f64 and rng.random() < 0.5, r_split=rng.choice([0.0, rng.uniform(0.5, 2.0)]), f64=f64)
    if kind == "lpt":
        return dict(kind=kind, **_mesh(rng, 16, 240), order=rng.choice([1, 2]), absolute=rng.random() < 0.5)
    if kind == "leapfrog":
        grad = rng.random() < 0.5
        return dict(kind=kind, **_mesh(rng, 16, 200), steps=rng.randint(3, 12), absolute=rng.random() < 0.7,
                    grad=grad, checkpoint=rng.choice([0, 2, 5]))
    if kind == "model":
        return dict(kind=kind, **_mesh(rng, 16, 96), steps=rng.randint(3, 12), order=rng.choice([1, 2]),
                    absolute=rng.random() < 0.7, checkpoint=rng.choice([0, 4]))
    if kind == "batch":
        sizes = sorted(rng.sample([16, 24, 32, 40, 48, 64, 80, 96], rng.randint(1, 3)))
        return dict(kind=kind, sizes=" ".join(f"{s}x{rng.randint(1, 3)}" for s in sizes), steps=rng.randint(3, 12),
                    checkpoint=rng.choice([0, 4]))
    if kind == "spectrum":
        return dict(kind=kind, **_mesh(rng, 16, 240), multipoles=rng.choice(["0", "0 2", "0 2 4"]),
                    cross=rng.random() < 0.5)
    return dict(kind="plane", **_mesh(rng, 32, 240), res=rng.choice([128, 200, 512, 750, 1024]),
                order=rng.choice(["random", "lattice"]), sigma=rng.choice([0.0, rng.uniform(0.8, 3.0)]),
                grad=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs

def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _lattice(shape):
    return torch.stack(torch.meshgrid(*[torch.arange(s, device=_dev(), dtype=torch.float32) for s in shape],
                                      indexing="ij"), -1)


def _displacements(shape, rms, seed, waves=16):
    """A smooth, curl-free, periodic displacement field (nx, ny, nz, 3) of
    the given rms in cells: random plane waves from the box down to 8 cells."""
    r = np.random.default_rng(seed)
    dev = _dev()
    axes = [torch.arange(s, device=dev, dtype=torch.float32).reshape([s if d == e else 1 for e in range(3)])
            for d, s in enumerate(shape)]
    out = torch.zeros((*shape, 3), dtype=torch.float32, device=dev)
    for _ in range(waves):
        while True:
            m = [int(r.integers(-max(1, s // 8), max(1, s // 8) + 1)) if s > 1 else 0 for s in shape]
            if any(m):
                break
        k = [2 * math.pi * a / s for a, s in zip(m, shape)]
        kn = math.sqrt(sum(a * a for a in k))
        wave = torch.sin(axes[0] * k[0] + axes[1] * k[1] + axes[2] * k[2] + float(r.uniform(0, 2 * math.pi)))
        amp = float(r.normal()) / math.sqrt(kn)
        for d in range(3):
            if k[d]:
                out[..., d].add_(wave, alpha=amp * k[d] / kn)
    return out.mul_(rms * math.sqrt(3) / max(float(out.square().sum(-1).mean().sqrt()), 1e-9))


def _positions(case, seed, rms=3.0):
    """Particles of a snapshot, (n, 3) in grid units: in the order of the
    lattice they started from, or uniform in no order."""
    shape = _shape(case)
    if case["order"] == "random":
        u = torch.rand((case.get("n", shape[0] * shape[1] * shape[2]), 3), generator=_gen(seed), device=_dev())
        return u.mul_(torch.tensor(shape, dtype=torch.float32, device=_dev()))
    return (_lattice(shape) + _displacements(shape, rms, seed)).reshape(-1, 3)


def _randn(shape, seed):
    return torch.randn(shape, generator=_gen(seed), device=_dev())


def _cosmo():
    return cosmology.Cosmology(Omega_c=OMEGA_C, Omega_b=OMEGA_B, h=0.7, n_s=0.96, sigma8=0.8)


def _pk_table():
    """A linear power spectrum of the usual shape [(Mpc/h)^3]."""
    k = np.logspace(-4, 1, 128)
    return k, 2.0e4 * (k / 0.02) / (1.0 + (k / 0.02) ** 2) ** 1.3


def _box(case):
    return tuple(4.0 * s for s in _shape(case))


def _a_steps(case):
    return np.linspace(A_START, 1.0, case["steps"] + 1)


def _batch_shapes(case):
    out = []
    for part in case["sizes"].split():
        s, b = part.split("x")
        out += [(int(s),) * 3] * int(b)
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=dict(case))
    if kind == "batch":
        shapes = _batch_shapes(case)
        r = np.random.default_rng(seed)
        om, s8 = r.uniform(0.2, 0.35, len(shapes)), r.uniform(0.7, 0.9, len(shapes))
        cosmos = [cosmology.Cosmology(Omega_c=float(a), Omega_b=OMEGA_B, h=0.7, n_s=0.96, sigma8=float(b))
                  for a, b in zip(om, s8)]
        s["model"] = diffsim.BatchLptNBody(shapes, [tuple(4.0 * a for a in sh) for sh in shapes], _a_steps(case),
                                           cosmos, order=1, checkpoint_every=case["checkpoint"] or None, graph=True)
        s["noise"] = _randn((sum(a ** 3 for a, _, _ in shapes),), seed)
        return s
    shape = _shape(case)
    if kind == "paint":
        s["pos"] = _positions(case, seed)
        s["weight"] = 0.5 + torch.rand(case["n"], generator=_gen(seed + 1000), device=_dev()) \
            if case["weighted"] else 1.0
        s["mesh"] = torch.zeros(shape, device=_dev())
    elif kind == "read":
        s["pos"] = _positions(case, seed)
        s["mesh"] = _randn(shape, seed + 1000)
        s["cot"] = _randn((case["n"],), seed + 2000) if case["grad"] else None
    elif kind == "forces":
        x = _displacements(shape, 3.0, seed)
        if case["absolute"]:
            x = (_lattice(shape) + x).reshape(-1, 3)
        s["pos"] = x.double() if case["f64"] else x
        s["cot"] = _randn(tuple(x.shape), seed + 1000) if case["grad"] else None
        if case["f64"]:
            config.update("jax_enable_x64", True)
    elif kind == "lpt":
        s["noise"] = _randn(shape, seed)
        s["pk"] = pm.TabulatedPk(*_pk_table())
        s["cosmo"] = _cosmo()
        s["particles"] = _lattice(shape) if case["absolute"] else None
    elif kind == "leapfrog":
        dx = _displacements(shape, 0.4, seed)
        # the growing mode at a = 0.1: p = a^2 f E dx
        s["vel"] = (0.174 * dx).reshape(-1, 3)
        s["pos"] = ((_lattice(shape) + dx) if case["absolute"] else dx).reshape(-1, 3)
        s["target"] = 1.0 + 0.1 * _randn(shape, seed + 1000) if case["grad"] else None
        s["cosmo"] = _cosmo()
    elif kind == "model":
        s["model"] = diffsim.LptNBody(shape, _box(case), _a_steps(case), base_cosmo=_cosmo(), order=case["order"],
                                      paint_absolute_pos=case["absolute"], checkpoint_every=case["checkpoint"] or None)
        s["noise"] = _randn(shape, seed)
        s["target"] = 1.0 + 0.1 * _randn(shape, seed + 1000)
    elif kind == "spectrum":
        s["mesh"] = _randn(shape, seed)
        s["mesh2"] = s["mesh"] + 0.5 * _randn(shape, seed + 1000) if case["cross"] else None
    elif kind == "plane":
        s["pos"] = _positions(case, seed)
        s["cot"] = _randn((case["res"], case["res"]), seed + 1000) if case["grad"] else None
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return s


# ------------------------------------------------------------------- calls

def _leaf(t):
    return t.detach().requires_grad_(True)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "paint":
        return painting.cic_paint(state["mesh"], state["pos"], state["weight"])
    if kind == "read":
        if not case["grad"]:
            return painting.cic_read(state["mesh"], state["pos"])
        mesh, pos = _leaf(state["mesh"]), _leaf(state["pos"])
        vals = painting.cic_read(mesh, pos)
        gmesh, gpos = torch.autograd.grad(vals, (mesh, pos), state["cot"])
        return {"values": vals.detach(), "grad_mesh": gmesh, "grad_pos": gpos}
    if kind == "forces":
        if not case["grad"]:
            return pm.pm_forces(state["pos"], mesh_shape=_shape(case), r_split=case["r_split"],
                                paint_absolute_pos=case["absolute"])
        pos = _leaf(state["pos"])
        f = pm.pm_forces(pos, mesh_shape=_shape(case), r_split=case["r_split"], paint_absolute_pos=case["absolute"])
        (g,) = torch.autograd.grad(f, pos, state["cot"])
        return {"forces": f.detach(), "grad_pos": g}
    if kind == "lpt":
        ic = pm.linear_field(_shape(case), _box(case), state["pk"], state["noise"])
        dx, p, f = pm.lpt(state["cosmo"], ic, state["particles"], a=A_START, order=case["order"])
        return {"field": ic, "dx": dx, "p": p, "f": f}
    if kind == "leapfrog":
        args = dict(a_steps=_a_steps(case), cosmo=state["cosmo"], mesh_shape=_shape(case),
                    paint_absolute_pos=case["absolute"], checkpoint_every=case["checkpoint"] or None)
        if not case["grad"]:
            x, v = integrate.leapfrog(state["pos"], state["vel"], **args)
            return {"pos": x, "vel": v}
        x0, v0 = _leaf(state["pos"]), _leaf(state["vel"])
        x, v = integrate.leapfrog(x0, v0, **args)
        rho = _density(x, case)
        loss = ((rho - state["target"]) ** 2).sum()
        gx, gv = torch.autograd.grad(loss, (x0, v0))
        return {"density": rho.detach(), "pos": x.detach(), "vel": v.detach(), "grad_pos": gx, "grad_vel": gv}
    if kind == "model":
        noise = _leaf(state["noise"])
        params = state["model"].parameter_vector().float().requires_grad_(True)
        rho = state["model"](noise, params)
        loss = ((rho - state["target"]) ** 2).sum()
        gn, gp = torch.autograd.grad(loss, (noise, params))
        return {"density": rho.detach(), "grad_noise": gn, "grad_params": gp}
    if kind == "batch":
        noise = _leaf(state["noise"])
        rho = state["model"].forward_fixed_cosmology(noise)
        loss = ((rho - 1.0) ** 2).sum()
        (gn,) = torch.autograd.grad(loss, noise)
        return {"density": rho.detach(), "grad_noise": gn}
    if kind == "spectrum":
        k, p = utils.power_spectrum(state["mesh"], state["mesh2"], box_shape=np.array(_box(case)),
                                    kedges=_k_width(case), multipoles=_poles(case))
        return {"k": k, "p": p}
    pos = state["pos"]
    depth = case["nz"]
    args = (_shape(case), 0.4 * depth, 0.25 * depth, case["res"], case["sigma"] or None)
    if not case["grad"]:
        return lensing.density_plane(pos, *args)
    pos = _leaf(pos)
    plane = lensing.density_plane(pos, *args)
    (g,) = torch.autograd.grad(plane, pos, state["cot"])
    return {"plane": plane.detach(), "grad_pos": g}


def _density(x, case):
    if case["absolute"]:
        return painting.cic_paint(torch.zeros(_shape(case), device=x.device), x)
    return painting.cic_paint_dx(x.reshape(*_shape(case), 3))


def _poles(case):
    p = [int(v) for v in case["multipoles"].split()]
    return p[0] if len(p) == 1 else p


def _k_width(case):
    """Bins of 2.17 fundamental modes of the longest axis."""
    return float(2.17 * 2 * math.pi / (4.0 * max(_shape(case))))


# -------------------------------------------------------------------- work

def _fft_flops(m):
    return 2.5 * m * math.log2(max(m, 2))


def work(case):
    """Bytes and operations of one pass that the path cannot do without:
    inputs and outputs once; in a time loop, each step's positions and
    velocities in and out, and its mesh out and in around the transforms."""
    kind = case["kind"]
    if kind == "batch":
        shapes = _batch_shapes(case)
        ms = [a * b * c for a, b, c in shapes]
        m = sum(ms)
        evals = 2 * case["steps"] + 2
        return {"bytes": 8.0 * m + evals * 56.0 * m, "flops": evals * sum(2 * _fft_flops(a) + 150.0 * a for a in ms)}
    shape = _shape(case)
    m = shape[0] * shape[1] * shape[2]
    if kind == "paint":
        n = case["n"]
        return {"bytes": 12.0 * n + (4.0 * n if case["weighted"] else 0.0) + 8.0 * m, "flops": 40.0 * n}
    if kind == "read":
        n = case["n"]
        b = 16.0 * n + 4.0 * m
        return {"bytes": b + (16.0 * n + 4.0 * m if case["grad"] else 0.0), "flops": (120.0 if case["grad"] else 40.0) * n}
    if kind == "forces":
        w = 8.0 if case["f64"] else 4.0
        g = 2 if case["grad"] else 1
        return {"bytes": w * (6.0 * m + 2.0 * m) * g, "flops": g * (2 * _fft_flops(m) + 150.0 * m)}
    if kind == "lpt":
        return {"bytes": 4.0 * m + 4.0 * m + 36.0 * m + (12.0 * m if case["absolute"] else 0.0),
                "flops": (12 if case["order"] == 2 else 6) * _fft_flops(m) + 60.0 * m}
    if kind in ("leapfrog", "model"):
        grad = kind == "model" or case["grad"]
        evals = (case["steps"] + 1) * (2 if grad else 1)
        return {"bytes": evals * 56.0 * m + (8.0 * m if kind == "model" else 48.0 * m),
                "flops": evals * (2 * _fft_flops(m) + 150.0 * m)}
    if kind == "spectrum":
        f = 2 if case["cross"] else 1
        return {"bytes": 4.0 * m * f, "flops": f * _fft_flops(m) + 20.0 * m}
    n, p = m, case["res"] ** 2
    return {"bytes": 12.0 * n + 4.0 * p + (12.0 * n + 4.0 * p if case["grad"] else 0.0),
            "flops": 40.0 * 0.25 * n + (2 * _fft_flops(p) if case["sigma"] else 0.0)}


# ------------------------------------------------------------ 64-bit values

def _corners(pos, dims):
    """(flat index, weight) of the 2^d CIC corners of pos (n, d), float64."""
    f = torch.floor(pos.detach())
    frac = pos - f
    base = f.long()
    for o in range(2 ** len(dims)):
        idx, w = 0, 1.0
        for d, n in enumerate(dims):
            b = (o >> d) & 1
            idx = idx * n + torch.remainder(base[:, d] + b, n)
            w = w * (frac[:, d] if b else 1.0 - frac[:, d])
        yield idx, w


def _paint64(pos, dims, weight=None):
    out = torch.zeros(int(np.prod(dims)), dtype=torch.float64, device=pos.device)
    for idx, w in _corners(pos, dims):
        out = out.index_add(0, idx, w if weight is None else w * weight)
    return out.reshape(dims)


def _read64(mesh, pos):
    flat = mesh.reshape(-1)
    return sum(flat[idx] * w for idx, w in _corners(pos, mesh.shape))


def _fft(x):
    return torch.fft.rfftn(x.cpu())      # on the host: independent of the device's transforms


def _ifft(xk, shape, dev):
    return torch.fft.irfftn(xk, s=shape).to(dev)


def _k64(shape):
    return [(2 * math.pi * (torch.fft.rfftfreq if d == 2 else torch.fft.fftfreq)(s, dtype=torch.float64)).reshape(
        [-1 if d == e else 1 for e in range(3)]) for d, s in enumerate(shape)]


def _green64(shape, r_split=0.0):
    kk = sum(k * k for k in _k64(shape))
    kk[0, 0, 0] = 1.0
    g = -1.0 / kk
    g[0, 0, 0] = 0.0
    return g * torch.exp(-kk * r_split ** 2) if r_split else g


def _grad64(shape):
    """The 4-point difference i (8 sin w - sin 2w) / 6 of each axis."""
    return [1j * (8 * torch.sin(k) - torch.sin(2 * k)) / 6 for k in _k64(shape)]


def _fields64(field, r_split=0.0):
    """The three force meshes of a density."""
    shape = tuple(field.shape)
    pot = _fft(field) * _green64(shape, r_split)
    return [_ifft(-g * pot, shape, field.device) for g in _grad64(shape)]


def _forces64(pos, shape, r_split=0.0):
    return torch.stack([_read64(f, pos) for f in _fields64(_paint64(pos, shape), r_split)], -1)


def _growth64(a):
    """Coefficients of lpt at scale factor a: [D1, a^2 f1 E, a^2 E (a^3 E D1')'] and
    [3/7 D2, a^2 f2 E, a^2 E (a^3 E D2')'], from the growth equations integrated
    in ln a from the matter era (a = 1e-3)."""
    om = OMEGA_C + OMEGA_B

    def e2(x):
        return om * x ** -3 + 1.0 - om

    def rhs(lna, y):
        x = math.exp(lna)
        oma = om * x ** -3 / e2(x)
        q = (2.0 - 0.5 * (oma - 2.0 * (1.0 - oma))) / x
        r = 1.5 * oma / (x * x)
        d1, d2, v1, v2 = y
        return np.array([v1, v2, -q * v1 + r * d1, -q * v2 + r * d2 - r * d1 * d1]) * x

    y = np.array([1e-3, -3.0 / 7.0 * 1e-6, 1.0, -6.0 / 7.0 * 1e-3])
    t0, found = math.log(1e-3), None
    for t1 in (math.log(a), 0.0):
        h = (t1 - t0) / 6000
        for i in range(6000):
            t = t0 + i * h
            k1 = rhs(t, y)
            k2 = rhs(t + h / 2, y + h / 2 * k1)
            k3 = rhs(t + h / 2, y + h / 2 * k2)
            k4 = rhs(t + h, y + h * k3)
            y = y + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
        t0 = t1
        found = y if found is None else found
    d1, d2, v1, v2 = found
    n1, n2 = y[0], y[1]
    e = math.sqrt(e2(a))
    src = a ** 3 * e * 1.5 * om * a ** -3 / (e * e) / (a * a)
    first = [d1 / n1, a ** 2 * (v1 * a / d1) * e, a ** 2 * e * src * d1 / n1]
    second = [3 / 7 * d2 / n2, a ** 2 * (v2 * a / d2) * e, a ** 2 * e * src * (d2 - d1 * d1) / n2]
    return first, second


def _leapfrog64(x, v, case):
    om = OMEGA_C + OMEGA_B
    shape = _shape(case)
    a = _a_steps(case)

    def e(t):
        return math.sqrt(om * t ** -3 + 1.0 - om)

    lat = 0.0 if case["absolute"] else _lattice(shape).double().reshape(-1, 3)
    f = _forces64(lat + x, shape)
    for a0, a1 in zip(a[:-1], a[1:]):
        h, am = a1 - a0, 0.5 * (a0 + a1)
        v = v + 0.5 * h * 1.5 * om / (a0 ** 2 * e(a0)) * f
        x = x + h / (am ** 3 * e(am)) * v
        f = _forces64(lat + x, shape)
        v = v + 0.5 * h * 1.5 * om / (a1 ** 2 * e(a1)) * f
    return x, v


def _spectrum64(state):
    case = state["case"]
    shape = _shape(case)
    box = np.array(_box(case))
    width = _k_width(case)
    edges = np.arange(width, np.pi * np.min(np.array(shape) / box), width) + width / 2
    m = shape[0] * shape[1] * shape[2]
    k = [np.fft.fftfreq(s) * (2 * np.pi * s / b) if d < 2 else np.fft.rfftfreq(s) * (2 * np.pi * s / b)
         for d, (s, b) in enumerate(zip(shape, box))]
    kn = np.sqrt((k[0] ** 2)[:, None, None] + (k[1] ** 2)[None, :, None] + (k[2] ** 2)[None, None, :])
    kn = kn.astype(np.float32)       # modes are binned by their float32 wave number
    which = np.digitize(kn.reshape(-1), edges)
    both = np.where((np.arange(shape[2] // 2 + 1) == 0) | (2 * np.arange(shape[2] // 2 + 1) == shape[2]), 1.0, 2.0)
    w = np.broadcast_to(both, kn.shape).reshape(-1)
    count = np.bincount(which, w, len(edges) + 1)
    ksum = np.bincount(which, w * kn.reshape(-1), len(edges) + 1)
    f1 = _fft(state["mesh"].double()).numpy()
    f2 = _fft(state["mesh2"].double()).numpy() if case["cross"] else f1
    p = f1 * np.conj(f2)
    with np.errstate(divide="ignore", invalid="ignore"):
        mu = np.where(kn > 0, np.abs(k[2])[None, None, :] / kn, 0.0)
        out = []
        for ell in np.atleast_1d(_poles(case)):
            leg = np.polynomial.legendre.legval(mu, [0] * int(ell) + [2 * int(ell) + 1])
            v = (leg * p).reshape(-1)
            re = np.bincount(which, w * v.real, len(edges) + 1)
            # a mode and its mirror are conjugates: imaginary parts cancel
            tot = np.abs(re) if case["cross"] else re
            out.append((tot / count)[1:-1] / m * (box / np.array(shape)).prod())
        kavg = (ksum / count)[1:-1]
    out = np.stack(out)
    return {"k": kavg, "p": out[0] if np.ndim(_poles(case)) == 0 else out}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("model", "batch"):
        return None
    m = case["nx"] * case["ny"] * case["nz"]
    if kind == "leapfrog" and m * (case["steps"] + 1) * (3 if case["grad"] else 1) > 6e7:
        return None
    state = prepare(case, seed)
    shape = _shape(case)
    if kind == "spectrum":
        return _spectrum64(state)
    if kind == "paint":
        w = state["weight"].double() if case["weighted"] else None
        return _paint64(state["pos"].double(), shape, w)
    if kind == "read":
        pos, mesh = state["pos"].double(), state["mesh"].double()
        if not case["grad"]:
            return _read64(mesh, pos)
        pos, mesh = _leaf(pos), _leaf(mesh)
        vals = _read64(mesh, pos)
        gm, gp = torch.autograd.grad(vals, (mesh, pos), state["cot"].double())
        return {"values": vals.detach(), "grad_mesh": gm, "grad_pos": gp}
    if kind == "forces":
        x = _leaf(state["pos"].double())
        lat = 0.0 if case["absolute"] else _lattice(shape).double()
        with torch.set_grad_enabled(case["grad"]):
            f = _forces64((lat + x).reshape(-1, 3), shape, case["r_split"]).reshape(x.shape)
        if not case["grad"]:
            return f.detach()
        (g,) = torch.autograd.grad(f, x, state["cot"].double())
        return {"forces": f.detach(), "grad_pos": g}
    if kind == "lpt":
        k, pk = (np.asarray(v, np.float32).astype(np.float64) for v in _pk_table())
        kn = torch.sqrt(sum((kv / 4.0) ** 2 for kv in _k64(shape))).numpy()
        mult = np.sqrt(np.interp(kn, k, pk) * m / np.prod(_box(case)))
        ic = _ifft(_fft(state["noise"].double()) * torch.as_tensor(mult), shape, _dev())
        first, second = _growth64(A_START)
        psi = torch.stack(_fields64(ic), -1)
        dx = first[0] * psi
        p, f = first[1] * dx, first[2] * psi
        if case["order"] == 2:
            pot = _fft(ic) * _green64(shape)
            g = _grad64(shape)
            d = {(a, b): _ifft(g[a] * g[b] * pot, shape, _dev()) for a in range(3) for b in range(a, 3)}
            src = d[0, 0] * d[1, 1] + d[1, 1] * d[2, 2] + d[2, 2] * d[0, 0] - d[0, 1] ** 2 - d[0, 2] ** 2 - d[1, 2] ** 2
            psi2 = torch.stack(_fields64(src), -1)
            dx2 = second[0] * psi2
            dx, p, f = dx + dx2, p + second[1] * dx2, f + second[2] * psi2
        return {"field": ic, "dx": dx, "p": p, "f": f}
    if kind == "leapfrog":
        x0, v0 = _leaf(state["pos"].double()), _leaf(state["vel"].double())
        with torch.set_grad_enabled(case["grad"]):
            x, v = _leapfrog64(x0, v0, case)
        if not case["grad"]:
            return {"pos": x.detach(), "vel": v.detach()}
        lat = 0.0 if case["absolute"] else _lattice(shape).double().reshape(-1, 3)
        rho = _paint64(lat + x, shape)
        loss = ((rho - state["target"].double()) ** 2).sum()
        gx, gv = torch.autograd.grad(loss, (x0, v0))
        return {"density": rho.detach(), "pos": x.detach(), "vel": v.detach(), "grad_pos": gx, "grad_vel": gv}
    pos = _leaf(state["pos"].double())
    nx, res, depth = float(shape[0]), case["res"], case["nz"]
    z = state["pos"][:, 2]
    lo, hi = (np.float32(0.4 * depth + s * 0.125 * depth) for s in (-1.0, 1.0))
    inside = (z > float(lo)) & (z <= float(hi))
    with torch.set_grad_enabled(case["grad"]):
        xy = torch.remainder(pos[inside][:, :2], nx) / nx * res
        plane = _paint64(xy, (res, res)) / ((nx / res) * (float(shape[1]) / res) * (0.25 * depth))
        if case["sigma"]:
            k2 = torch.fft.fftfreq(res, dtype=torch.float64)[:, None] ** 2 + \
                torch.fft.rfftfreq(res, dtype=torch.float64)[None, :] ** 2
            filt = torch.exp(-k2 * (2 * math.pi * case["sigma"]) ** 2 / 2)
            plane = torch.fft.irfft2(torch.fft.rfft2(plane.cpu()) * filt, s=(res, res)).to(pos.device)
    if not case["grad"]:
        return plane.detach()
    (g,) = torch.autograd.grad(plane, pos, state["cot"].double())
    return {"plane": plane.detach(), "grad_pos": g}
