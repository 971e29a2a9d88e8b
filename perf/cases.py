"""What a user of this package has it do, as measurable cases.

Four kinds of work over the range that the package's own scenes, workloads and benchmark cover:

* whole runs of a world (`run`): a scene uploaded, stepped, and its state read back, as the headless driver and the
  benchmark do it: the full hydro + gravity + diffusion step under both stopping rules, the gas and gravity alone, the
  burning gas with the cold pressure; and a batch of worlds stepped together (`batch`);
* the gravity field of a given surface density (`gravity`);
* the diffusion system on its own: one multigrid preconditioner application (`precond`), the stiff solve (`solve`);
* the learned preconditioner's network: one application (`apply`), one training step (`train`).

`exact` restates each in plain torch in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
NS = 10
# per species H He C O Ne Mg Si S Fe n: (Z + 1) / A and Z / A
IMU = [2.0, 3 / 4, 7 / 12, 9 / 16, 11 / 20, 13 / 24, 15 / 28, 17 / 32, 27 / 56, 1.0]
ZA = [1.0, 0.5, 0.5, 0.5, 0.5, 0.5, 0.5, 0.5, 26 / 56, 0.0]
ASHES = [0.05, 0.35, 0.2, 0.2, 0.08, 0.04, 0.04, 0.02, 0.02, 0.0]


def listed():
    return [
        # the smallest full step that the tests and the smoke run use: launches and host decisions are all there is
        dict(name="run_64", kind="run", scene="turbulent", w=64, h=64, steps=10),
        # the plain-method workload: a self-gravitating blob, dumped every few steps
        dict(name="run_blob_256", kind="run", scene="blob", w=256, h=256, steps=10),
        # a disk in vacuum on a ragged world between walls, under the reference's own constants and stopping rule
        dict(name="run_disk_360x232", kind="run", scene="disk", w=360, h=232, steps=10),
        # the benchmark's headline: the turbulent 1024^2 full step
        dict(name="run_1024", kind="run", scene="turbulent", w=1024, h=1024, steps=10),
        # gas and gravity without the heat pass, the largest world the default FFT cap takes
        dict(name="run_gas_2048", kind="run", scene="gas", w=2048, h=2048, steps=40),
        # burning with the cold pressure on, stepped with the gas and its gravity
        dict(name="run_burn_512", kind="run", scene="burn", w=512, h=512, steps=20),
        # a batch of uneven scenes stepped together over host threads
        dict(name="batch_8", kind="batch", count=8, lo=64, hi=512, steps=4, threads=8),
        # the gravity field of one surface density, odd sides (an analysis of a dump)
        dict(name="gravity_601x433", kind="gravity", w=601, h=433),
        # one V-cycle on a ragged system with cells off the gas
        dict(name="precond_500x300", kind="precond", w=500, h=300, holes=True),
        # the benchmark's stiff diffusion solve
        dict(name="solve_2048", kind="solve", w=2048, h=2048, holes=False),
        # one application of the trained network at the benchmark's size
        dict(name="apply_2048", kind="apply", w=2048, h=2048),
        # one training step at the larger training size
        dict(name="train_512", kind="train", w=512, h=512),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def sides(lo, hi, step, cells):
        while True:
            w = max(lo, int(log(lo, hi + step)) // step * step)
            h = max(lo, int(w * log(0.5, 2.0)) // step * step)
            if w <= hi and h <= hi and w * h <= cells:
                return dict(w=w, h=h)

    kind = rng.choice(["turbulent", "blob", "disk", "gas", "burn", "batch", "gravity", "precond", "solve", "apply",
                       "train"])
    if kind in ("turbulent", "blob", "disk"):
        return dict(kind="run", scene=kind, steps=rng.randint(4, 10), **sides(64, 1024, 8, 700 * 700))
    if kind == "gas":
        return dict(kind="run", scene=kind, steps=rng.randint(10, 40), **sides(64, 2048, 8, 1400 * 1400))
    if kind == "burn":
        return dict(kind="run", scene=kind, steps=rng.randint(5, 20), **sides(64, 512, 8, 512 * 512))
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(3, 8), lo=8 * rng.randint(8, 16), hi=8 * rng.randint(20, 60),
                    steps=rng.randint(2, 4), threads=rng.choice([2, 4, 8]))
    if kind == "gravity":
        return dict(kind=kind, **sides(16, 2048, 1, 2048 * 2048))
    if kind in ("precond", "solve"):
        return dict(kind=kind, holes=rng.random() < 0.5, **sides(32, 2048, 1, 1500 * 1500))
    if kind == "apply":
        return dict(kind=kind, **sides(64, 2048, 4, 1800 * 1800))
    return dict(kind=kind, **sides(64, 512, 4, 512 * 512))


# ---------------------------------------------------------------------------------------------------------- inputs


def generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def smooth(gen, h, w):
    """A zero-mean unit-variance Gaussian field with P(k) ~ k^-3, as the workloads' lognormal fields have it."""
    f = torch.fft.rfft2(torch.randn((h, w), generator=gen, device=DEV, dtype=F64))
    ky = torch.fft.fftfreq(h, 1.0 / h, device=DEV, dtype=F64)[:, None] * (max(w, h) / h)
    kx = torch.fft.rfftfreq(w, 1.0 / w, device=DEV, dtype=F64)[None, :] * (max(w, h) / w)
    k = torch.sqrt(kx * kx + ky * ky)
    g = torch.fft.irfft2(torch.where(k >= 1.0, f * k.clamp(min=1.0) ** -1.5, 0.0 * f), s=(h, w))
    g = g - g.mean()
    return g / g.std()


def lognormal(gen, h, w, sigma):
    return torch.exp(sigma * smooth(gen, h, w) - 0.5 * sigma * sigma)


def box_physics(n, **more):
    """A unit box of ideal gas, gamma 5/3, Kramers opacity, open edges (the workloads')."""
    return dict(gamma=5 / 3, G=1.0, dx=1.0 / n, mu=1.0, opacity=1, kappa0=1.0, edge=1, max_padded=4096, **more)


# the benchmark's heat pass: multigrid PCG in inexact Newton, the last pass to 1e-8
INEXACT = dict(stop=1, solve_tol=1e-8, newton_heat=1e-6, newton_cell=1e-3, forcing=0.1, coarse_scale=1.2)
COLD = dict(k1e=21.3, k2e=134.0, k1n=2.67, k2n=58.2)


def scene(kind, w, h, seed):
    """(planes (14, h, w) f32 on the host, physics keywords, heat settings or None, whether it burns)"""
    gen = generator(seed)
    n = max(w, h)
    p = torch.zeros((14, h, w), device=DEV, dtype=F64)
    uv = [torch.zeros((h, w), device=DEV, dtype=F64)] * 2
    x = (torch.arange(w, device=DEV, dtype=F64) + 0.5 - 0.5 * w) / n
    y = (torch.arange(h, device=DEV, dtype=F64) + 0.5 - 0.5 * h) / n
    r2 = x[None, :] ** 2 + y[:, None] ** 2
    phys, heat, burns = box_physics(n), INEXACT, False
    p[4] = 1.0
    cold = 0.0
    if kind == "blob":
        rho = 1e-2 + torch.exp(-r2 / (2 * 0.1 ** 2))
        t = 1.0 + 0.01 * (2.0 * torch.rand((h, w), generator=gen, device=DEV, dtype=F64) - 1.0)
    elif kind in ("turbulent", "gas"):
        rho, t = lognormal(gen, h, w, 1.0), lognormal(gen, h, w, 0.5)
        uv = [smooth(gen, h, w), smooth(gen, h, w)]
        mach = torch.sqrt(((uv[0] ** 2 + uv[1] ** 2) / (phys["gamma"] * t)).mean())
        uv = [v * (0.5 / mach) for v in uv]
        if kind == "gas":
            heat = None
    elif kind == "disk":
        # the reference's constants (gamma 2, unit cells, its opacity), walls, a disk over vacuum
        a = 0.4 * min(w, h) / n
        inside = r2 < a * a
        rho = torch.where(inside, torch.sqrt((1.0 - r2 / (a * a)).clamp(min=0.0)).clamp(min=0.02), 1e-8)
        t = torch.where(inside, 30.0 * lognormal(gen, h, w, 0.2), 0.05)
        phys, heat = dict(edge=0), dict()
        p[4], p[5] = 0.75, 0.25
    else:
        # burning: fresh and burnt gas mixed, dense and hot enough for every record
        rho, t = 30.0 * lognormal(gen, h, w, 0.3), 100.0 * lognormal(gen, h, w, 0.3)
        mix = 0.5 * (1.0 + torch.tanh(smooth(gen, h, w)))
        ash, fresh = (torch.tensor(v, device=DEV, dtype=F64)[:, None, None] for v in (ASHES, [0.75, 0.25] + [0.0] * 8))
        p[4:] = mix * ash + (1.0 - mix) * fresh
        phys, heat, burns = dict(COLD), None, True
        cold = Cold(COLD).eps(rho, dot(p[4:], ZA), p[13])
    gamma = phys.get("gamma", 2.0)
    imu = 1.0 / phys["mu"] if phys.get("mu", 0.0) > 0.0 else dot(p[4:], IMU)
    p[0], p[1], p[2] = rho, rho * uv[0], rho * uv[1]
    p[3] = rho * (t * imu / (gamma - 1.0) + cold) + 0.5 * rho * (uv[0] ** 2 + uv[1] ** 2)
    return p.float().cpu().numpy(), phys, heat, burns


def world(kind, w, h, seed):
    import sandbox_reactions_amd as sr
    from sandbox_reactions_amd import react
    planes, phys, heat, burns = scene(kind, w, h, seed)
    wd = sr.World(w, h, physics=sr.physics(**phys), gravity=True, hydro=True, heat=heat is not None,
                  heat_settings=sr.heat_settings(**(heat or {})))
    if burns:
        wd.set_reactions(react.params(overrides={"burn_k": 10.0}))
    wd.upload(planes)  # the world's plans settle on its first step
    wd.run(1)
    return wd, planes


def system(w, h, holes, seed):
    """The stiff diffusion system of a lognormal field (Kramers opacity, the limiter on the faces, diffusion number
    1e3), with `holes` a tenth of the cells off the gas: (own, kx, ky, gas or None, right-hand side in f64)."""
    gen = generator(seed)
    n = max(w, h)
    rho, t = lognormal(gen, h, w, 1.5), lognormal(gen, h, w, 0.8)
    ks, er = rho * rho * t ** -3.5, 6.25e-7 * t ** 4

    def face(ea, eb, ka, kb):
        fe, k = 0.5 * (ea + eb), 0.5 * (ka + kb)
        r = (eb - ea).abs() * n / (k * fe)
        return 12800.0 * (2.0 + r) / (6.0 + 3.0 * r + r * r) / k * n * n

    kx = torch.zeros((h, w + 1), device=DEV, dtype=F64)
    ky = torch.zeros((h + 1, w), device=DEV, dtype=F64)
    kx[:, 1:-1] = face(er[:, :-1], er[:, 1:], ks[:, :-1], ks[:, 1:])
    ky[1:-1] = face(er[:-1], er[1:], ks[:-1], ks[1:])
    total = kx[:, :-1] + kx[:, 1:] + ky[:-1] + ky[1:]
    own = 1.5 * rho / (4.0 * 6.25e-7 * t ** 3)
    own = own / (1e3 / (total / own).median())
    b = own * er * (0.9 + 0.2 * torch.rand((h, w), generator=gen, device=DEV, dtype=F64))
    gas = None
    if holes:
        on = smooth(gen, h, w) < 1.3
        side = torch.nn.functional.pad(on, (1, 1, 1, 1))
        left, right, up, down = side[1:-1, :-2], side[1:-1, 2:], side[:-2, 1:-1], side[2:, 1:-1]
        # a face onto a cell off the gas is folded into the gas cell's own term
        own = own + (kx[:, :-1] * ~left + kx[:, 1:] * ~right + ky[:-1] * ~up + ky[1:] * ~down)
        own, b = torch.where(on, own, 1.0), torch.where(on, b, 0.0)
        kx[:, 1:-1] *= on[:, :-1] & on[:, 1:]
        ky[1:-1] *= on[:-1] & on[1:]
        gas = on.to(torch.uint8).contiguous()
    return own.float().contiguous(), kx.float().contiguous(), ky.float().contiguous(), gas, b.contiguous()


def diagonal(own, kx, ky):
    return own + kx[:, :-1] + kx[:, 1:] + ky[:-1] + ky[1:]


def batch_sides(case):
    k = case["count"] - 1
    return [max(8, int(case["lo"] * (case["hi"] / case["lo"]) ** (i / k)) // 8 * 8) for i in range(k + 1)]


def prepare(case, seed):
    import sandbox_reactions_amd as sr
    from sandbox_reactions_amd import train
    kind = case["kind"]
    if kind == "run":
        wd, planes = world(case["scene"], case["w"], case["h"], seed)
        return dict(kind=kind, world=wd, planes=planes, steps=case["steps"])
    if kind == "batch":
        ws = [world("blob" if i % 2 else "turbulent", s, s, seed + 101 * i) for i, s in enumerate(batch_sides(case))]
        return dict(kind=kind, worlds=[a for a, _ in ws], planes=[b for _, b in ws], steps=case["steps"],
                    threads=case["threads"])
    w, h = case["w"], case["h"]
    if kind == "gravity":
        return dict(kind=kind, plan=sr.Gravity(w, h, dx=1.0 / max(w, h)),
                    sigma=lognormal(generator(seed), h, w, 1.0).float().contiguous())
    own, kx, ky, gas, b = system(w, h, case.get("holes", False), seed)
    s = dict(kind=kind, own=own, kx=kx, ky=ky)
    if kind in ("precond", "solve"):
        s["solver"] = sr.Fld(w, h, coarse_scale=1.2)
        s["solver"].set_system(own, kx, ky, gas)
        s["b"] = b if kind == "solve" else (b / b.std()).float().contiguous()
        s["x"] = torch.zeros_like(s["b"])
        return s
    s["net"] = sr.Net(w, h, train.load())
    s["r"], s["e"] = pair(own, kx, ky, seed)
    s["z"] = torch.empty_like(s["r"])
    return s


def pair(own, kx, ky, seed):
    """(r, e) with A e = r: a rough error and its residual, the network's input and target."""
    gen = generator(seed + 7)
    d = diagonal(own.double(), kx.double(), ky.double())
    h, w = own.shape
    e = (smooth(gen, h, w) + 0.3 * torch.randn((h, w), generator=gen, device=DEV, dtype=F64)) / d.sqrt()
    e = e.float()
    return matvec(own.double(), kx.double(), ky.double(), e.double()).float().contiguous(), e.contiguous()


def run(s):
    import sandbox_reactions_amd as sr
    kind = s["kind"]
    if kind == "run":
        s["world"].upload(s["planes"])
        s["world"].run(s["steps"])
        p = s["world"].readback()
        return dict(sigma=p[0], momentum=p[1:3], energy=p[3], x=p[4:])
    if kind == "batch":
        for wd, planes in zip(s["worlds"], s["planes"]):
            wd.upload(planes)
        sr.ensemble_run(s["worlds"], s["steps"], s["threads"])
        got = [wd.readback() for wd in s["worlds"]]
        return [dict(sigma=p[0], momentum=p[1:3], energy=p[3], x=p[4:]) for p in got]
    if kind == "gravity":
        return s["plan"].field(s["sigma"])
    if kind == "precond":
        s["solver"].apply_precond(s["b"], s["x"])
        return s["x"]
    if kind == "solve":
        s["x"].zero_()
        s["solver"].solve(s["b"], s["x"], tol=1e-8)
        return s["x"]
    if kind == "apply":
        s["net"].apply(s["own"], s["kx"], s["ky"], s["r"], s["z"])
        return s["z"]
    loss = s["net"].loss_grad(s["own"], s["kx"], s["ky"], s["r"], s["e"])
    grads = s["net"].grads()
    s["net"].adam(1e-4)
    return dict(loss=loss, grads=grads, params=s["net"].params())


def work(case):
    """Bytes: every input and output once, and for a run the state (60 B a cell) read and written once a step; for an
    iterative solve its system, right-hand side and answer once. Flops: the transforms, the convolutions; for a step
    about 1000 a cell, with the heat pass about 50 multigrid iterations of 100 more."""
    kind = case["kind"]
    if kind == "run":
        n = case["w"] * case["h"]
        per = 1000 + (5000 if case["scene"] in ("turbulent", "blob", "disk") else 0)
        return dict(bytes=n * (112 + 120 * case["steps"]), flops=n * per * case["steps"])
    if kind == "batch":
        n = sum(s * s for s in batch_sides(case))
        return dict(bytes=n * (112 + 120 * case["steps"]), flops=6000 * n * case["steps"])
    n = case["w"] * case["h"]
    if kind == "gravity":
        p = 4 * n
        return dict(bytes=16 * n, flops=2 * 2.5 * p * math.log2(p))
    if kind == "precond":
        return dict(bytes=20 * n, flops=100 * n)
    if kind == "solve":
        return dict(bytes=28 * n, flops=140 * 130 * n)
    mac = sum(9 * ci * co * f for ci, co, f in ((3, 16, 1), (16, 16, 1), (16, 32, .25), (32, 32, .25), (32, 64, 1 / 16),
                                                (64, 64, 1 / 16), (96, 32, .25), (32, 32, .25), (48, 16, 1),
                                                (16, 16, 1))) + 16
    if kind == "apply":
        return dict(bytes=20 * n, flops=2 * mac * n)
    return dict(bytes=20 * n, flops=6 * mac * n)


def tolerance(case):
    """About four times the largest difference from `exact` that is measured over the ranges; for the network, whose
    difference from it is its 16-bit activations', what a few of them rounded the other way would show."""
    kind = case["kind"]
    if kind == "run" and case["scene"] == "burn":  # rates as T^40 on a 32-bit energy: 4e-5 (momentum), 1e-2
        return dict(rel=1.6e-4, max=4e-2)
    if kind in ("run", "batch"):  # the disk's momentum, 7.3e-6 and 4.6e-4 at its edge
        return dict(rel=3e-5, max=2e-3)
    if kind == "gravity":  # differences of a 32-bit potential: 1.7e-5, 8.6e-5
        return dict(rel=7e-5, max=4e-4)
    if kind == "precond":  # 2.5e-7, 1e-6
        return dict(rel=1e-6, max=4e-6)
    if kind == "solve":  # the stopping rule's 1e-8 of the right-hand side leaves 2.3e-10, 9.4e-9
        return dict(rel=2e-9, max=1e-7)
    return dict(rel=1e-2, max=0.2)


# ------------------------------------------------------------------------------------------------- exact, in 64 bits


def exact(case, seed):
    kind = case["kind"]
    if kind == "run":
        most = dict(turbulent=11_000_000, blob=900_000, disk=900_000).get(case["scene"], 200_000_000)
        if case["w"] * case["h"] * case["steps"] > most:
            return None  # its diffusion solves by plain conjugate gradients would take minutes
        planes, phys, hs, burns = scene(case["scene"], case["w"], case["h"], seed)
        p = Exact(planes, phys, hs is not None, burns).run(case["steps"])
        return dict(sigma=p[0], momentum=p[1:3], energy=p[3], x=p[4:])
    if kind == "batch":
        return None  # each of its worlds is a `run`
    w, h = case["w"], case["h"]
    if kind == "gravity":
        sigma = lognormal(generator(seed), h, w, 1.0).float().double()
        phi = potential(sigma, 1.0, 1.0 / max(w, h), 1e-6)
        gx, gy = gradient(phi, 1.0 / max(w, h))
        return phi, gx, gy
    own, kx, ky, gas, b = system(w, h, case.get("holes", False), seed)
    a = [v.double() for v in (own, kx, ky)]
    if kind == "solve":
        return conjugate_gradients(*a, b, torch.zeros_like(b), 1e-11)
    if kind == "precond":
        return vcycle(a, gas, (b / b.std()).float().double(), 1.2)
    from sandbox_reactions_amd import train
    flat = torch.tensor(train.load(), device=DEV, dtype=F64, requires_grad=kind == "train")
    r, e = (v.double() for v in pair(own, kx, ky, seed))
    with torch.set_grad_enabled(kind == "train"):
        z = network(flat, *a, r)
    if kind == "apply":
        return z
    err = z - e
    loss = (err * matvec(*a, err)).sum() / (e * matvec(*a, e)).sum()
    loss.backward()
    return dict(loss=float(loss.detach()), grads=flat.grad.clone(), params=None)


def dot(x, weights):
    return sum(w * x[i] for i, w in enumerate(weights))


def matvec(own, kx, ky, v):
    out = own * v
    dx, dy = kx[:, 1:-1] * (v[:, 1:] - v[:, :-1]), ky[1:-1] * (v[1:] - v[:-1])
    out[:, :-1] -= dx
    out[:, 1:] += dx
    out[:-1] -= dy
    out[1:] += dy
    return out


def conjugate_gradients(own, kx, ky, b, x, tol):
    d = diagonal(own, kx, ky)
    x = x.clone()
    r = b - matvec(own, kx, ky, x)
    goal = tol * b.norm()
    z = r / d
    p, rz = z.clone(), (r * z).sum()
    for it in range(100_000):
        if it % 50 == 0 and r.norm() <= goal:
            break
        q = matvec(own, kx, ky, p)
        alpha = rz / (p * q).sum()
        x += alpha * p
        r -= alpha * q
        z = r / d
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x


def vcycle(a, gas, r, omega):
    """V(2,2): red-black Gauss-Seidel, red first down and black first up, Galerkin 2x2 aggregation, the correction scaled
    by omega, the coarsest (at most 16 cells) solved exactly."""
    own, kx, ky = a
    h, w = own.shape
    if h * w <= 16:
        m = torch.stack([matvec(own, kx, ky, e.reshape(h, w)).reshape(-1) for e in torch.eye(h * w, device=DEV, dtype=F64)])
        return torch.linalg.solve(m, r.reshape(-1)).reshape(h, w)
    d = diagonal(own, kx, ky)
    colour = (torch.arange(h, device=DEV)[:, None] + torch.arange(w, device=DEV)[None, :]) % 2

    def sweep(z, c):
        return torch.where(colour == c, z + (r - matvec(own, kx, ky, z)) / d, z)

    def sums(v):  # over the 2x2 aggregates
        v = torch.nn.functional.pad(v, (0, w % 2, 0, h % 2))
        return v[::2, ::2] + v[1::2, ::2] + v[::2, 1::2] + v[1::2, 1::2]

    z = torch.zeros_like(r)
    for c in (0, 1, 0, 1):
        z = sweep(z, c)
    hc, wc = (h + 1) // 2, (w + 1) // 2
    oc = sums(own if gas is None else own * gas)
    kxc, kyc = torch.zeros((hc, wc + 1), device=DEV, dtype=F64), torch.zeros((hc + 1, wc), device=DEV, dtype=F64)
    fx = torch.nn.functional.pad(kx[:, 2:w:2], (0, 0, 0, h % 2))
    fy = torch.nn.functional.pad(ky[2:h:2], (0, w % 2))
    kxc[:, 1:wc], kyc[1:hc] = fx[::2] + fx[1::2], fy[:, ::2] + fy[:, 1::2]
    c = vcycle([torch.where(oc == 0.0, 1.0, oc), kxc, kyc], None, sums(r - matvec(own, kx, ky, z)), omega)
    z = z + omega * c.repeat_interleave(2, 0).repeat_interleave(2, 1)[:h, :w]
    for c in (1, 0, 1, 0):
        z = sweep(z, c)
    return z


def network(flat, own, kx, ky, r):
    """The U-Net (16, 32, 64 channels, 3x3 convolutions) on the scaled residual, the log coupling and the diagonal's
    share, its output scaled back: 64-bit sums over its 16-bit weights and activations."""
    from sandbox_reactions_amd.net import LAYERS
    import torch.nn.functional as nf
    def half(v):  # rounded as stored, its gradient passed through
        return v + (v.detach().bfloat16().double() - v.detach())

    p, o = {}, 0
    for name, ci, co in LAYERS:
        p[name] = (half(flat[o:o + 9 * ci * co]).reshape(3, 3, ci, co).permute(3, 2, 0, 1), flat[o + 9 * ci * co:][:co])
        o += 9 * ci * co + co
    d = diagonal(own, kx, ky)
    ks = (d - own).clamp(min=4e-30)
    rt = r / d.sqrt()
    s = rt.square().mean().sqrt()
    lk = torch.log(0.25 * ks)
    x = half(torch.stack([rt / s, (lk - lk.mean()).clamp(-20.0, 20.0), torch.log(own / d)])[None])

    def conv(name, v):  # a plain sum over the nine taps: 64-bit convolutions have no fast library path
        wt, b = p[name]
        hh, ww = v.shape[2:]
        vp = nf.pad(v, (1, 1, 1, 1))[0]
        out = b[:, None]
        for i in range(3):
            for j in range(3):
                out = out + wt[:, :, i, j] @ vp[:, i:i + hh, j:j + ww].reshape(v.shape[1], -1)
        return half(nf.relu(out)).reshape(1, -1, hh, ww)

    def up(v):
        return v.repeat_interleave(2, 2).repeat_interleave(2, 3)

    def pool(v):
        n, c, hh, ww = v.shape
        return half(v.reshape(n, c, hh // 2, 2, ww // 2, 2).mean(dim=(3, 5)))

    e1 = conv("e1", conv("e1a", x))
    e2 = conv("e2", conv("e2a", pool(e1)))
    e3 = conv("e3", conv("e3a", pool(e2)))
    d2 = conv("d2", conv("d2a", torch.cat([up(e3), e2], 1)))
    d1 = conv("d1", conv("d1a", torch.cat([up(d2), e1], 1)))
    out = (d1[0] * flat[o:o + 16][:, None, None]).sum(0) + flat[o + 16]
    return out * s / d.sqrt()


def potential(sigma, g, dx, vac):
    """The thin sheet's potential on the box and the ring around it, by a zero-padded convolution."""
    h, w = sigma.shape
    px, py = (max(32, 1 << (2 * v - 1).bit_length()) for v in (w, h))
    ix, iy = torch.fft.fftfreq(px, 1.0 / px, device=DEV, dtype=F64), torch.fft.fftfreq(py, 1.0 / py, device=DEV, dtype=F64)
    r = torch.sqrt(ix[None, :] ** 2 + iy[:, None] ** 2)
    r[0, 0] = 1.0 / (4.0 * math.log(1.0 + math.sqrt(2.0)))
    src = torch.zeros((py, px), device=DEV, dtype=F64)
    src[:h, :w] = torch.where(sigma >= vac, sigma, 0.0)
    f = torch.fft.irfft2(torch.fft.rfft2(src) * torch.fft.rfft2(-g * dx / r), s=(py, px))
    return torch.roll(f, (1, 1), (0, 1))[:h + 2, :w + 2].contiguous()


def gradient(phi, dx):
    return -(phi[1:-1, 2:] - phi[1:-1, :-2]) / (2 * dx), -(phi[2:, 1:-1] - phi[:-2, 1:-1]) / (2 * dx)


class Cold:
    """The cold pressure's pairs: P(x) = 1 / (1 / (K1 x^2) + 1 / (K2 x^1.5)) and its energy, tabulated as the package
    defines it (512 nodes in ln x, linear in ln u)."""

    def __init__(self, phys):
        self.pairs = [(phys.get("k1" + s, 0.0), phys.get("k2" + s, 0.0)) for s in "en"]
        self.on = self.pairs[0][0] > 0.0
        x = np.exp(np.linspace(math.log(1e-8), math.log(1e8), 512))
        self.tables = []
        for k1, k2 in self.pairs if self.on else ():
            # u / x = int P / s^2 ds = int 2 k1 t / (1 + (k1 / k2) t) dt in t = sqrt(s)
            a, t = k1 / k2, np.sqrt(x)
            j = np.where(a * t > 1e-3, 2 * k1 * (t / a - np.log1p(a * t) / a ** 2),
                         2 * k1 * t * t * (0.5 - a * t / 3 + (a * t) ** 2 / 4 - (a * t) ** 3 / 5))
            self.tables.append(torch.tensor(np.log(x * j), device=DEV, dtype=F64))

    def energy(self, x, k):
        pos = (torch.log(x.clamp(min=1e-300)) - math.log(1e-8)) / ((math.log(1e8) - math.log(1e-8)) / 511)
        i = pos.floor().long().clamp(0, 510)
        t = self.tables[k]
        u = torch.exp(t[i] + (pos - i) * (t[i + 1] - t[i]))
        return torch.where(x > 0.0, torch.where(pos < 0.0, torch.exp(t[0]) * (x / 1e-8) ** 2, u), 0.0)

    def eps(self, s, ye, xn):
        return (self.energy(ye * s, 0) + self.energy(xn * s, 1)) / s if self.on else 0.0 * s

    def pressure(self, s, ye, xn):
        out = 0.0 * s
        for x, (k1, k2) in zip((ye * s, xn * s), self.pairs if self.on else ()):
            y = x.clamp(min=1e-300)
            out = out + torch.where(x > 0.0, 1.0 / (1.0 / (k1 * y * y) + 1.0 / (k2 * y ** 1.5)), 0.0)
        return out


def mc(l, c, r):
    a, b = c - l, r - c
    m = torch.minimum(torch.minimum(0.5 * (a + b).abs(), 2 * a.abs()), 2 * b.abs())
    return torch.where(a * b > 0.0, torch.copysign(m, a), 0.0)


class Exact:
    """The step in 64 bits: P1, P2, P4, P5, P6, P8, P9 over whole planes."""

    def __init__(self, planes, phys, heat, burns):
        d = dict(gamma=2.0, G=1.0, dx=1.0, sigma_vac=1e-6, sigma_floor=1e-8, t_floor=0.05, cfl=0.4, eta_g=0.3,
                 a_r=6.25e-7, c_sb=12800.0, kappa0=1.0, opacity=0, mu=0.0, edge=1)
        d.update(phys)
        self.__dict__.update(d)
        self.q = torch.tensor(planes, device=DEV, dtype=F64)
        self.h, self.w = self.q.shape[1:]
        self.gm1, self.cold, self.heat, self.flux = self.gamma - 1.0, Cold(phys), heat, None
        self.burn = Burn(self.cold, self.t_floor, self.sigma_vac) if burns else None
        self.g = gradient(potential(self.q[0], self.G, self.dx, self.sigma_vac), self.dx)
        self.dt = self.next_dt()

    def run(self, steps):
        for _ in range(steps):
            self.g = gradient(potential(self.q[0], self.G, self.dx, self.sigma_vac), self.dx)
            self.hydro()
            if self.heat:
                self.diffuse()
            if self.burn:
                self.q = self.burn.step(self.q, self.dt)
            self.floors()
            self.dt = self.next_dt()
        return self.q

    def imu(self, x):
        return torch.full_like(x[0], 1.0 / self.mu) if self.mu > 0.0 else dot(x, IMU)

    def primitives(self, q):
        """(sigma, u, v, Pi, 1/mu, Y_e, X_n), the floor state below sigma_vac"""
        x = q[4:]
        im, ye, xn = self.imu(x), dot(x, ZA), x[9]
        low = q[0] < self.sigma_vac
        s = torch.where(low, self.sigma_floor, q[0])
        u, v = (torch.where(low, 0.0, q[k] / s) for k in (1, 2))
        raw = q[3] / s - 0.5 * (u * u + v * v) - self.cold.eps(s, ye, xn)
        floor = self.t_floor / self.gm1 * im
        eps = torch.where(low, floor, torch.maximum(raw, floor))
        return torch.stack([s, u, v, self.gm1 * s * eps + self.cold.pressure(s, ye, xn), im, ye, xn])

    def energy(self, p):
        s, u, v, pi, im, ye, xn = p
        eps = torch.maximum((pi - self.cold.pressure(s, ye, xn)) / (self.gm1 * s), self.t_floor / self.gm1 * im)
        return s * (eps + self.cold.eps(s, ye, xn)) + 0.5 * s * (u * u + v * v)

    def ghosts(self, p, x):
        """Two ghost cells a side: mirrored at a wall, the edge's own state without inflow at an open edge."""
        h, w = self.h, self.w
        iy, ix = (torch.arange(-2, n + 2, device=DEV) for n in (h, w))

        def source(i, n):
            if self.edge == 0:
                return torch.where(i < 0, -i - 1, torch.where(i >= n, 2 * n - 1 - i, i))
            return i.clamp(0, n - 1)
        sy, sx = source(iy, h), source(ix, w)
        p, x = p[:, sy][:, :, sx].clone(), x[:, sy][:, :, sx]
        for k, i, n in ((1, ix[None, :], w), (2, iy[:, None], h)):
            lo, hi = i < 0, i >= n
            if self.edge == 0:
                p[k] = torch.where(lo | hi, -p[k], p[k])
            else:
                p[k] = torch.where(lo, p[k].clamp(max=0.0), torch.where(hi, p[k].clamp(min=0.0), p[k]))
        return p, x

    def flux4(self, p, e, axis):
        un, ut = (p[2], p[1]) if axis else (p[1], p[2])
        m = p[0] * un
        f = [m, None, None, (e + p[3]) * un]
        f[1 + axis], f[2 - axis] = m * un + p[3], m * ut
        return torch.stack(f)

    def faces(self):
        """The evolved face states of the cells and their ring, and what the sources need."""
        p, x = self.ghosts(self.primitives(self.q), self.q[4:])
        c, xc = p[:, 1:-1, 1:-1], x[:, 1:-1, 1:-1]
        gx, gy = (torch.nn.functional.pad(v[None, None], (1, 1, 1, 1), mode="replicate")[0, 0] for v in self.g)
        half = 0.5 * self.dt
        start, xs = [], []
        for axis in (0, 1):
            l, r = (p[:, 1:-1, :-2], p[:, 1:-1, 2:]) if axis == 0 else (p[:, :-2, 1:-1], p[:, 2:, 1:-1])
            xl, xr = (x[:, 1:-1, :-2], x[:, 1:-1, 2:]) if axis == 0 else (x[:, :-2, 1:-1], x[:, 2:, 1:-1])
            slope = mc(l, c, r)
            central = 0.5 * (xr - xl)
            ratio = torch.where(central != 0.0, mc(xl, xc, xr) / torch.where(central != 0.0, central, 1.0), 1.0)
            theta = ratio.min(0).values.clamp(max=1.0)
            slope[4:] = theta * 0.5 * (r[4:] - l[4:])
            hottest = torch.maximum(torch.maximum(l[3] / l[0], c[3] / c[0]), r[3] / r[0])
            hot = torch.zeros_like(c[0], dtype=torch.bool)
            for f in (-0.5, 0.5):
                hot |= ~(c[3] + f * slope[3] <= 2.0 * hottest * (c[0] + f * slope[0]))
            slope[0], slope[3] = (torch.where(hot, 0.0, slope[k]) for k in (0, 3))
            for f in (-0.5, 0.5):
                start.append(c + f * slope)
                xs.append(xc + f * theta * central)
        e = [self.energy(v) for v in start]
        fl = [self.flux4(v, ev, k // 2) for k, (v, ev) in enumerate(zip(start, e))]

        def change(of):
            return half / self.dx * (of(0) - of(1) + of(2) - of(3))
        d = change(lambda k: fl[k])
        dx = change(lambda k: fl[k][0] * xs[k])
        ds = [change(lambda k: fl[k][0] * start[k][j]) for j in (4, 5, 6)]
        mid = [c[0] + d[0], c[0] * c[1] + d[1] + half * c[0] * gx, c[0] * c[2] + d[2] + half * c[0] * gy]
        out, ex, xf = [], [], []
        for k in range(4):
            v = start[k]
            s = v[0] + d[0]
            mx = v[0] * v[1] + d[1] + half * v[0] * gx
            my = v[0] * v[2] + d[2] + half * v[0] * gy
            en = e[k] + d[3] + half * v[0] * ((v[1] + 0.5 * half * gx) * gx + (v[2] + 0.5 * half * gy) * gy)
            u, w = mx / s, my / s
            im, ye, xn = ((v[0] * v[4 + j] + ds[j]) / s for j in range(3))
            raw = en / s - 0.5 * (u * u + w * w) - self.cold.eps(s, ye, xn)
            good = (s > 0.0) & (raw > 0.0)
            pi = self.gm1 * s * torch.maximum(raw, self.t_floor / self.gm1 * im) + self.cold.pressure(s, ye, xn)
            new = torch.stack([s, u, w, pi])
            out.append(torch.where(good, new, v[:4]))
            ex.append(torch.where(good, en, e[k]))
            xf.append(torch.where(good, (v[0] * xs[k] + dx) / s, xs[k]))
        return out, ex, xf, mid

    def hll(self, l, el, r, er, axis):
        un = 2 if axis else 1
        cl, cr = (torch.sqrt((self.gamma * v[3] / v[0]).clamp(min=0.0)) for v in (l, r))
        sl, sr = torch.minimum(l[un] - cl, r[un] - cr), torch.maximum(l[un] + cl, r[un] + cr)
        fl, fr = self.flux4(l, el, axis), self.flux4(r, er, axis)
        ul, ur = (torch.stack([v[0], v[0] * v[1], v[0] * v[2], ev]) for v, ev in ((l, el), (r, er)))
        f = (sr * fl - sl * fr + sl * sr * (ur - ul)) / (sr - sl)
        return torch.where(sl >= 0.0, fl, torch.where(sr <= 0.0, fr, f))

    def hydro(self):
        h, w, q, dt, k = self.h, self.w, self.q, self.dt, self.dt / self.dx
        st, e, xf, mid = self.faces()
        flux, xflux = [], []
        for axis in (0, 1):
            lo, hi = ((slice(1, -1), slice(0, -1)), (slice(1, -1), slice(1, None)))
            if axis:
                lo, hi = lo[::-1], hi[::-1]
            a, b = 2 * axis + 1, 2 * axis
            l, r = st[a][(slice(None),) + lo], st[b][(slice(None),) + hi]
            f = self.hll(l, e[a][lo], r, e[b][hi], axis)
            x = torch.where(f[0] > 0.0, xf[a][(slice(None),) + lo], xf[b][(slice(None),) + hi])
            first, last = ((slice(None), 0), (slice(None), -1)) if axis == 0 else ((0,), (-1,))
            for edge, own, inflow in ((first, r, 1.0), (last, l, -1.0)):
                at = (slice(None),) + edge
                wall = torch.zeros_like(f[at])
                wall[1 + axis] = own[at][3]
                closed = (inflow * f[at][0] > 0.0) if self.edge == 1 else torch.ones_like(f[at][0], dtype=torch.bool)
                f[at] = torch.where(closed, wall, f[at])
            flux.append(f)
            xflux.append(f[0] * x)

        def div(f):
            return (f[0][..., 1:] - f[0][..., :-1]) + (f[1][..., 1:, :] - f[1][..., :-1, :])
        low = q[0] < self.sigma_vac
        pad = torch.nn.functional.pad(low, (1, 1, 1, 1), value=True)
        empty = low & pad[1:-1, :-2] & pad[1:-1, 2:] & pad[:-2, 1:-1] & pad[2:, 1:-1]
        s0 = torch.where(low, self.sigma_floor, q[0])
        s_mid = 0.5 * (q[0] + (s0 - k * div([f[0] for f in flux])))
        s_mid = torch.where(empty | (s_mid < self.sigma_vac), 0.0, s_mid)
        phi = potential(s_mid, self.G, self.dx, self.sigma_vac)
        gmx, gmy = gradient(phi, self.dx)
        u = torch.stack([s0, torch.where(low, 0.0, q[1]), torch.where(low, 0.0, q[2]),
                         torch.where(low, self.energy(self.primitives(q)), q[3])]) - k * div(flux)
        kick = [dt * s_mid * gmx, dt * s_mid * gmy]
        net = [float(torch.where(empty, 0.0, v).sum()) for v in kick]
        dense = int(torch.where(empty, 0.0, s_mid).reshape(-1).argmax())
        # gravity's work through the faces, by the half-step states either side; none at the world's edge
        pc = phi[1:-1, 1:-1]
        m = [v[1:-1, 1:-1] for v in mid]
        gain = torch.zeros_like(pc)
        for axis in (0, 1):
            f, mom = flux[axis][0], m[1 + axis]

            def sides(v):
                if axis == 0:
                    return torch.cat([v[:, :1], v], 1), torch.cat([v, v[:, -1:]], 1)
                return torch.cat([v[:1], v]), torch.cat([v, v[-1:]])
            (sl, sh), (ml, mh), (pl, ph) = sides(m[0]), sides(mom), sides(pc)
            kk, el, eh = self.face_work(f, sl, sh, ml, mh, (pl - ph) / self.dx)
            if axis == 0:
                kick[0] = kick[0] + kk[:, 1:] - kk[:, :-1]
                gain += el[:, 1:] + eh[:, :-1]
            else:
                kick[1] = kick[1] + kk[1:] - kk[:-1]
                gain += el[1:] + eh[:-1]
        u[1] += kick[0]
        u[2] += kick[1]
        u[3] += gain
        if self.flux is not None:
            self.push(u, q, low, empty)
        x = (s0 * q[4:] - k * div(xflux)) / u[0]
        new = torch.cat([u, x])
        new = torch.where(empty, q, new)
        if float(torch.where(empty, 0.0, s_mid).max()) > 0.0:
            new[1].reshape(-1)[dense] -= net[0]
            new[2].reshape(-1)[dense] -= net[1]
        if self.flux is not None:
            share = torch.where(empty, 0.0, torch.sqrt(self.pushed[0] ** 2 + self.pushed[1] ** 2))
            if float(share.sum()) > 0.0:
                for j in (0, 1):
                    new[1 + j] -= share * torch.where(empty, 0.0, self.pushed[j]).sum() / share.sum()
        self.q = new

    def face_work(self, f, sl, sh, pl, ph, d):
        dt = self.dt
        a, b = sl.clamp(min=0.0), sh.clamp(min=0.0)
        w = torch.where(a + b > 0.0, a / (a + b).clamp(min=1e-300), 0.5)
        extra = dt * (f - 0.5 * (pl + ph)) * d
        both = (extra < 0.0) & (a > 0.0) & (b > 0.0)
        a1, b1 = torch.where(both, a, 1.0), torch.where(both, b, 1.0)
        ul, uh = pl / a1, ph / b1
        du, inv = ul - uh, 1.0 / a1 + 1.0 / b1
        c = torch.where(both, torch.minimum(-extra, 0.25 * du * du / inv), 0.0)
        some = c > 0.0
        disc = torch.sqrt((du * du - 2.0 * inv * c).clamp(min=0.0))
        down = torch.where(some, du + torch.copysign(disc, du), 1.0)
        kick = torch.where(some, -2.0 * c / down, 0.0)
        el = torch.where(some, ul * kick + 0.5 * kick * kick / a1, 0.0)
        eh = torch.where(some, -uh * kick + 0.5 * kick * kick / b1, 0.0)
        rest = extra + c
        return kick, 0.5 * dt * pl * d + w * rest + el, 0.5 * dt * ph * d + (1.0 - w) * rest + eh

    def opacity_of(self, s, t, x):
        return self.kappa0 * s * t ** -3.5 if self.opacity == 1 else self.kappa0 * (1.0 + x[0])

    def push(self, u, q, low, empty):
        """The radiation force of the last step's flux, no more than the heat above the floor allows."""
        im = self.imu(q[4:])
        s = torch.where(low, 1.0, q[0])
        raw = q[3] / s - 0.5 * (q[1] ** 2 + q[2] ** 2) / s ** 2
        t = self.gm1 * torch.maximum(raw, self.t_floor / self.gm1 * im) / im
        ks = torch.where(low, 0.0, self.opacity_of(s, t, q[4:]) * s / self.c_sb)
        d = [self.dt * ks * f for f in self.flux]
        d2 = d[0] ** 2 + d[1] ** 2
        a = u[0] * (u[3] / u[0] - 0.5 * (u[1] ** 2 + u[2] ** 2) / u[0] ** 2 - self.t_floor / self.gm1 * im)
        qd = u[1] * d[0] + u[2] * d[1]
        disc = torch.sqrt((qd * qd + 2.0 * u[0] * a * d2).clamp(min=0.0))
        share = torch.where(qd >= 0.0, 2.0 * u[0] * a / (qd + disc).clamp(min=1e-300), (disc - qd) / d2.clamp(min=1e-300))
        share = torch.where(a > 0.0, share.clamp(max=1.0), 0.0)
        self.pushed = [torch.where((d2 > 0.0) & ~empty, share * v, 0.0) for v in d]
        u[1] += self.pushed[0]
        u[2] += self.pushed[1]

    def diffuse(self):
        """Backward Euler for u = a_r T^4 over the flux-limited faces, Newton on T to the end, then the delta closure."""
        q, dt = self.q, self.dt
        s, x = q[0], q[4:]
        gas = s >= self.sigma_vac
        im = self.imu(x)
        s1 = torch.where(gas, s, 1.0)
        raw = q[3] / s1 - 0.5 * (q[1] ** 2 + q[2] ** 2) / s1 ** 2
        t0 = torch.where(gas, self.gm1 * torch.maximum(raw, self.t_floor * im / self.gm1) / im, self.t_floor)
        sg = torch.where(gas, s, self.sigma_floor)
        ks = self.opacity_of(sg, t0, x) * sg  # of a gas cell; the vacuum beside it takes the gas cell's opacity
        kap = self.opacity_of(sg, t0, x)
        cap = sg * im / self.gm1
        uvac = self.a_r * self.t_floor ** 4

        def law(axis):
            def sides(v, fill):
                v = torch.nn.functional.pad(v, (1, 1, 0, 0) if axis == 0 else (0, 0, 1, 1), value=fill)
                return (v[:, :-1], v[:, 1:]) if axis == 0 else (v[:-1], v[1:])
            (ga, gb), (ta, tb), (ka, kb), (na, nb) = sides(gas, False), sides(t0, self.t_floor), sides(ks, 0.0), sides(kap, 0.0)
            ka, kb = torch.where(ga, ka, nb * self.sigma_floor), torch.where(gb, kb, na * self.sigma_floor)
            any_ = ga | gb
            ea, eb = self.a_r * ta ** 4, self.a_r * tb ** 4
            fe, k = 0.5 * (ea + eb), torch.where(any_, 0.5 * (ka + kb), 1.0)
            r = (eb - ea).abs() / (self.dx * k * fe)
            d = self.c_sb * (2.0 + r) / (6.0 + 3.0 * r + r * r) / k / self.dx ** 2
            return torch.where(any_, d, 0.0), torch.where(ga & gb, d, 0.0)
        (kx, ax), (ky, ay) = law(0), law(1)
        kvac = diagonal(torch.zeros_like(s), kx - ax, ky - ay) * gas
        t = t0.clone()
        eta = 1e-2
        for _ in range(60):
            heat = cap / dt
            c = heat / (4.0 * self.a_r * t ** 3)
            u = self.a_r * t ** 4
            own = torch.where(gas, c + kvac, 1.0)
            rhs = torch.where(gas, c * u - heat * (t - t0) + kvac * uvac, 0.0)
            v = conjugate_gradients(own, ax, ay, rhs, torch.where(gas, u, 0.0), eta)
            new = torch.where(gas, (v.clamp(min=uvac) / self.a_r) ** 0.25, t)
            new = torch.minimum(torch.maximum(new, 0.5 * t), 2.0 * t)
            moved = float(((new - t).abs() / t).max())
            t = new
            if eta <= 1e-11 and moved < 1e-9:
                break
            eta = min(1e-2, max(1e-11, 1e-2 * moved))
        u = torch.where(gas, self.a_r * t ** 4, uvac)
        gas_cap = cap * gas
        lost = (dt * kvac * (u - uvac)).sum()
        delta = -((gas_cap * (t - t0)).sum() + lost) / (gas_cap * t).sum()
        up = torch.nn.functional.pad(u, (1, 1, 1, 1), value=uvac)
        fx, fy = -kx * self.dx * (up[1:-1, 1:] - up[1:-1, :-1]), -ky * self.dx * (up[1:, 1:-1] - up[:-1, 1:-1])
        self.flux = [0.5 * (fx[:, 1:] + fx[:, :-1]), 0.5 * (fy[1:] + fy[:-1])]
        self.q = q.clone()
        self.q[3] += gas_cap * ((1.0 + delta) * t - t0)

    def floors(self):
        q = self.q.clone()
        x = q[4:].clamp(min=0.0)
        x = x / x.sum(0)
        im, ye = self.imu(x), dot(x, ZA)
        floor = self.t_floor / self.gm1 * im
        low = q[0] < self.sigma_vac
        vac = torch.full_like(q[0], self.sigma_floor)
        s = torch.where(low, vac, q[0])
        raw = q[3] / s - 0.5 * (q[1] ** 2 + q[2] ** 2) / s ** 2 - self.cold.eps(s, ye, x[9])
        e = torch.where(low, vac * (floor + self.cold.eps(vac, ye, x[9])), q[3] + s * (floor - raw).clamp(min=0.0))
        self.q = torch.cat([torch.stack([s, torch.where(low, 0.0, q[1]), torch.where(low, 0.0, q[2]), e]), x])

    def next_dt(self):
        s, u, v, pi, *_ = self.primitives(self.q)
        c = torch.sqrt(self.gamma * pi / s)
        g = torch.hypot(*self.g).max()
        dt = self.cfl * self.dx / (u.abs() + v.abs() + 2.0 * c).max()
        return float(torch.minimum(dt, self.eta_g * torch.sqrt(self.dx / g)) if g > 0.0 else dt)


class Burn:
    """The burning pass: every record but N_Fe (whose gate these scenes never open) by linearised backward Euler,
    sub-cycled cell by cell."""

    def __init__(self, cold, t_floor, sigma_vac):
        from sandbox_reactions_amd import react
        self.p, self.cold, self.t_floor, self.sigma_vac = react.params(overrides={"burn_k": 10.0}), cold, t_floor, sigma_vac
        self.recs = [self.p.rec[i] for i in range(self.p.n_records) if i != self.p.nfe]
        self.gate = self.p.rec[self.p.nfe].sigma_g
        self.nu = torch.zeros((len(self.recs), NS), device=DEV, dtype=F64)
        self.tables = []
        for i, r in enumerate(self.recs):
            for j in range(r.n_out):
                self.nu[i, r.out_species[j]] += r.out_share[j]
            for j in range(r.n_in):
                self.nu[i, r.in_species[j]] -= r.in_share[j]
            nodes = r.t_thr * torch.exp(math.log(2.5) * torch.arange(256, device=DEV, dtype=F64) / 255)
            self.tables.append(torch.log(self.gamow(r, nodes)))
        self.q = torch.tensor([r.q for r in self.recs], device=DEV, dtype=F64)
        self.imu = torch.tensor(IMU, device=DEV, dtype=F64)

    @staticmethod
    def gamow(r, t):
        out = 0.0
        for k in range(r.n_terms):
            u = torch.log(t / r.t_k[k])
            out = out + torch.exp(math.log(r.w[k]) - 2 / 3 * u - (3 * r.nu[k] + 2) * torch.expm1(-u / 3))
        return out

    def factor(self, i, t):
        r, tab = self.recs[i], self.tables[i]
        pos = torch.log(t / r.t_thr) / (math.log(2.5) / 255)
        k = pos.clamp(min=0.0).floor().long().clamp(max=254)
        inside = torch.exp(tab[k] + (pos - k) * (tab[k + 1] - tab[k]))
        return torch.where(t < r.t_thr, 0.0, torch.where(pos >= 255, self.gamow(r, t), inside))

    def temperature(self, s, x, e):
        mu = 1.0 / (x @ self.imu)
        cold = self.cold.eps(s, x @ torch.tensor(ZA, device=DEV, dtype=F64), x[:, 9])
        return mu, mu * torch.maximum(e - cold, self.t_floor / mu)

    def step(self, planes, dt):
        shape = planes.shape[1:]
        sigma = planes[0].reshape(-1)
        kinetic = 0.5 * (planes[1] ** 2 + planes[2] ** 2).reshape(-1) / sigma ** 2
        x = planes[4:].reshape(NS, -1).T.contiguous()
        e0 = planes[3].reshape(-1) / sigma - kinetic
        e = e0.clone()
        if float((sigma * (x @ torch.tensor(ZA, device=DEV, dtype=F64))).max()) > self.gate:
            raise RuntimeError("a cell opens N_Fe's gate")
        done, h_try = torch.zeros_like(e), torch.full_like(e, math.inf)
        retry = torch.full_like(e, math.inf)
        live = torch.nonzero(sigma >= self.sigma_vac)[:, 0]
        while live.numel():
            s, xi, ei = sigma[live], x[live], e[live]
            mu, t = self.temperature(s, xi, ei)
            omega = torch.zeros((live.numel(), len(self.recs)), device=DEV, dtype=F64)
            grad = torch.zeros((live.numel(), len(self.recs), NS), device=DEV, dtype=F64)
            for i, r in enumerate(self.recs):
                f = r.a_coef * s ** r.a_sigma * self.factor(i, t)
                ins = [(r.in_species[k], r.in_order[k]) for k in range(r.n_in)]
                prod = f
                for j, n in ins:
                    prod = prod * xi[:, j] ** n
                omega[:, i] = prod
                for j, n in ins:
                    others = f
                    for m, o in ins:
                        if m != j:
                            others = others * xi[:, m] ** o
                    grad[:, i, j] += n * xi[:, j] ** (n - 1) * others
            rate = omega @ self.nu
            qdot = omega @ self.q
            eps = t / mu
            clock = (qdot / (eps * torch.sqrt(2.0 * eps) / self.p.burn_k)).clamp(min=1.0)
            left = (dt - done[live]) / clock
            idle = (omega == 0.0).all(1)
            h = torch.minimum(left, self.p.burn_dx / rate.abs().max(1).values.clamp(min=1e-300))
            warming = (mu * qdot - t * mu * (rate @ self.imu)).abs()
            h = torch.minimum(h, self.p.burn_dt * t / warming.clamp(min=1e-300))
            h = torch.minimum(torch.minimum(h, h_try[live]), retry[live])
            last = h >= left
            a = torch.eye(NS, device=DEV, dtype=F64) - h[:, None, None] * torch.einsum("ri,nrj->nij", self.nu, grad)
            dx = torch.linalg.solve(a, (h[:, None] * rate)[:, :, None])[:, :, 0]
            new = xi + dx
            negative = (new < -1e-12).any(1)
            moved = h[:, None] * (omega + (grad @ dx[:, :, None])[:, :, 0])
            en = ei + moved @ self.q
            new = new.clamp(min=0.0)
            new = new / new.sum(1, keepdim=True)
            _, tn = self.temperature(s, new, en)
            bad = negative | (dx.abs().max(1).values > self.p.burn_dx * (1 + 1e-12))
            bad |= (tn - t).abs() / t > self.p.burn_dt * (1 + 1e-12)
            bad &= ~idle
            take = ~bad & ~idle
            on = live[take]
            x[on], e[on] = new[take], en[take]
            done[on] = torch.where(last, dt, done[live] + h * clock)[take]
            h_try[on] = 2.0 * h[take]
            retry[on] = math.inf
            retry[live[bad]] = 0.5 * h[bad]
            done[live[idle]] = dt
            live = live[done[live] < dt]
        out = planes.clone()
        out[3] = (planes[3].reshape(-1) + sigma * (e - e0)).reshape(shape)
        out[4:] = x.T.reshape(NS, *shape)
        return out
