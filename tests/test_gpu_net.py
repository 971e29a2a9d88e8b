"""The learned preconditioner's network on the GPU against the f64 numpy oracle (oracle/unet.py): every layer from
the GPU's own inputs (which pins the matrix-core lane layout and the implicit-GEMM indexing), the whole forward pass,
every parameter's gradient, Adam, and the network inside flexible CG (convergence, fallback to plain multigrid).

Tolerances: activations and weights are BF16 (8 significant bits), so a layer from its exact input agrees to about
2^-8 of its scale; gradients flow through ten BF16 layers and are compared by relative L2 and direction.
"""
import numpy as np
import pytest

from oracle import unet

pytestmark = pytest.mark.gpu


def bf16(a):
    """Round to BF16 (nearest even), returned as float64."""
    b = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    r = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16) << 16
    return r.astype(np.uint32).view(np.float32).astype(np.float64)


def system(n, seed, contrast=2.0):
    rng = np.random.default_rng(seed)
    own = np.exp(rng.normal(0.0, 1.0, (n, n))).astype(np.float32)
    kx = np.exp(rng.normal(0.0, contrast, (n, n + 1))).astype(np.float32)
    ky = np.exp(rng.normal(0.0, contrast, (n + 1, n))).astype(np.float32)
    kx[:, 0] = kx[:, n] = 0.0
    ky[0, :] = ky[n, :] = 0.0
    return own, kx, ky


def cuda(*arrs):
    import torch
    return [torch.tensor(np.ascontiguousarray(a, np.float32), device="cuda") for a in arrs]


def random_params(seed):
    from sandbox_reactions_amd import net as N
    p = N.init_params(seed)
    rng = np.random.default_rng(seed + 100)
    for k in p:
        if k.endswith(".b"):
            p[k] = (rng.normal(size=p[k].shape) * 0.1).astype(np.float32)
    p["out.w"] = (rng.normal(size=16) * 0.3).astype(np.float32)
    return p


def close(gpu, ref, frac):
    scale = max(np.abs(ref).max(), 1e-30)
    return np.abs(gpu - ref).max() / scale <= frac


def test_every_layer_matches_the_oracle(gpu_lib):
    import torch
    import sandbox_reactions_amd as sr
    print("net layers 64x48", flush=True)
    w, h = 64, 48
    p = random_params(1)
    net = sr.Net(w, h, p)
    own, kx, ky = system(64, 2)
    own, kx, ky = own[:h, :w].copy(), kx[:h, :w + 1].copy(), ky[:h + 1, :w].copy()
    kx[:, w] = 0.0
    ky[h, :] = 0.0
    r = np.random.default_rng(3).normal(size=(h, w)).astype(np.float32)
    t_own, t_kx, t_ky, t_r = cuda(own, kx, ky, r)
    z = torch.empty((h, w), dtype=torch.float32, device="cuda")
    net.apply(t_own, t_kx, t_ky, t_r, z)
    torch.cuda.synchronize()
    A = {k: net.activation(k, w, h).astype(np.float64) for k in
         ["x", "e1a", "e1", "p1", "e2a", "e2", "p2", "e3a", "e3", "d2a", "d2", "d1a", "d1"]}
    # features
    xo, s, dis = unet.features(own.astype(np.float64), kx.astype(np.float64), ky.astype(np.float64),
                               r.astype(np.float64))
    xo[:, :, 1] = np.clip(xo[:, :, 1], -20, 20)
    assert np.abs(A["x"][:, :, :3] - xo).max() <= 2 ** -7 * np.abs(xo).max(axis=(0, 1)).max()
    assert np.all(A["x"][:, :, 3:] == 0.0)
    W = {k: bf16(v) for k, v in p.items() if k.endswith(".w") and not k.startswith("out")}
    B = {k: np.asarray(v, np.float64) for k, v in p.items() if k.endswith(".b")}

    def layer(name, inp):
        return unet.relu(unet.conv3(inp, W[name + ".w"], B[name + ".b"]))

    checks = [("e1a", A["x"][:, :, :3]), ("e1", A["e1a"]), ("e2a", A["p1"]), ("e2", A["e2a"]), ("e3a", A["p2"]),
              ("e3", A["e3a"]), ("d2a", np.concatenate([unet.up(A["e3"]), A["e2"]], axis=2)), ("d2", A["d2a"]),
              ("d1a", np.concatenate([unet.up(A["d2"]), A["e1"]], axis=2)), ("d1", A["d1a"])]
    for name, inp in checks:
        ref = layer(name, inp)
        err = np.abs(A[name] - ref).max() / max(np.abs(ref).max(), 1e-30)
        assert err <= 2 ** -7, (name, err)
    assert close(A["p1"], unet.pool(A["e1"]), 2 ** -7)
    assert close(A["p2"], unet.pool(A["e2"]), 2 ** -7)
    zref = (A["d1"] @ p["out.w"].astype(np.float64) + p["out.b"][0]) * s * dis
    assert close(z.cpu().numpy(), zref, 1e-4)


def test_forward_matches_the_f64_network(gpu_lib):
    import torch
    import sandbox_reactions_amd as sr
    print("net forward 64x64", flush=True)
    n = 64
    p = random_params(4)
    net = sr.Net(n, n, p)
    own, kx, ky = system(n, 5)
    r = np.random.default_rng(6).normal(size=(n, n)).astype(np.float32)
    t = cuda(own, kx, ky, r)
    z = torch.empty((n, n), dtype=torch.float32, device="cuda")
    net.apply(*t, z)
    pd = {k: np.asarray(v, np.float64) for k, v in p.items()}
    zref = unet.apply(pd, own.astype(np.float64), kx.astype(np.float64), ky.astype(np.float64),
                      r.astype(np.float64))
    rel = np.linalg.norm(z.cpu().numpy() - zref) / np.linalg.norm(zref)
    assert rel <= 3e-2, rel


def dense_solve(own, kx, ky, r):
    """e = A^-1 r by a sparse direct solve of the face-form operator (interior faces)."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as spla
    h, w = own.shape
    idx = np.arange(w * h).reshape(h, w)
    kxi, kyi = kx[:, 1:w], ky[1:h, :]
    a, b = idx[:, :-1].ravel(), idx[:, 1:].ravel()
    c, d = idx[:-1, :].ravel(), idx[1:, :].ravel()
    rows = np.concatenate([a, b, c, d])
    cols = np.concatenate([b, a, d, c])
    vals = -np.concatenate([kxi.ravel(), kxi.ravel(), kyi.ravel(), kyi.ravel()])
    diag = own.ravel().astype(np.float64).copy()
    np.add.at(diag, a, kxi.ravel())
    np.add.at(diag, b, kxi.ravel())
    np.add.at(diag, c, kyi.ravel())
    np.add.at(diag, d, kyi.ravel())
    A = sp.coo_matrix((vals, (rows, cols)), shape=(w * h, w * h)).tocsr() + sp.diags(diag)
    return spla.spsolve(A.tocsc(), r.ravel()).reshape(h, w)


def test_gradients_match_the_oracle(gpu_lib):
    import sandbox_reactions_amd as sr
    from sandbox_reactions_amd import net as N
    print("net gradients 32x32", flush=True)
    n = 32
    p = random_params(7)
    net = sr.Net(n, n, p)
    own, kx, ky = system(n, 8, contrast=1.0)
    r = np.random.default_rng(9).normal(size=(n, n)).astype(np.float32)
    o64, kx64, ky64, r64 = (a.astype(np.float64) for a in (own, kx, ky, r))
    e = dense_solve(o64, kx64, ky64, r64).astype(np.float32)
    loss = net.loss_grad(*cuda(own, kx, ky, r, e))
    g = N.unflatten(net.grads())
    pd = {k: bf16(v) if (k.endswith(".w") and not k.startswith("out")) else np.asarray(v, np.float64)
          for k, v in p.items()}
    lref, gref = unet.energy_loss(pd, o64, kx64, ky64, r64, e.astype(np.float64))
    assert abs(loss - lref) <= 2e-2 * lref, (loss, lref)
    for k in gref:
        a, b = g[k].astype(np.float64).ravel(), gref[k].ravel()
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        cos = a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30)
        assert rel <= 0.15 and cos >= 0.99, (k, rel, cos)


def test_adam_matches_the_algorithm(gpu_lib):
    import sandbox_reactions_amd as sr
    print("net adam", flush=True)
    n = 32
    p = random_params(10)
    net = sr.Net(n, n, p)
    own, kx, ky = system(n, 11, contrast=1.0)
    r = np.random.default_rng(12).normal(size=(n, n)).astype(np.float32)
    e = dense_solve(*(a.astype(np.float64) for a in (own, kx, ky, r))).astype(np.float32)
    t = cuda(own, kx, ky, r, e)
    p0 = net.params().astype(np.float64)
    net.loss_grad(*t)
    g = net.grads().astype(np.float64)
    net.adam(1e-3)
    p1 = net.params().astype(np.float64)
    # first Adam step: the bias-corrected moments are g and g^2, so each parameter moves by lr g / (|g| + eps)
    expect = p0 - 1e-3 * g / (np.abs(g) + 1e-8)
    assert np.allclose(p1, expect, atol=1e-6)


def test_training_lowers_the_loss(gpu_lib):
    import sandbox_reactions_amd as sr
    print("net training 64x64", flush=True)
    n = 64
    net = sr.Net(n, n)
    own, kx, ky = system(n, 13)
    rng = np.random.default_rng(14)
    samples = []
    o64, kx64, ky64 = (a.astype(np.float64) for a in (own, kx, ky))
    for _ in range(4):
        r = rng.normal(size=(n, n)).astype(np.float32)
        samples.append(cuda(own, kx, ky, r, dense_solve(o64, kx64, ky64, r.astype(np.float64))))
    first = np.mean([net.loss_grad(*s) for s in samples])
    for it in range(150):
        net.loss_grad(*samples[it % 4])
        net.adam(2e-3)
    last = np.mean([net.loss_grad(*s) for s in samples])
    assert first > 0.9 and last < 0.6 * first, (first, last)


def test_learned_fcg_converges_and_falls_back(gpu_lib):
    import torch
    import sandbox_reactions_amd as sr
    print("learned FCG 128x128", flush=True)
    n = 128
    own, kx, ky = system(n, 15)
    own *= 1e-2
    b = np.random.default_rng(16).normal(size=(n, n))
    f = sr.Fld(n, n)
    f.set_system(*cuda(own, kx, ky))
    bt = torch.tensor(b, device="cuda")
    xm = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    it_m, rel_m = f.solve(bt, xm, tol=1e-8)
    net = sr.Net(n, n, random_params(17))
    with pytest.raises(sr.SrError):
        f.solve(bt, torch.zeros_like(xm), tol=1e-8, precond=sr.PRECOND_LEARNED)
    f.set_network(net)
    xl = torch.zeros_like(xm)
    it_l, rel_l, li, fb = f.solve_stats(bt, xl, tol=1e-8, precond=sr.PRECOND_LEARNED)
    assert rel_l <= 1e-8 and (fb or li == it_l)
    assert torch.linalg.norm(xl - xm) <= 1e-6 * torch.linalg.norm(xm)
    f.set_network(net, fallback_iterations=2)
    xf = torch.zeros_like(xm)
    it_f, rel_f, li, fb = f.solve_stats(bt, xf, tol=1e-8, precond=sr.PRECOND_LEARNED)
    assert fb and li <= 8 and rel_f <= 1e-8
    assert torch.linalg.norm(xf - xm) <= 1e-6 * torch.linalg.norm(xm)


def test_trained_network_gains_over_the_v_cycle_alone(gpu_lib):
    """The committed network, trained on 256^2 / 512^2 systems, on a held-out 256^2 system drawn the same way: the
    A-norm of what one V-cycle leaves, after the network's correction, against the V-cycle alone (1 by definition).
    Inside flexible CG the correction does not pay (the iteration counts are printed, not asserted); the solve with
    fallback converges within a few iterations of plain multigrid."""
    import torch
    import sandbox_reactions_amd as sr
    from sandbox_reactions_amd import scenes, train
    print("trained network 256x256", flush=True)
    n = 256
    net = sr.Net(n, n, train.load())
    own, kx, ky = train.system_tensors(n, scenes.SEED_BASE + 777)
    f = sr.Fld(n, n)
    f.set_system(own, kx, ky)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    losses = []
    for cg in (0, 5, 10, 20, 30, 40):
        r1, e1 = train.make_sample(f, own, kx, ky, gen, tol=1e-8, cg_steps=cg)
        losses.append(net.loss_grad(own, kx, ky, r1, e1))
    print(f"error energy left by V + network / V alone: {np.round(losses, 4)}", flush=True)
    assert np.mean(losses) <= 0.95, losses
    c, kx64, ky64, b, dt = scenes.fld_system(n, seed=scenes.SEED_BASE + 777)
    bt = torch.tensor(b, device="cuda")
    x = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    it_p, rel_p, _, _ = f.solve_stats(bt, x, tol=1e-8)
    f.set_network(net, fallback_iterations=it_p)
    x2 = torch.zeros_like(x)
    it_l, rel_l, li, fb = f.solve_stats(bt, x2, tol=1e-8, precond=sr.PRECOND_LEARNED)
    f.set_network(net, fallback_iterations=0)
    x3 = torch.zeros_like(x)
    it_n, rel_n, li_n, fb_n = f.solve_stats(bt, x3, tol=1e-8, precond=sr.PRECOND_LEARNED)
    print(f"iterations: plain {it_p}, learned with fallback {it_l} ({li} with the network, fell back {fb}), "
          f"learned without fallback {it_n}", flush=True)
    assert rel_l <= 1e-8 and rel_n <= 1e-8 and not fb_n and li_n == it_n
    assert it_l <= it_p + 20


# Sizes at which the convolution's tiles of 64 pixels x 2, 4 or 8 rows all run, each with ragged edges: 68 x 36 (two rows
# everywhere), 516 x 260 (four at full resolution), 2052 x 1028 (eight, eight and four).
@pytest.mark.parametrize("w,h", [(68, 36), (516, 260), (2052, 1028)])
def test_layers_match_over_every_tile_height(gpu_lib, w, h):
    """Every layer, the pooled means and the output from the GPU's own inputs, in FP32 on the device: a layer's BF16
    output is within half an ulp (2^-9 of its size, 2^-8 allowing the FP32 sums' order to tip a rounding)."""
    import torch
    import sandbox_reactions_amd as sr
    print(f"net layers {w}x{h}", flush=True)
    p = random_params(21)
    net = sr.Net(w, h, p)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(22)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    own, kx, ky = rnd(h, w).exp(), rnd(h, w + 1).exp(), rnd(h + 1, w).exp()
    r, z = rnd(h, w), torch.empty(h, w, device="cuda")
    net.apply(own, kx, ky, r, z)
    A = {k: torch.tensor(net.activation(k, w, h), device="cuda") for k in
         ["x", "e1a", "e1", "p1", "e2a", "e2", "p2", "e3a", "e3", "d2a", "d2", "d1a", "d1"]}
    up = lambda a: a.repeat_interleave(2, 0).repeat_interleave(2, 1)
    for name, inp in [("e1a", A["x"][:, :, :3]), ("e1", A["e1a"]), ("e2a", A["p1"]), ("e2", A["e2a"]),
                      ("e3a", A["p2"]), ("e3", A["e3a"]), ("d2a", torch.cat([up(A["e3"]), A["e2"]], 2)),
                      ("d2", A["d2a"]), ("d1a", torch.cat([up(A["d2"]), A["e1"]], 2)), ("d1", A["d1a"])]:
        wt = torch.tensor(bf16(p[name + ".w"]), device="cuda").float()
        hh, ww, ci = inp.shape
        padded = torch.zeros(hh + 2, ww + 2, ci, device="cuda")
        padded[1:-1, 1:-1] = inp
        ref = torch.tensor(p[name + ".b"], device="cuda").expand(hh * ww, -1).clone()
        for t in range(9):
            ref += padded[t // 3:t // 3 + hh, t % 3:t % 3 + ww].reshape(hh * ww, ci) @ wt[t // 3, t % 3]
        ref = ref.clamp(min=0.0).reshape(hh, ww, -1)
        err = float(((A[name] - ref).abs() - 2.0 ** -8 * ref.abs()).max()) / float(ref.max())
        assert err <= 1e-5, (name, err)
    for name, src in (("p1", "e1"), ("p2", "e2")):
        a = A[src]
        mean = 0.25 * (a[::2, ::2] + a[::2, 1::2] + a[1::2, ::2] + a[1::2, 1::2])
        assert torch.equal(A[name], mean.bfloat16().float()), name
    ks = kx[:, :-1] + kx[:, 1:] + ky[:-1] + ky[1:]
    dis = (own + ks).double().rsqrt()
    s = (r.double() * dis).square().mean().sqrt()
    ref = (A["d1"].double() @ torch.tensor(p["out.w"], device="cuda").double() + float(p["out.b"][0])) * s * dis
    assert float((z - ref).abs().max()) <= 1e-5 * float(ref.abs().max())


# one tile row, ragged tiles in both axes (32 x 4), and more tiles than blocks (553 blocks walk two each)
@pytest.mark.parametrize("w,h", [(32, 4), (68, 36), (516, 260)])
def test_last_layers_weight_gradient_over_ragged_tiles(gpu_lib, w, h):
    """dW and db of the last 3x3 layer from its own input and output: ga = dL/d(out) w_out where the output is positive,
    stored in BF16 (2^-9 of each term, so at most that of the sum of the terms' sizes)."""
    import torch
    import sandbox_reactions_amd as sr
    from sandbox_reactions_amd import net as N
    print(f"net dW {w}x{h}", flush=True)
    p = random_params(23)
    net = sr.Net(w, h, p)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(24)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    own, kx, ky = rnd(h, w).exp(), rnd(h, w + 1).exp(), rnd(h + 1, w).exp()
    kx[:, 0] = kx[:, w] = 0.0
    ky[0] = ky[h] = 0.0
    r, e, z = rnd(h, w), rnd(h, w), torch.empty(h, w, device="cuda")
    net.apply(own, kx, ky, r, z)
    net.loss_grad(own, kx, ky, r, e)
    g = N.unflatten(net.grads().astype(np.float64))
    A = {k: torch.tensor(net.activation(k, w, h), device="cuda").double() for k in ("d1a", "d1")}
    ks = (kx[:, :-1] + kx[:, 1:] + ky[:-1] + ky[1:]).double()

    def op(v):
        out = own.double() * v
        dx, dy = kx[:, 1:-1].double() * (v[:, 1:] - v[:, :-1]), ky[1:-1].double() * (v[1:] - v[:-1])
        out[:, :-1] -= dx
        out[:, 1:] += dx
        out[:-1] -= dy
        out[1:] += dy
        return out

    dis = (own.double() + ks).rsqrt()
    s = (r.double() * dis).square().mean().sqrt()
    gout = 2.0 * op(z.double() - e.double()) / (e.double() * op(e.double())).sum() * s * dis
    ga = gout[:, :, None] * torch.tensor(p["out.w"], device="cuda").double() * (A["d1"] > 0)
    padded = torch.zeros(h + 2, w + 2, 16, device="cuda", dtype=torch.float64)
    padded[1:-1, 1:-1] = A["d1a"]
    for t in range(9):
        x = padded[t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(-1, 16)
        ref, size = x.T @ ga.reshape(-1, 16), x.abs().T @ ga.abs().reshape(-1, 16)
        err = (torch.tensor(g["d1.w"][t // 3, t % 3], device="cuda") - ref).abs()
        assert bool((err <= 2.0 ** -8 * size + 1e-30).all()), (t, float((err / size).max()))
    err = (torch.tensor(g["d1.b"], device="cuda") - ga.sum((0, 1))).abs()
    assert bool((err <= 2.0 ** -8 * ga.abs().sum((0, 1)) + 1e-30).all())


def one_infinite_pixel(w, h, x, y):
    """A system whose share of the diagonal is 0 at one cell: its third feature, log(own / d), is -inf there alone."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(31)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    own, kx, ky = rnd(h, w).exp(), rnd(h, w + 1).exp(), rnd(h + 1, w).exp()
    own[y, x] = 0.0
    return own, kx, ky, rnd(h, w), rnd(h, w)


def single_path(p):
    """e1a passes minus the third feature of its own pixel into channel 0, so that an infinite one stays one pixel of one
    channel; every other weight of the layer is 0 (0 times infinity is no number, which the ReLU makes 0)."""
    p["e1a.w"][:] = 0.0
    p["e1a.b"][:] = 0.0
    p["e1a.w"][1, 1, 2, 0] = -1.0


# R = 2 rows a wave, then 8 (68 x 36 and 2052 x 1028 as above), the pixel inside a tile and at its left border
@pytest.mark.parametrize("w,h,x,y", [(68, 36, 20, 9), (68, 36, 64, 35), (2052, 1028, 128, 200)])
def test_an_infinite_activation_meets_no_padding(gpu_lib, w, h, x, y):
    """An infinite input pixel reaches the nine outputs around it and those are infinite (or, negative, 0): a layer of 8
    or 16 input channels pads its products, and the padding reads no pixel."""
    import torch
    import sandbox_reactions_amd as sr
    print(f"net infinite {w}x{h}", flush=True)
    own, kx, ky, r, _ = one_infinite_pixel(w, h, x, y)
    z = torch.empty(h, w, device="cuda")
    for name, src in (("e1a", "x"), ("e1", "e1a")):
        p = random_params(32)
        if name == "e1":
            single_path(p)
        net = sr.Net(w, h, p)
        net.apply(own, kx, ky, r, z)
        inp = torch.tensor(net.activation(src, w, h))[:, :, :3 if name == "e1a" else 16].double()
        assert int(torch.isinf(inp).sum()) == 1 and not bool(torch.isnan(inp).any())
        got = torch.tensor(net.activation(name, w, h)).double()
        wt = torch.tensor(bf16(p[name + ".w"])).double()
        for dy in range(-1, 2):
            for dx in range(-1, 2):
                if 0 <= y + dy < h and 0 <= x + dx < w:
                    sign = wt[1 - dy, 1 - dx, 2 if name == "e1a" else 0] * (-1.0 if name == "e1a" else 1.0)
                    assert torch.equal(torch.isinf(got[y + dy, x + dx]), sign > 0), (name, dy, dx)
        assert int(torch.isinf(got).sum()) == int(torch.isinf(got[max(y - 1, 0):y + 2, max(x - 1, 0):x + 2]).sum())


def test_a_weight_gradient_reads_no_pixel_past_the_last_row(gpu_lib):
    """An infinite activation in the last row of a half-resolution layer whose outputs around it the ReLU all stops: the
    weight gradient's sums for the row taps whose output pixel would lie below the image hold no such pixel, in a tile of
    four rows that ends two rows past the image (six rows)."""
    import torch
    import sandbox_reactions_amd as sr
    print("net dW past the last row", flush=True)
    w, h = 16, 12
    own, kx, ky, r, e = one_infinite_pixel(w, h, 5, 11)
    p = random_params(33)
    single_path(p)
    for name in ("e1", "e2a"):
        p[name + ".w"][:, :, 0] = 0.0
        p[name + ".w"][1, 1, 0, 0] = 1.0  # the pixel goes on in channel 0 alone
    p["e2.w"][:, :, 0] = -1.0             # and is stopped here
    p["e2.b"][:] = 1.0
    net = sr.Net(w, h, p)
    net.loss_grad(own, kx, ky, r, e)
    x, y = torch.tensor(net.activation("e2a", w, h)), torch.tensor(net.activation("e2", w, h))
    assert torch.isinf(x).nonzero().tolist() == [[5, 2, 0]] and not bool(torch.isnan(x).any())
    assert bool((y[4:, 1:4] == 0).all()) and not bool(torch.isinf(y).any())
    g = sr.net.unflatten(net.grads())["e2.w"]
    assert np.isnan(g[1:, :, 0]).all()       # 0 times infinity, the pixel's own row and the one above
    assert np.isfinite(g[0, :, 0]).all() and np.isfinite(g[:, :, 1:]).all()
