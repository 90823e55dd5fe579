"""Performance cases of the NPA library: the calls a program makes through its public entry points.

* rollouts: create a device state from particles, take the steps between two frames, read it back;
* single steps of the ``NpaModel.step`` form, from a demo of a thousand particles to a dense cloud;
* the training pass: perception, update MLP and Euler step forward, the perception adjoint backward;
* drawing: the 2D splat, the render loss's particle views, the raster of decoded Gaussians.

The models are the library's presets (``NpaConfig.for_preset``) and the configurations of
``synthetic.py``; particles are drawn uniformly in a disk, a ball or a periodic square or on a closed
surface, states from N(0, 0.1) and weights from U(-0.1, 0.1), as ``synthetic.py`` draws them.
"""
from __future__ import annotations

import math

import torch

from burn_automata_amd import _abi, kernels
from burn_automata_amd.config import (ALL_VIEWS, Boundary, GaussianDecodeConfig, GaussianDecodeMode, HashGridConfig,
                                      HashGridMode, NpaConfig, RasterCamera, RasterColor, RenderLossConfig,
                                      Splat2dConfig)
from burn_automata_amd.executor import HipAutomataExecutor
from burn_automata_amd.model import NpaModel, NpaWeights
from burn_automata_amd.synthetic import config_c1

DT = 1.0
UPDATE_PROB = 0.5
DISK_RADIUS, BALL_RADIUS = 1.0, 0.5
SHELL = (0.6, 0.45, 0.35)  # semi-axes of the closed surface
SHELL_AREA = 2.7
# the clouds each model is run on
CLOUDS = {"c1": "disk", "growing_2d": "disk", "point_mnist": "disk", "texture_2d": "square",
          "growing_3dgs": "ball", "c4": "shell"}
ENGINES = {"valu": _abi.MLP_VALU, "mfma": _abi.MLP_MFMA}
DECODES = {"fixed": GaussianDecodeMode.GaussianSh0FixedScale,
           "learned": GaussianDecodeMode.GaussianSh0LearnedScale,
           "oriented": GaussianDecodeMode.GaussianSh0Oriented}


def listed():
    return [
        # one step of a small interactive demo: launches and host work count
        dict(name="step_1k", kind="step", preset="growing_2d", cloud="disk", batch=1, n=1000),
        # a dense, heavily skewed cloud (an 8-component Gaussian mixture): the largest single step
        dict(name="step_dense", kind="step", preset="c1", cloud="mixture", batch=1, n=200000),
        # the reference's own benchmark size, the steps between two frames
        dict(name="rollout_4k", kind="rollout", preset="c1", cloud="disk", batch=1, n=4096, steps=16, engine="valu"),
        # the headline rollout
        dict(name="rollout_64k", kind="rollout", preset="c1", cloud="disk", batch=1, n=65536, steps=16,
             engine="valu"),
        # 64 independent systems at once on the matrix-core engine
        dict(name="rollout_batch", kind="rollout", preset="c1", cloud="disk", batch=64, n=4096, steps=16,
             engine="mfma"),
        # the 3D preset: 24 channels, 256 hidden units
        dict(name="rollout_3d", kind="rollout", preset="growing_3dgs", cloud="ball", batch=1, n=8192, steps=12,
             engine="valu"),
        # a training batch forward: perception, update MLP, Euler step
        dict(name="forward_2d", kind="forward", preset="growing_2d", cloud="disk", batch=8, n=4001),
        # the same batch backward, and the 3D preset's
        dict(name="adjoint_2d", kind="adjoint", preset="growing_2d", cloud="disk", batch=8, n=4096),
        dict(name="adjoint_3d", kind="adjoint", preset="growing_3dgs", cloud="ball", batch=2, n=8192),
        # the render loss's four particle images
        dict(name="render", kind="render", cloud="shell", n=16384, channels=16, size=64, decode="fixed"),
        # a viewer frame of oriented Gaussians
        dict(name="raster", kind="raster", cloud="shell", n=16384, channels=16, width=1024, height=768,
             decode="oriented"),
        # the 2D frame of the headline rollout
        dict(name="splat", kind="splat", cloud="disk", batch=1, n=65536, size=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "rollout", "rollout", "rollout", "forward", "adjoint", "adjoint", "render",
                       "raster", "splat"])
    if kind == "render":
        return dict(kind=kind, cloud=rng.choice(["shell", "ball"]), n=_log(rng, 1000, 32768),
                    channels=rng.choice([8, 16, 24]), size=rng.randint(48, 200),
                    decode=rng.choice(["fixed", "learned"]))
    if kind == "raster":
        return dict(kind=kind, cloud=rng.choice(["shell", "ball"]), n=_log(rng, 1000, 32768),
                    channels=rng.choice([16, 24]), width=_log(rng, 128, 1280), height=_log(rng, 96, 1024),
                    decode=rng.choice(["fixed", "oriented"]))
    if kind == "splat":
        batch = rng.choice([1, 1, 4, 9])
        return dict(kind=kind, cloud="disk", batch=batch, n=_log(rng, 1000, 131072 // batch),
                    size=_log(rng, 96, 1024 // math.isqrt(batch)))
    preset = rng.choice(["c1", "growing_2d", "texture_2d", "growing_3dgs", "point_mnist", "c4"])
    # the wide-radius presets gather hundreds of neighbours well below the sizes the others run at
    most = 65536 if preset in ("c1", "c4") else 16384
    batch = rng.choice([1, 1, 1, 2, 5, 16])
    case = dict(kind=kind, preset=preset, cloud=CLOUDS[preset], batch=batch, n=_log(rng, 700, max(1400, most // batch)))
    if kind == "adjoint":
        # training clouds: forty neighbours and more in 2D, sixty in 3D, and no thin surface (below that, or there,
        # moment matrices are near singular and no 32-bit adjoint is sharp)
        if preset == "c4":
            case.update(preset="growing_3dgs", cloud="ball")
        least = {"c1": 16000, "texture_2d": 1300, "growing_3dgs": 8192}.get(case["preset"], 4000)
        case.update(batch=rng.randint(1, 4), n=_log(rng, least, 2 * least))
    if kind == "rollout":
        case.update(steps=rng.randint(4, 12), engine=rng.choice(["valu", "mfma"]))
    return case


# ---------------------------------------------------------------- inputs

def _setup(preset):
    """(NpaConfig, HashGridConfig) of a preset."""
    if preset == "c1":
        return config_c1()
    if preset == "c4":  # synthetic.workload("c4")'s model and grid
        model = NpaConfig.growing_3dgs().replace(state_dims=16, hidden_dims=128, eps0=0.04, density_grad=False, alpha=0.5)
        return model, HashGridConfig(3, Boundary.Clamped, HashGridMode.Particle, (32, 32, 32), 0.04, 64)
    return NpaConfig.for_preset(preset)


def _rand(seed, stream, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 16 + stream)
    return torch.rand(*shape, generator=g, device="cuda")


def _randn(seed, stream, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 16 + stream)
    return torch.randn(*shape, generator=g, device="cuda")


def _cloud(cloud, total, seed):
    pos = torch.zeros(total, 4, device="cuda")
    if cloud == "disk":
        u = _rand(seed, 0, total, 2)
        r, a = u[:, 0].sqrt() * DISK_RADIUS, u[:, 1] * (2 * math.pi)
        pos[:, 0], pos[:, 1] = r * a.cos(), r * a.sin()
    elif cloud == "square":
        pos[:, :2] = _rand(seed, 0, total, 2) * 1.999 - 0.9995
    elif cloud == "mixture":  # synthetic.gaussian_mixture's law
        k = (_rand(seed, 0, total) * 8).long().clamp_(max=7)
        sigma = 0.02 * 10.0 ** (k / 7)
        means = _rand(42, 1, 8, 2) * 1.2 - 0.6  # the same eight centres for every seed: their overlap sets the work
        pos[:, :2] = means[k] + sigma[:, None] * _randn(seed, 2, total, 2)
    else:
        v = _randn(seed, 0, total, 3)
        v = v / v.norm(dim=1, keepdim=True)
        if cloud == "ball":
            pos[:, :3] = v * (_rand(seed, 1, total, 1) ** (1.0 / 3.0) * BALL_RADIUS)
        else:
            pos[:, :3] = v * torch.tensor(SHELL, device="cuda")
    return pos


def _weights(cfg, seed, bf16):
    F, H, O = cfg.perception_dims(), cfg.hidden_dims, cfg.update_dims()
    w = (_rand(seed, 4, H * F + O * H) * 2 - 1) * 0.1
    if bf16:  # bf16-valued weights in 32-bit storage
        w = w.bfloat16().float()
    return NpaWeights(w[: H * F].clone(), torch.zeros(H, device="cuda"), w[H * F:].clone(), torch.zeros(O, device="cuda"))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("render", "raster"):
        n = case["n"]
        s = dict(case=case, pos=_cloud(case["cloud"], n, seed), states=_randn(seed, 3, n, case["channels"]) * 0.1)
        if kind == "render":
            s["cfg"] = RenderLossConfig(image_size=case["size"], gaussian_decode_mode=DECODES[case["decode"]])
        else:
            s["cfg"] = GaussianDecodeConfig(mode=DECODES[case["decode"]])
            s["camera"] = RasterCamera.look_at((0.9, 1.2, 2.6), (0.0, 0.0, 0.1), width=case["width"],
                                               height=case["height"], color_mode=RasterColor.Rgb)
        return s
    if kind == "splat":
        total, size = case["batch"] * case["n"], case["size"]
        return dict(case=case, pos=_cloud("disk", total, seed), colors=_rand(seed, 5, total, 3),
                    cfg=Splat2dConfig(image_size=size, sigma=0.004 * (size - 1) / 2, pixel_size=2.0 / size))
    cfg, grid = _setup(case["preset"])
    total, S = case["batch"] * case["n"], cfg.state_dims
    s = dict(case=case, grid=grid, model=NpaModel(cfg, _weights(cfg, seed, case.get("engine") == "mfma")),
             pos=_cloud(case["cloud"], total, seed), states=_randn(seed, 3, total, S) * 0.1)
    if kind == "step" or kind == "forward":
        s["mask"] = (_rand(seed, 6, total) < UPDATE_PROB).float()
    if kind == "rollout":
        s["executor"], s["seed"] = HipAutomataExecutor(), int(seed)
    if kind == "adjoint":
        s["options"] = cfg.perception_options()
        s["fadj"] = _randn(seed, 7, total, s["options"].feature_dims(S, grid.dim)) * 0.1
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "step":
        o = s["model"].step(s["pos"], s["states"], c["batch"], c["n"], s["grid"], DT, s["mask"])
        return [o.next_positions, o.next_states, o.density]
    if kind == "rollout":
        ex = s["executor"]
        st = ex.create_state(s["model"], s["pos"], s["states"], c["batch"], c["n"], s["grid"], DT, UPDATE_PROB, s["seed"])
        st.set_mlp_engine(ENGINES[c["engine"]])
        ex.step_state_many(st, c["steps"])
        out = ex.read_state(st)
        st.close()
        return list(out)
    if kind == "forward":
        m, grid, B, N = s["model"], s["grid"], c["batch"], c["n"]
        S = m.config.state_dims
        p = kernels.perceive_with_options(s["pos"], s["states"], B, N, S, grid, m.config.perception_options())
        dx, ds = m.forward_from_features_with_eps(p.features, grid.eps)
        npos, nst = kernels.euler_step(s["pos"], s["states"], dx, ds, B, N, S, grid, DT, s["mask"])
        return [p.features, p.density, p.blurred_state, p.state_gradient, p.density_gradient, dx, ds, npos, nst]
    if kind == "adjoint":
        o = kernels.perceive_adjoint_with_options(s["pos"], s["states"], c["batch"], c["n"],
                                                  s["model"].config.state_dims, s["grid"], s["options"], s["fadj"])
        return [o.state, o.position]
    if kind == "render":
        col, op, sg, dv = kernels.render_attributes(s["states"], c["channels"], s["cfg"])
        return [col, op, sg, dv, kernels.render_views(s["pos"], col, op, sg, s["cfg"], ALL_VIEWS)]
    if kind == "raster":
        g = kernels.decode_gaussians_3d(s["pos"], s["states"], c["channels"], s["cfg"])
        img = kernels.raster_gaussians_3d(g["position_visibility"], g["spherical_harmonic"], g["rotation"],
                                          g["scale_opacity"], s["camera"])
        return [g["position_visibility"], g["spherical_harmonic"], g["rotation"], g["scale_opacity"], img]
    if c["batch"] == 1:
        return [kernels.splat_particles_2d(s["pos"], s["colors"], s["cfg"])]
    return [kernels.splat_particles_2d_tiled(s["pos"], s["colors"], c["batch"], c["n"], s["cfg"], math.isqrt(c["batch"]))]


# ---------------------------------------------------------------- what a pass cannot do without

def _pairs(case, eps):
    """Expected neighbour pairs of the whole batch, each particle its own neighbour too."""
    n = case["n"]
    share = {"disk": (eps / DISK_RADIUS) ** 2, "square": math.pi * eps * eps / 4.0, "ball": (eps / BALL_RADIUS) ** 3,
             "shell": math.pi * eps * eps / SHELL_AREA, "mixture": 12.6 * eps * eps}[case["cloud"]]
    return case["batch"] * n * (1.0 + (n - 1) * min(1.0, share))


def work(case):
    kind = case["kind"]
    if kind == "splat":
        total, size = case["batch"] * case["n"], case["size"]
        side = 2 * math.ceil(5 * 0.004 * (size - 1) / 2) + 1
        return dict(bytes=total * 28 + case["batch"] * size * size * 16, flops=total * side * side * 16)
    if kind == "render":
        n, S, size = case["n"], case["channels"], case["size"]
        return dict(bytes=n * (16 + 4 * S + 24) + 4 * size * size * 20, flops=4 * n * 27 * 27 * 29)
    if kind == "raster":
        n, S, w, h = case["n"], case["channels"], case["width"], case["height"]
        sigma = 0.02 * h / 2 / math.tan(math.pi / 8) / 2.8
        return dict(bytes=n * (16 + 4 * S + 60) + w * h * 16, flops=n * math.pi * (3 * sigma + 1) ** 2 * 25)
    cfg, grid = _setup(case["preset"])
    S, d, H = cfg.state_dims, grid.dim, cfg.hidden_dims
    F, O = cfg.perception_dims(), cfg.update_dims()
    total, pairs = case["batch"] * case["n"], _pairs(case, grid.eps)
    density = 5 * pairs * (2.9 if d == 2 else 6.4) + 5 * pairs  # tests of the 3^d cells' particles
    second = pairs * (12 + 2 * S + d + S * (1 + 2 * d) + 2 * d * d) + total * (15 + 2 * S * d * d + S * d + S * (3 * d + 23))
    mlp = total * 2 * (F * H + H * O)
    weights = 4 * (F * H + H + H * O + O)
    if kind == "adjoint":
        return dict(bytes=total * (2 * 16 + 8 * S + 4 * F), flops=density + second + pairs * 38 * S)
    if kind == "forward":
        out = F + 1 + S + S * d + (d if cfg.density_grad else 0) + 2 * (4 + S)
        return dict(bytes=total * (16 + 4 * S + 4 + 4 * out) + weights, flops=density + second + mlp)
    step = dict(bytes=total * (2 * 16 + 8 * S + 8) + weights, flops=density + UPDATE_PROB * (second + mlp))
    if kind == "rollout":  # the particles stay resident between the steps
        step["flops"] *= case["steps"]
    return step


# ---------------------------------------------------------------- how far two correct results lie apart

def tolerance(case):
    """About four times what the present code differs by from exact() over the ranges of draw()."""
    kind = case["kind"]
    if kind == "rollout":  # a difference in the last bit grows by up to a half in each step
        return {"rel": min(0.03, 2e-5 * 2.0 ** case["steps"]), "max": 0.99}
    if kind == "adjoint":
        return {"rel": 4e-6, "max": 2e-4}
    if kind == "render":
        return {"rel": 1e-6, "max": 5e-6}
    if kind == "raster":  # a Gaussian's 1/255 and transmittance cuts fall on one side or the other
        return {"rel": 2e-5, "max": 1e-2}
    if kind == "splat":
        return {"rel": 4e-5, "max": 5e-4}
    # a thin surface's and a skewed cloud's moment matrices amplify rounding
    return {"rel": 3e-5, "max": 2e-3} if case["cloud"] in ("shell", "mixture") else {"rel": 4e-6, "max": 2e-4}


# ---------------------------------------------------------------- 64-bit results

def _neighbours(pos, case, grid):
    """(i, j, delta, r2) of every pair within eps, in chunks of whole targets."""
    B, N, eps, d = case["batch"], case["n"], grid.eps, grid.dim
    periodic = grid.boundary == Boundary.Periodic
    p = pos[:, :d]
    ext = torch.tensor([grid.grid_size[a] * eps for a in range(d)], dtype=torch.float64, device=pos.device)
    total = B * N
    c = torch.floor((p + ext / 2 if periodic else p) / eps).long()
    size = torch.tensor(grid.grid_size[:d], device=pos.device)
    if periodic:
        c = c % size
    else:
        c = c - c.amin(0) + 1
        size = c.amax(0) + 2
    stride = torch.cumprod(torch.cat([torch.ones(1, dtype=torch.long, device=pos.device), size]), 0)
    sys_ = torch.arange(total, device=pos.device) // N
    key = sys_ * stride[d] + (c * stride[:d]).sum(1)
    skey, order = torch.sort(key)
    offs = torch.cartesian_prod(*[torch.arange(-1, 2, device=pos.device)] * d)
    lo, cnt = [], []
    for o in offs:
        q = c + o
        if periodic:
            q = q % size
        k = sys_ * stride[d] + (q * stride[:d]).sum(1)
        a, b = torch.searchsorted(skey, k), torch.searchsorted(skey, k, right=True)
        lo.append(a)
        cnt.append(b - a)
    lo, cnt = torch.stack(lo, 1), torch.stack(cnt, 1)
    per = cnt.sum(1).cumsum(0)
    at, chunk = 0, 40_000_000
    while at < total:
        base = int(per[at - 1]) if at else 0
        to = max(at + 1, int(torch.searchsorted(per, base + chunk, right=True)))
        l, n_ = lo[at:to].reshape(-1), cnt[at:to].reshape(-1)
        i = torch.arange(at, to, device=pos.device).repeat_interleave(cnt[at:to].sum(1))
        start = torch.cumsum(n_, 0) - n_
        j = order[torch.arange(len(i), device=pos.device) + (l - start).repeat_interleave(n_)]
        dl = p[j] - p[i]
        if periodic:
            dl = dl - ext * (dl > ext / 2) + ext * (dl < -ext / 2)
        r2 = (dl * dl).sum(1)
        near = r2 < eps * eps
        yield i[near], j[near], dl[near], r2[near]
        at = to


def _gather(v, i, total):
    """Sums of v's rows by target; i ascends."""
    n = torch.bincount(i, minlength=total)
    return torch.segment_reduce(v.reshape(len(v), -1), "sum", lengths=n, axis=0).reshape(total, *v.shape[1:])


def _safe_inverse(m, d):
    ok = torch.linalg.det(m).abs() >= 1e-3
    eye = torch.eye(d, dtype=m.dtype, device=m.device).expand_as(m)
    return torch.where(ok[:, None, None], torch.linalg.inv(torch.where(ok[:, None, None], m, eye)), eye)


def _log_norm(v):
    n = (v.square().sum(-1, keepdim=True) + 1e-12).sqrt()
    return v * (torch.log1p(n) / n)


def _perceive64(pos, st, case, grid, o):
    """features, density, blurred state, state gradient, density gradient; float64 in and out."""
    eps, d, N = grid.eps, grid.dim, case["n"]
    T, S = st.shape
    k6 = 4 / (math.pi * eps ** 8) if d == 2 else 315 / (64 * math.pi * eps ** 9)
    k5 = 10 / (math.pi * eps ** 5) if d == 2 else 15 / (math.pi * eps ** 6)
    zeros = lambda *s: torch.zeros(*s, dtype=torch.float64, device=pos.device)  # noqa: E731
    rho, kept, pairs = zeros(T), [], 0
    for i, j, dl, r2 in _neighbours(pos, case, grid):
        rho = rho + _gather(k6 * (eps * eps - r2) ** 3, i, T)
        pairs += len(i)
        kept.append((i, j, dl, r2))
        if pairs > 30_000_000:  # a dense cloud's pairs are found again rather than held
            kept = None
            break
    if kept is None:
        rho = zeros(T)
        for i, j, dl, r2 in _neighbours(pos, case, grid):
            rho = rho + _gather(k6 * (eps * eps - r2) ** 3, i, T)
    blur, sg, mom, dg = zeros(T, S), zeros(T, S, d), zeros(T, d, d), zeros(T, d)
    for i, j, dl, r2 in (kept if kept is not None else _neighbours(pos, case, grid)):
        vol = 1.0 / rho[j]
        blur = blur + _gather(st[j] * (k6 * (eps * eps - r2) ** 3 * vol)[:, None], i, T)
        other = r2 > 0
        i, j, dl, r2 = i[other], j[other], dl[other], r2[other]
        r = r2.sqrt()
        g1 = dl * (k5 * 3 * (eps - r) ** 2 / r)[:, None]
        g = g1 * (1.0 / rho[j])[:, None]
        sg = sg + _gather((st[j] - st[i])[:, :, None] * g[:, None, :], i, T)
        mom = mom + _gather(dl[:, :, None] * g[:, None, :], i, T)
        dg = dg + _gather(g1, i, T)
    feats = [st, blur]
    if o.state_grad:
        if o.hybrid_state_gradient:
            sg = sg @ _safe_inverse(mom, d)
        sg = sg * (eps / o.eps0 if o.scale_equivariance else 1.0)
        sg = _log_norm(sg) if o.log_norm_grad else sg
        feats.append(sg.reshape(T, S * d))
    if o.density_grad:
        scale = (eps / o.eps0) ** (1 + d) if o.scale_equivariance else 1.0
        dg = dg * (scale / max(N, 1) if o.particle_density_equivariance else scale)
        dg = _log_norm(dg) if o.log_norm_density_grad else dg
        feats.append(dg)
    return torch.cat(feats, 1), rho, blur, sg.reshape(T, S * d), dg


def _mlp64(feats, m, grid):
    cfg = m.config
    w = [t.double() for t in (m.weights.w1, m.weights.b1, m.weights.w2, m.weights.b2)]
    h = torch.relu(feats @ w[0].reshape(cfg.hidden_dims, -1).T + w[1])
    u = h @ w[2].reshape(cfg.update_dims(), -1).T + w[3]
    d = grid.dim
    dx = torch.zeros(len(u), 4, dtype=torch.float64, device=u.device)
    dx[:, :d] = cfg.alpha * u[:, :d] * cfg.motion_eps(grid.eps) / (1 + u[:, :d].norm(dim=1, keepdim=True))
    return dx, u[:, d:]


def _euler64(pos, st, dx, ds, mask, grid):
    p, s = pos + DT * dx * mask[:, None], st + DT * ds * mask[:, None]
    if grid.boundary == Boundary.Periodic:
        for a in range(grid.dim):
            e = grid.grid_size[a] * grid.eps
            p[:, a] = torch.remainder(p[:, a] + e / 2, e) - e / 2
    if grid.dim == 3:
        for ch in (3, 8):
            if ch < s.shape[1] and s.shape[1] > 3:
                s[:, ch] = s[:, ch].clamp(-8.0, 24.0)
    return p, s


def _mask64(case, step, seed):
    """The executor's update mask: an integer hash of particle, step and seed."""
    m32 = 0xFFFFFFFF

    def h(x):
        x = (x ^ 61) ^ (x >> 16)
        x = (x + (x << 3)) & m32
        x = x ^ (x >> 4)
        x = (x * 0x27D4EB2D) & m32
        return x ^ (x >> 15)

    i = torch.arange(case["n"], device="cuda").repeat(case["batch"])
    lane = torch.arange(case["batch"], device="cuda").repeat_interleave(case["n"])
    base = ((seed & m32) ^ (seed >> 32)) ^ ((lane * case["n"]) & m32)
    mixed = h((i ^ h((step + 0x9E3779B9) & m32) ^ base) & m32)
    return ((mixed >> 8).double() / 16777216.0 < UPDATE_PROB).double()


def _footprints64(px, py, sigma, size, floor):
    """(particle, pixel, weight) of each particle's in-image footprint of +-ceil(5 sigma) pixels, weights summing to one,
    in chunks; sigma a tensor."""
    n = len(px)
    radius = torch.ceil(5 * sigma).clamp(min=1).long()
    most = int(radius.max()) if n else 1
    o = torch.arange(-most, most + 1, device=px.device)
    oy, ox = [t.reshape(-1) for t in torch.meshgrid(o, o, indexing="ij")]
    step = max(1, 30_000_000 // len(ox))
    for a in range(0, n, step):
        q = slice(a, a + step)
        bx, by = torch.floor(px[q]), torch.floor(py[q])
        x, y = bx[:, None] + ox, by[:, None] + oy
        live = (x >= 0) & (y >= 0) & (x < size) & (y < size)
        live &= torch.maximum(ox.abs(), oy.abs())[None] <= radius[q][:, None]
        w = torch.exp(-((x - px[q][:, None]) ** 2 + (y - py[q][:, None]) ** 2) / (2 * sigma[q][:, None] ** 2)) * live
        w = w / w.sum(1, keepdim=True).clamp(min=floor)
        k = torch.arange(a, a + len(bx), device=px.device)[:, None].expand_as(w)
        yield k[live], (y * size + x)[live].long(), w[live]


def _splat64(pos, col, cfg):
    size = cfg.image_size
    t = size * cfg.pixel_size / (cfg.hi - cfg.lo)
    to = (pos[:, :2] - cfg.lo) / (cfg.hi - cfg.lo) * (size - 1)
    sigma = torch.full((len(pos),), cfg.sigma * t, dtype=torch.float64, device=pos.device)
    img = torch.zeros(size * size, 4, dtype=torch.float64, device=pos.device)
    src = torch.cat([col, torch.ones_like(col[:, :1])], 1)
    for k, at, w in _footprints64(to[:, 0], (size - 1) - to[:, 1], sigma, size, 1e-8):
        img.index_add_(0, at, src[k] * (w * t * t)[:, None])
    return img


def _render64(s):
    c, cfg, st, pos = s["case"], s["cfg"], s["states"].double(), s["pos"].double()[:, :3]
    n, S, size, ws = c["n"], c["channels"], cfg.image_size, cfg.world_scale
    col = (st[:, S - 3:] + 0.5).clamp(0, 1)
    op = torch.sigmoid(st[:, 8 if S > 8 else 3] + cfg.opacity_logit_bias).clamp(0.001, 0.95)
    dv = torch.zeros(n, dtype=torch.float64, device=st.device)
    sg = torch.full_like(dv, min(max(cfg.sigma, cfg.min_sigma), cfg.max_sigma))
    if c["decode"] == "learned":
        raw = cfg.sigma * torch.exp(st[:, S - 5].clamp(-8, 8))
        sg = raw.clamp(cfg.min_sigma, cfg.max_sigma)
        dv = torch.where((raw > cfg.min_sigma) & (raw < cfg.max_sigma), raw, dv)
    r2, r6, r3 = math.sqrt(2), math.sqrt(6), math.sqrt(3)
    bases = [((1, 0, 0), (0, 1, 0), (0, 0, 1)), ((1, 0, 0), (0, 0, 1), (0, 1, 0)), ((0, 1, 0), (0, 0, 1), (1, 0, 0)),
             ((1 / r2, -1 / r2, 0), (1 / r6, 1 / r6, 2 / r6), (-1 / r3, -1 / r3, 1 / r3))]
    out = torch.zeros(4, size * size, 5, dtype=torch.float64, device=st.device)
    for v, basis in enumerate(bases):
        right, up, fwd = (pos @ torch.tensor(b, dtype=torch.float64, device=st.device) for b in basis)
        depth = (0.5 + 0.5 * fwd / ws).clamp(0, 1)
        src = torch.cat([col, torch.ones_like(col[:, :1]), depth[:, None]], 1) * (op / n)[:, None]
        px, py = (right + ws) / (2 * ws) * (size - 1), (ws - up) / (2 * ws) * (size - 1)
        for k, at, w in _footprints64(px, py, sg, size, 1e-8):
            out[v].index_add_(0, at, src[k] * w[:, None])
    return [col, op, sg, dv, out.reshape(4, size, size, 5)]


def _decode64(s):
    c, cfg, st = s["case"], s["cfg"], s["states"].double()
    n, S = c["n"], c["channels"]
    pv = torch.cat([s["pos"].double()[:, :3], torch.ones(n, 1, dtype=torch.float64, device=st.device)], 1)
    sh = (st[:, S - 3:] + 0.5).clamp(0, 1)
    rot = torch.zeros_like(pv)
    rot[:, 0] = 1
    so = torch.full_like(pv, min(max(cfg.sigma, cfg.min_scale), cfg.max_scale))
    so[:, 3] = min(max(cfg.opacity_scale, cfg.min_opacity), cfg.max_opacity)
    if c["decode"] == "oriented":
        q, t = st[:, S - 7:S - 3], torch.tanh(st[:, S - 11:S - 7] / cfg.max_anisotropy) * cfg.max_anisotropy
        rot = q / q.norm(dim=1, keepdim=True)
        so = torch.cat([(cfg.sigma * torch.exp(t[:, :3])).clamp(cfg.min_scale, cfg.max_scale),
                        (cfg.opacity_scale * torch.exp(t[:, 3:])).clamp(cfg.min_opacity, cfg.max_opacity)], 1)
    return pv, sh[:, None, :], rot, so


def _raster64(pv, sh, rot, so, cam):
    dev, f64 = pv.device, torch.float64
    V = torch.tensor(cam.view, dtype=f64, device=dev).reshape(4, 4)
    W = V[:3, :3] * torch.tensor([[1.0], [-1.0], [-1.0]], dtype=f64, device=dev)
    t = pv[:, :3] @ W.T + V[:3, 3] * torch.tensor([1.0, -1.0, -1.0], dtype=f64, device=dev)
    w, x, y, z = rot.unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y), 2 * (x * y + w * z),
                     1 - 2 * (x * x + z * z), 2 * (y * z - w * x), 2 * (x * z - w * y), 2 * (y * z + w * x),
                     1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)
    M = R * so[:, None, :3]
    tz = t[:, 2]
    lim = [1.3 * max(cam.cx, cam.width - cam.cx) / cam.fx, 1.3 * max(cam.cy, cam.height - cam.cy) / cam.fy]
    J = torch.zeros(len(pv), 2, 3, dtype=f64, device=dev)
    for a, f in enumerate((cam.fx, cam.fy)):
        J[:, a, a] = f / tz
        J[:, a, 2] = -f * (t[:, a] / tz).clamp(-lim[a], lim[a]) / tz
    T = J @ W
    cov = T @ (M @ M.transpose(1, 2)) @ T.transpose(1, 2)
    a, b, c = cov[:, 0, 0] + 0.3, cov[:, 0, 1], cov[:, 1, 1] + 0.3
    det, mid = a * c - b * b, 0.5 * (a + c)
    radius = torch.ceil(3 * (mid + (mid * mid - det).clamp(min=0.1).sqrt()).sqrt())
    mx, my = cam.cx + cam.fx * t[:, 0] / tz, cam.cy + cam.fy * t[:, 1] / tz
    tiles = [-(-cam.width // 16), -(-cam.height // 16)]
    rect = [torch.floor((m + k * radius) / 16) + (k > 0) for m in (mx, my) for k in (-1, 1)]
    live = (tz > cam.near_plane) & (tz <= cam.far_plane)
    order = torch.argsort(torch.where(live, tz, math.inf), stable=True)[: int(live.sum())]
    qa, qb, qc = -0.5 * c / det, b / det, -0.5 * a / det
    img = torch.zeros(cam.height, cam.width, 4, dtype=f64, device=dev)
    g = torch.stack([mx, my, qa, qb, qc, so[:, 3], sh[:, 0, 0], sh[:, 0, 1], sh[:, 0, 2]], 1)[order]
    rect = [r[order] for r in rect]
    for ty in range(tiles[1]):
        row = ((rect[2] <= ty) & (ty < rect[3])).nonzero()[:, 0]
        # the row's items: (Gaussian, tile) for every tile of the rectangle, front to back in each tile
        x0, x1 = rect[0][row].clamp(0, tiles[0]).long(), rect[1][row].clamp(0, tiles[0]).long()
        cnt = (x1 - x0).clamp(min=0)
        who = row.repeat_interleave(cnt)
        tile = torch.arange(len(who), device=dev) - (cnt.cumsum(0) - cnt - x0).repeat_interleave(cnt)
        by_tile = torch.argsort(tile, stable=True)
        who, sizes = who[by_tile], torch.bincount(tile, minlength=tiles[0]).tolist()
        at = 0
        for tx, size in enumerate(sizes):
            k, at = who[at:at + size], at + size
            if not size:
                continue
            ys = torch.arange(ty * 16, min(ty * 16 + 16, cam.height), device=dev)
            xs = torch.arange(tx * 16, min(tx * 16 + 16, cam.width), device=dev)
            e = g[k][:, :, None, None]
            dx, dy = e[:, 0] - (xs + 0.5)[None, None], e[:, 1] - (ys + 0.5)[None, :, None]
            power = e[:, 2] * dx * dx + e[:, 4] * dy * dy + e[:, 3] * dx * dy
            alpha = (e[:, 5] * torch.exp(power)).clamp(max=0.99)
            alpha = torch.where((power > 0) | (alpha < 1 / 255), 0.0, alpha)
            trans = torch.cumprod(1 - alpha, 0)
            drawn = (trans >= 1e-4).cumprod(0)  # the first that would go below ends the pixel
            before = torch.cat([torch.ones_like(trans[:1]), trans[:-1]])
            wgt = alpha * before * drawn
            block = img[ty * 16:ty * 16 + 16, tx * 16:tx * 16 + 16]
            block[..., :3] = (wgt[:, :, :, None] * e[:, 6:9, 0, 0][:, None, None, :]).sum(0)
            block[..., 3] = wgt.sum(0)
    return img


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "render":
        return _render64(s)
    if kind == "raster":
        g = _decode64(s)
        return [*g, _raster64(*g, s["camera"])]
    if kind == "splat":
        pos, col, B, cfg = s["pos"].double(), s["colors"].double(), case["batch"], s["cfg"]
        if B == 1:
            return [_splat64(pos, col, cfg)]
        cols, size = math.isqrt(B), cfg.image_size
        rows = -(-B // cols)
        out = torch.zeros(rows * size, cols * size, 4, dtype=torch.float64, device=pos.device)
        for b in range(B):
            q = slice(b * case["n"], (b + 1) * case["n"])
            y, x = b // cols * size, b % cols * size
            out[y:y + size, x:x + size] = _splat64(pos[q], col[q], cfg).reshape(size, size, 4)
        return [out]
    grid, m = s["grid"], s["model"]
    if _pairs(case, grid.eps) * case.get("steps", 1) > 2.5e9:
        return None
    o = m.config.perception_options()
    pos, st = s["pos"].double(), s["states"].double()
    if kind == "adjoint":
        pos.requires_grad_(True)
        st.requires_grad_(True)
        f = _perceive64(pos, st, case, grid, o)[0]
        f.backward(s["fadj"].double())
        return [st.grad.reshape(-1), pos.grad]
    if kind == "rollout":
        for k in range(case["steps"]):
            f, rho = _perceive64(pos, st, case, grid, o)[:2]
            pos, st = _euler64(pos, st, *_mlp64(f, m, grid), _mask64(case, k, s["seed"]), grid)
        return [pos, st, rho]
    f, rho, blur, sg, dg = _perceive64(pos, st, case, grid, o)
    dx, ds = _mlp64(f, m, grid)
    p, q = _euler64(pos, st, dx, ds, s["mask"].double(), grid)
    if kind == "step":
        return [p, q, rho]
    return [f, rho, blur, sg if o.state_grad else None, dg if o.density_grad else None, dx, ds, p, q]
