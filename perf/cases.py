"""What a user of this framework has it do, as cases to be timed.

Six kinds of work, each through the entry points that a program calls:

  steps    a simulation that stays on the GPU: upload a state, advance it, read it back into device memory
           (fs2d_hip_upload_device, set_sources, step_n, fs2d_hip_download_device), in both sweep orders
  solve    fluid_solver::solve with host arrays, one frame per call, as an interactive program calls it
  batch    many simulations of different sizes advanced together, their states read back to the host
  project  one projection from the multigrid seed to a residual tolerance
  predict  the pressure network's prediction for host arrays
  train    one Adam step of the network on a batch of crops, and its gradients

Sizes, time steps, viscosities, sweep counts and starts are those of the benchmark's workloads (128, 1024 and 4096
cells a side with 20, 40 and 80 sweeps; 256 simulations of sides 64 to 512; 16 crops of 256 x 256; 1024 x 1024
fields) with ragged sizes beside them.  Inputs come from the seed alone.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "fluid-2d_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

NET_PARAMS = os.path.join(PKG, "fs2d_amd", "pressure_net_params.npz")
# (input, output) channels of the network's 15 convolutions, as its parameter vector lays them out
NET_LAYERS = [(16, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
              (192, 64), (64, 64), (96, 32), (32, 32), (48, 16), (16, 16), (16, 16)]
BATCH_SIDES = (64, 96, 128, 192, 256, 384, 512)


def listed():
    return [
        # The interactive size: a closed box that starts at rest, a plume fed by sources at every step, no diffusion.
        {"name": "gs_128_plume", "kind": "steps", "order": "gs", "n": 128, "sweeps": 20, "steps": 20, "dt": 0.1,
         "diffusion": 0.0, "viscosity": 0.0, "start": "plume"},
        # A production run of middle size in the reference's sweep order.
        {"name": "gs_1024", "kind": "steps", "order": "gs", "n": 1024, "sweeps": 40, "steps": 4, "dt": 0.05,
         "diffusion": 1e-5, "viscosity": 1e-6, "start": "vortices"},
        # A ragged grid: no side a multiple of a tile, the reference's default sweep count, sources on.
        {"name": "gs_1531_ragged", "kind": "steps", "order": "gs", "n": 1531, "sweeps": 20, "steps": 3, "dt": 0.05,
         "diffusion": 1e-5, "viscosity": 1e-5, "start": "forced"},
        # The headline: the largest grid whose steps are quoted.
        {"name": "gs_4096", "kind": "steps", "order": "gs", "n": 4096, "sweeps": 80, "steps": 1, "dt": 0.05,
         "diffusion": 1e-5, "viscosity": 1e-6, "start": "vortices"},
        # The Jacobi order on a small ragged grid.
        {"name": "jacobi_201_ragged", "kind": "steps", "order": "jacobi", "n": 201, "sweeps": 20, "steps": 20,
         "dt": 0.1, "diffusion": 1e-5, "viscosity": 1e-5, "start": "vortices"},
        # The Jacobi order at the middle and the headline size.
        {"name": "jacobi_1024", "kind": "steps", "order": "jacobi", "n": 1024, "sweeps": 40, "steps": 10, "dt": 0.05,
         "diffusion": 1e-5, "viscosity": 1e-6, "start": "vortices"},
        {"name": "jacobi_4096", "kind": "steps", "order": "jacobi", "n": 4096, "sweeps": 80, "steps": 2, "dt": 0.05,
         "diffusion": 1e-5, "viscosity": 1e-6, "start": "vortices"},
        # The drop-in call: host arrays in, host arrays out, one frame.
        {"name": "solve_host_254", "kind": "solve", "n": 254, "sweeps": 20, "dt": 0.05, "diffusion": 1e-5,
         "viscosity": 1e-5},
        # The batched workload, states read back every 40 steps.
        {"name": "batch_256_sims", "kind": "batch", "count": 256, "side_max": 512, "steps": 40, "shapes": 1},
        # A projection to 1 % of the divergence by multigrid.
        {"name": "project_mg_1024", "kind": "project", "n": 1024, "tol": 0.01},
        # The learned guess for one field, and one training step of the trainer's shape.
        {"name": "predict_1024", "kind": "predict", "batch": 1, "h": 1024, "w": 1024},
        {"name": "train_16x256", "kind": "train", "batch": 16, "h": 256, "w": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps"] * 6 + ["solve", "batch", "project", "predict", "train", "train"])
    if kind == "steps":
        n = _log_int(rng, 32, 4000)
        sweeps = rng.choice([rng.randint(16, 32), 20, 40, rng.randint(33, 80)])
        steps = max(1, min(20, int(6e8 / (n * n * sweeps))))
        return {"kind": kind, "order": rng.choice(["gs", "jacobi"]), "n": n, "sweeps": sweeps, "steps": steps,
                "dt": round(rng.uniform(0.02, 0.1), 4), "diffusion": rng.choice([0.0, 1e-6, 1e-5]),
                "viscosity": rng.choice([0.0, 1e-6, 1e-5]), "start": rng.choice(["vortices", "forced", "plume"])}
    if kind == "solve":
        return {"kind": kind, "n": _log_int(rng, 48, 900), "sweeps": rng.randint(16, 40),
                "dt": round(rng.uniform(0.02, 0.1), 4), "diffusion": 1e-5, "viscosity": rng.choice([0.0, 1e-5])}
    if kind == "batch":
        return {"kind": kind, "count": _log_int(rng, 8, 200), "side_max": rng.choice(BATCH_SIDES[2:]),
                "steps": rng.randint(10, 30), "shapes": rng.randint(2, 1 << 20)}
    if kind == "project":
        return {"kind": kind, "n": rng.choice([32, 8, 4]) * rng.randint(16, 60), "tol": rng.choice([0.05, 0.02, 0.01])}
    if kind == "predict":
        return {"kind": kind, "batch": rng.randint(1, 4), "h": 32 * rng.randint(2, 32), "w": 32 * rng.randint(2, 32)}
    return {"kind": kind, "batch": _log_int(rng, 1, 16), "h": 32 * rng.randint(2, 8), "w": 32 * rng.randint(2, 8)}


# ---- inputs -------------------------------------------------------------------------------------
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def _rng(seed, salt=0):
    return torch.Generator(device=DEVICE).manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEVICE, dtype=torch.float64)


def _smooth(x, sigma):
    """Separable Gaussian blur of the last two dimensions, truncated at 4 sigma, edges clamped."""
    r = int(4 * sigma)
    w = [math.exp(-0.5 * (k / sigma) ** 2) for k in range(-r, r + 1)]
    for dim in (-1, -2):
        n = x.shape[dim]
        at = torch.arange(-r, n + r, device=x.device).clamp(0, n - 1)
        p = x.index_select(dim, at)
        x = sum(p.narrow(dim, k, n) * (wk / sum(w)) for k, wk in enumerate(w))
    return x


def _ring(x, mode):
    """The boundary ring of a field [.., R, R], in place (0 continuous, 1 u, 2 v)."""
    tb, lr = (-1.0 if mode == 2 else 1.0), (-1.0 if mode == 1 else 1.0)
    x[..., 0, 1:-1] = tb * x[..., 1, 1:-1]
    x[..., -1, 1:-1] = tb * x[..., -2, 1:-1]
    x[..., 1:-1, 0] = lr * x[..., 1:-1, 1]
    x[..., 1:-1, -1] = lr * x[..., 1:-1, -2]
    for i, a in ((0, 1), (-1, -2)):
        for j, b in ((0, 1), (-1, -2)):
            x[..., i, j] = 0.5 * (x[..., i, b] + x[..., a, j])
    return x


def _vortices(g, n, count, reference):
    """Density, u and v of `count` Gaussian vortices (radii 10 to 40 cells at side `reference`, scaled with the side;
    at most 2 cells per unit time) over smoothed noise, rings set, float32."""
    R = n + 2
    i = torch.arange(R, device=DEVICE, dtype=torch.float64)
    c = 1.0 + _uniform(g, 2, count, 1) * (n - 1)
    r = (10.0 + 30.0 * _uniform(g, count, 1)) * (n / reference)
    s = torch.randn(count, 1, generator=g, device=DEVICE, dtype=torch.float64) / r ** 2
    di, dj = i - c[0], i - c[1]
    ei, ej = torch.exp(-di ** 2 / (2 * r ** 2)), torch.exp(-dj ** 2 / (2 * r ** 2))
    u = -(s * di * ei).t() @ ej
    v = (s * ei).t() @ (dj * ej)
    speed = torch.sqrt(u ** 2 + v ** 2)[1:-1, 1:-1].max()
    rho = torch.zeros(R, R, device=DEVICE, dtype=torch.float64)
    rho[1:-1, 1:-1] = _smooth(_uniform(g, n, n), 4.0)
    return tuple(_ring(x.float(), m) for x, m in ((rho, 0), (u * (2.0 / R / speed), 1), (v * (2.0 / R / speed), 2)))


def _plume(g, n):
    """Sources of density 100 and upward velocity 5 over a disc of radius 8 cells (n / 16 on smaller grids) near the centre."""
    R = n + 2
    c = (R - 1) / 2.0 + (_uniform(g, 2) - 0.5) * (n / 8.0)
    i = torch.arange(R, device=DEVICE, dtype=torch.float64)
    disc = ((i[:, None] - c[0]) ** 2 + (i[None, :] - c[1]) ** 2 <= min(8.0, n / 16.0) ** 2).float()
    disc[0] = disc[-1] = 0.0
    disc[:, 0] = disc[:, -1] = 0.0
    return 100.0 * disc, torch.zeros_like(disc), -5.0 * disc


def _stirring(g, n):
    """Smooth sources over the whole grid: density everywhere, a force field of a few tenths of a cell per unit time."""
    R = n + 2
    a = torch.zeros(3, R, R, device=DEVICE, dtype=torch.float64)
    a[:, 1:-1, 1:-1] = _smooth(_uniform(g, 3, n, n) - 0.5, 6.0)
    a[0] = (a[0] + 0.5) * 0.1
    a[0][0] = a[0][-1] = 0.0
    a[0][:, 0] = a[0][:, -1] = 0.0
    a[1:] *= 1.0 / (R * a[1:].std())
    return tuple(x.float().contiguous() for x in a)


def _inputs(case, seed):
    """(density, u, v, density source, u source, v source) as float32 on the device; sources None where there are none."""
    g, n = _rng(seed, case["n"]), case["n"]
    start = case.get("start", "forced")
    if start == "plume":
        z = torch.zeros(3, n + 2, n + 2, device=DEVICE)
        return (*z, *_plume(g, n))
    state = _vortices(g, n, 64, 1024)
    return (*state, *(_stirring(g, n) if start == "forced" else (None, None, None)))


def _batch_sims(case):
    """[(rows, sweeps, dt, diffusion, viscosity)]: sides and sweep counts drawn uniformly, dt in [0.02, 0.1]."""
    g = torch.Generator().manual_seed(case["shapes"])
    sides = [s for s in BATCH_SIDES if s <= case["side_max"]]
    a, b, c = torch.rand(3, case["count"], generator=g, dtype=torch.float64)
    return [(sides[int(x * len(sides))] + 2, 20 if y < 0.5 else 40, float(np.float32(0.02 + 0.08 * float(z))), 1e-5, 1e-6)
            for x, y, z in zip(a, b, c)]


def _poisson(d):
    """p with 4 p - (its neighbours) = d - mean(d), mirrored at the edges, mean 0: by the FFT of the mirrored field."""
    h, w = d.shape[-2:]
    e = torch.cat([d, d.flip(-1)], -1)
    e = torch.cat([e, e.flip(-2)], -2)
    k = 2 - 2 * torch.cos(math.pi * torch.arange(2 * h, device=d.device, dtype=torch.float64) / h)
    m = 2 - 2 * torch.cos(math.pi * torch.arange(w + 1, device=d.device, dtype=torch.float64) / w)
    lam = k[:, None] + m[None, :]
    lam[0, 0] = 1.0
    f = torch.fft.rfft2(e) / lam
    f[..., 0, 0] = 0.0
    return torch.fft.irfft2(f, s=(2 * h, 2 * w))[..., :h, :w]


def _net_fields(case, seed):
    """Divergence, previous pressure and converged pressure (n, h, w): the pressure of a smooth divergence, and the
    pressure of a step before (most of it, and some of another)."""
    g = _rng(seed, 17)
    d = _smooth(_uniform(g, 2, case["batch"], case["h"], case["w"]) - 0.5, 3.0) * 1e-3
    p = _poisson(d)
    return d[0].float(), (0.9 * p[0] + 0.2 * p[1]).float(), p[0].float()


def _net_start(seed):
    """He-initialised parameters; the padded channels' (input 2 to 15 of the first layer, output 1 to 15 of the last) zero."""
    g = _rng(seed, 29)
    out = []
    for k, (cin, cout) in enumerate(NET_LAYERS):
        real = 2 if k == 0 else cin
        w = torch.randn(9, cout, cin, generator=g, device=DEVICE, dtype=torch.float64) * math.sqrt(2.0 / (9 * real))
        if k == 0:
            w[:, :, 2:] = 0.0
        if k == len(NET_LAYERS) - 1:
            w[:, 1:] = 0.0
        out += [w.reshape(-1), torch.zeros(cout, device=DEVICE, dtype=torch.float64)]
    return torch.cat(out).float()


def _velocity_to_project(case, seed):
    """A velocity as a step's first projection gets it after strong forcing: vortices and a divergent push."""
    g = _rng(seed, 31)
    _, u, v = _vortices(g, case["n"], 64, 1024)
    _, fu, fv = _stirring(g, case["n"])
    return _ring(u + fu, 1), _ring(v + fv, 2)


# ---- the program's own objects --------------------------------------------------------------------
_solvers, _nets = {}, {}


def _solver(n, sweeps, order):
    """A program keeps one solver for a grid and gives it new states."""
    import fs2d_amd

    key = (n, sweeps, order)
    if key not in _solvers:
        while len(_solvers) >= 4:
            _solvers.pop(next(iter(_solvers))).close()
        _solvers[key] = fs2d_amd.Solver(n + 2, diffuse_iterations=sweeps, pressure_iterations=sweeps,
                                        order=fs2d_amd.GS_LEX if order == "gs" else fs2d_amd.JACOBI)
    return key


def _handle(key):
    s = _solvers.get(key)
    if s is None:
        s = _solvers[_solver(*key)]
    return s


def _check(rc):
    if rc != 0:
        raise RuntimeError("fs2d call failed (%d)" % rc)


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


def prepare(case, seed):
    import fs2d_amd
    from fs2d_amd import pressure_net as PN

    kind = case["kind"]
    s = {"case": case}
    if kind == "steps":
        x = _inputs(case, seed)
        s["in"] = [t.contiguous() for t in x[:3]]
        s["sources"] = None if x[3] is None else [_host(t) for t in x[3:]]
        s["out"] = [torch.empty_like(t) for t in s["in"]]
        s["solver"] = _solver(case["n"], case["sweeps"], case["order"])
        _handle(s["solver"]).set_sources(None, None, None)
    elif kind == "solve":
        x = [_host(t) for t in _inputs(case, seed)]
        s["in"], s["sources"], s["out"] = x[:3], x[3:], [np.empty_like(a) for a in x[:3]]
        s["solver"] = _solver(case["n"], case["sweeps"], "gs")
    elif kind == "batch":
        sims = _batch_sims(case)
        b = s["batch"] = fs2d_amd.Batch(sims)
        for k, sim in enumerate(sims):
            b.upload(k, *(_host(t) for t in _vortices(_rng(seed, k), sim[0] - 2, 16, 256)))
        cells = sum(sim[0] ** 2 for sim in sims)
        s["out"] = np.zeros((3, cells), np.float32)
        at = np.cumsum([0] + [sim[0] ** 2 for sim in sims])
        s["to"] = [[s["out"][f].ctypes.data + 4 * int(a) for f in range(3)] for a in at[:-1]]
    elif kind == "project":
        s["in"] = [t.contiguous() for t in _velocity_to_project(case, seed)]
        s["rho"] = torch.zeros_like(s["in"][0])
        s["out"] = [torch.empty_like(t) for t in s["in"]]
        s["solver"] = _solver(case["n"], 20, "jacobi")
    elif kind == "predict":
        s["in"] = [_host(t) for t in _net_fields(case, seed)[:2]]
        if "trained" not in _nets:
            _nets["trained"] = PN.PressureNet()
            _nets["trained"].load(NET_PARAMS)
        s["net"] = _nets["trained"]
    else:
        s["in"] = [_host(t) for t in _net_fields(case, seed)]
        s["net"] = PN.PressureNet()
        s["net"].set_params(_host(_net_start(seed)))
    if torch.cuda.is_available():
        torch.cuda.synchronize()  # the solver's stream is its own: the inputs are there before it reads them
    return s


def run(s):
    import fs2d_amd

    case, kind = s["case"], s["case"]["kind"]
    if kind == "steps":
        L, h = fs2d_amd.library(), _handle(s["solver"])
        _check(L.fs2d_hip_upload_device(h._h, *(t.data_ptr() for t in s["in"])))
        if s["sources"] is not None:
            h.set_sources(*s["sources"])
        h.step_n(case["steps"], case["diffusion"], case["viscosity"], case["dt"])
        _check(L.fs2d_hip_download_device(h._h, *(t.data_ptr() for t in s["out"])))
        return s["out"]
    if kind == "solve":
        rho, u, v = s["out"]
        for a, b in zip(s["out"], s["in"]):
            np.copyto(a, b)  # each call starts from this frame's state
        rs, us, vs = s["sources"]
        _handle(s["solver"]).solve(rho, rs, case["diffusion"], u, v, us, vs, case["viscosity"], case["dt"])
        return s["out"]
    if kind == "batch":
        L, b = fs2d_amd.library(), s["batch"]
        b.step_n(case["steps"])
        for k, to in enumerate(s["to"]):
            _check(L.fs2d_hip_batch_download(b._h, k, *to))
        return s["out"]
    if kind == "project":
        from fs2d_amd import pressure_net as PN

        L, h = fs2d_amd.library(), _handle(s["solver"])
        _check(L.fs2d_hip_upload_device(h._h, s["rho"].data_ptr(), *(t.data_ptr() for t in s["in"])))
        sweeps = PN.seeded_projection(h, None, 3, case["tol"], 64, 16, False)[0]
        _check(L.fs2d_hip_download_device(h._h, None, *(t.data_ptr() for t in s["out"])))
        return {"velocity": s["out"], "pressure": h.pressure(), "sweeps": sweeps}
    if kind == "predict":
        return s["net"].predict(*s["in"])
    loss = s["net"].train_step(*s["in"], 1e-3)
    return {"loss": loss, "grads": s["net"].grads()}


# ---- the work that cannot be left out ---------------------------------------------------------------
def _step_flops(n, kd, kp):
    # a diffuse sweep is 4 additions, a product and a quotient, a pressure sweep 4 additions and a product; about 90
    # more for the sources, the scatter, the gather, two divergences and two gradients
    return n * n * (3 * 6 * kd + 2 * 5 * kp + 90)


def work(case):
    kind = case["kind"]
    if kind in ("steps", "solve"):
        R, steps = case["n"] + 2, case.get("steps", 1)
        sources = kind == "solve" or case["start"] != "vortices"
        return {"bytes": R * R * 4 * (9 if sources else 6), "flops": steps * _step_flops(case["n"], case["sweeps"], case["sweeps"])}
    if kind == "batch":
        sims = _batch_sims(case)
        return {"bytes": sum(24 * s[0] ** 2 for s in sims),
                "flops": case["steps"] * sum(_step_flops(s[0] - 2, s[1], s[1]) for s in sims)}
    if kind == "project":
        # one V(2,2) cycle at least: 4 sweeps, a restriction and a correction, over 4/3 of the cells; velocity in and
        # out, pressure out
        n = case["n"]
        return {"bytes": 20 * (n + 2) ** 2, "flops": n * n * (4 * 8 + 12 + 9) * 4 / 3 + 25 * n * n}
    cells = case["batch"] * case["h"] * case["w"]
    scale = [1, 1, 4, 4, 16, 16, 64, 64, 16, 16, 4, 4, 1, 1, 1]
    real = [(2, 16)] + NET_LAYERS[1:-1] + [(16, 1)]
    macs = sum(9 * a * b * cells / f for (a, b), f in zip(real, scale))
    params = 4 * sum(9 * a * b + b for a, b in NET_LAYERS)
    if kind == "predict":
        return {"bytes": 12 * cells + params / 2, "flops": 2 * macs}
    return {"bytes": 12 * cells + 8 * params, "flops": 6 * macs}


# ---- the same in 64 bits ----------------------------------------------------------------------------
def _column(x):
    return torch.as_tensor(x, dtype=torch.float64, device=DEVICE).reshape(-1, 1, 1)


def _relax_jacobi(x, b, a, denom, modes, sweeps):
    for _ in range(sweeps):
        s = x[:, :-2, 1:-1] + x[:, 2:, 1:-1] + x[:, 1:-1, :-2] + x[:, 1:-1, 2:]
        x[:, 1:-1, 1:-1] = (b[:, 1:-1, 1:-1] + a * s) / denom
        _ring_modes(x, modes)
    return x


def _ring_modes(x, modes):
    for m in sorted(set(modes)):
        if all(k == m for k in modes):
            _ring(x, m)
        else:
            for k, mode in enumerate(modes):
                if mode == m:
                    _ring(x[k], m)
    return x


def _relax_gs(x, b, a, denom, modes, sweeps):
    """In-place lexicographic sweeps.  Cell (i, j) of sweep k depends on hyperplanes i + j + 2 k before its own only, so
    all cells of a hyperplane are relaxed together; fields are held skewed, Y[s, i] = x[i, s - i], so that one sweep's
    cells of a hyperplane are a row and those of all sweeps every second row."""
    B, R, _ = x.shape
    n = R - 2
    i = torch.arange(R, device=x.device)

    def skew(f):
        Y = torch.zeros(B, 2 * R, R, dtype=f.dtype, device=f.device)
        ii, jj = torch.meshgrid(i, i, indexing="ij")
        Y[:, ii + jj, ii] = f
        return Y

    X, Z = skew(x), skew(b)
    rows = torch.arange(2 * R, device=x.device)
    inside = ((rows[:, None] - i >= 1) & (rows[:, None] - i <= n) & (i >= 1) & (i <= n))[:, 1:n + 1]
    tb = _column([-1.0 if m == 2 else 1.0 for m in modes])[:, :, 0]
    lr = _column([-1.0 if m == 1 else 1.0 for m in modes])[:, :, 0]
    for t in range(2, 2 * n + 2 * (sweeps - 1) + 1):
        lo = max(2, t - 2 * (sweeps - 1))
        lo += (t - lo) & 1
        hi = min(2 * n, t)
        hi -= (t - hi) & 1
        if lo > hi:
            continue
        here, up, down = slice(lo, hi + 1, 2), slice(lo - 1, hi, 2), slice(lo + 1, hi + 2, 2)
        s = X[:, up, 0:n] + X[:, down, 2:n + 2] + X[:, up, 1:n + 1] + X[:, down, 1:n + 1]
        new = torch.where(inside[here], (Z[:, here, 1:n + 1] + a * s) / denom, X[:, here, 1:n + 1])
        X[:, here, 1:n + 1] = new
        # rings: the cells (1, j), (n, j), (i, 1) and (i, n) of these rows
        e = min(hi, n + 1)  # rows with a cell in the first row and column: s - 1 <= n
        e -= (e - lo) & 1
        if e >= lo:
            c = (e - lo) // 2 + 1
            r = rows[lo - 1:e:2]
            X[:, lo - 1:e:2, 0] = tb * new[:, :c, 0]
            X[:, r, r] = lr * X[:, r + 1, r]
        f = max(lo, n + 1)
        f += (f - lo) & 1
        if f <= hi:
            c = (f - lo) // 2
            r = rows[f:hi + 1:2]
            X[:, f + 1:hi + 2:2, n + 1] = tb * new[:, c:, n - 1]
            X[:, r + 1, r - n] = lr * X[:, r, r - n]
    ii, jj = torch.meshgrid(i, i, indexing="ij")
    x.copy_(X[:, ii + jj, ii])
    return _ring_modes(x, modes)


def _relax(order):
    return _relax_gs if order == "gs" else _relax_jacobi


def _project(u, v, sweeps, order):
    B, R, _ = u.shape
    h = 1.0 / R
    d, p = torch.zeros_like(u), torch.zeros_like(u)
    d[:, 1:-1, 1:-1] = -0.5 * h * (u[:, 1:-1, 2:] - u[:, 1:-1, :-2] + v[:, 2:, 1:-1] - v[:, :-2, 1:-1])
    _relax(order)(p, d, 1.0, 4.0, [0] * B, sweeps)
    _subtract_gradient(u, v, p)
    return p


def _subtract_gradient(u, v, p):
    R = u.shape[-1]
    u[..., 1:-1, 1:-1] -= 0.5 * (p[..., 1:-1, 2:] - p[..., 1:-1, :-2]) * R
    v[..., 1:-1, 1:-1] -= 0.5 * (p[..., 2:, 1:-1] - p[..., :-2, 1:-1]) * R
    _ring(u, 1)
    _ring(v, 2)


def _scatter(rho, u, v, dt0):
    B, R, _ = rho.shape
    k = torch.arange(1, R - 1, device=rho.device, dtype=torch.float64)
    x = k[None, None, :] + dt0 * u[:, 1:-1, 1:-1]
    y = k[None, :, None] + dt0 * v[:, 1:-1, 1:-1]
    ok = (x >= 0.5) & (x <= R - 1.5) & (y >= 0.5) & (y <= R - 1.5)
    b = torch.arange(B, device=rho.device).reshape(-1, 1, 1).expand_as(ok)[ok]
    x, y, q = x[ok], y[ok], rho[:, 1:-1, 1:-1][ok]
    j, i = x.long(), y.long()
    fx, fy = x - j, y - i
    out = torch.zeros(B * R * R, dtype=torch.float64, device=rho.device)
    at = (b * R + i) * R + j
    for off, w in ((0, (1 - fx) * (1 - fy)), (R, (1 - fx) * fy), (1, fx * (1 - fy)), (R + 1, fx * fy)):
        out.index_add_(0, at + off, w * q)
    return _ring(out.reshape(B, R, R), 0)


def _gather(u, v, dt0):
    B, R, _ = u.shape
    k = torch.arange(1, R - 1, device=u.device, dtype=torch.float64)
    x = (k[None, None, :] - dt0 * u[:, 1:-1, 1:-1]).clamp(1.5, R - 1.5)
    y = (k[None, :, None] - dt0 * v[:, 1:-1, 1:-1]).clamp(1.5, R - 1.5)
    j, i = x.long(), y.long()
    fx, fy = x - j, y - i
    at = (torch.arange(B, device=u.device).reshape(-1, 1, 1) * R + i) * R + j
    out = []
    for f, mode in ((u, 1), (v, 2)):
        q, r = f.reshape(-1), f.clone()
        r[:, 1:-1, 1:-1] = (1 - fy) * ((1 - fx) * q[at] + fx * q[at + 1]) + fy * ((1 - fx) * q[at + R] + fx * q[at + R + 1])
        out.append(_ring(r, mode))
    return out


def _step(rho, u, v, sources, diff, visc, dt, sweeps, order):
    """One step of [B, R, R] fields in float64; dt [B, 1, 1]."""
    B, R, _ = rho.shape
    dt0 = R * dt
    if sources is not None:
        for x, s in zip((rho, u, v), sources):
            x[:, 1:-1, 1:-1] += dt * s[1:-1, 1:-1]
        # the density moves with the velocity before its sources are added
    old_u, old_v = (u, v) if sources is None else (u - 0, v - 0)
    if sources is not None:
        old_u[:, 1:-1, 1:-1] -= dt * sources[1][1:-1, 1:-1]
        old_v[:, 1:-1, 1:-1] -= dt * sources[2][1:-1, 1:-1]
    x = torch.cat([rho, u, v])
    a = torch.cat([(dt * R * R * diff).expand(B, 1, 1), (dt * R * R * visc).expand(2 * B, 1, 1) if B == 1
                   else torch.cat([dt * R * R * visc] * 2)])
    _relax(order)(x, x.clone(), a, 1 + 4 * a, [0] * B + [1] * B + [2] * B, sweeps)
    rho, u, v = x[:B], x[B:2 * B].clone(), x[2 * B:].clone()
    rho = _scatter(rho, old_u, old_v, dt0)
    _project(u, v, sweeps, order)
    u, v = _gather(u, v, dt0)
    _project(u, v, sweeps, order)
    return rho, u, v


def _exact_steps(case, seed):
    x = [None if t is None else t.double() for t in _inputs(case, seed)]
    f = [t[None].clone() for t in x[:3]]
    dt = _column(float(np.float32(case["dt"])))
    for _ in range(case.get("steps", 1)):
        f = _step(*f, None if x[3] is None else x[3:], float(np.float32(case["diffusion"])),
                  float(np.float32(case["viscosity"])), dt, case["sweeps"], case.get("order", "gs"))
    return [t[0] for t in f]


def _exact_batch(case, seed):
    sims = _batch_sims(case)
    got = [None] * len(sims)
    for key in sorted({(s[0], s[1]) for s in sims}):
        which = [k for k, s in enumerate(sims) if (s[0], s[1]) == key]
        f = [torch.stack(t).double() for t in zip(*(_vortices(_rng(seed, k), key[0] - 2, 16, 256) for k in which))]
        dt = _column([sims[k][2] for k in which])
        diff, visc = float(np.float32(1e-5)), float(np.float32(1e-6))
        for _ in range(case["steps"]):
            f = _step(*f, None, diff, visc, dt, key[1], "jacobi")
        for q, k in enumerate(which):
            got[k] = [t[q].reshape(-1) for t in f]
    return torch.stack([torch.cat([g[k] for g in got]) for k in range(3)])


def _residual(p, b):
    r = torch.zeros_like(p)
    r[1:-1, 1:-1] = b[1:-1, 1:-1] - (4 * p[1:-1, 1:-1] - p[:-2, 1:-1] - p[2:, 1:-1] - p[1:-1, :-2] - p[1:-1, 2:])
    return r


def _v_cycle(p, b):
    n = p.shape[0] - 2

    def smooth(count):
        for _ in range(count):
            p[1:-1, 1:-1] += 0.8 * 0.25 * _residual(p, b)[1:-1, 1:-1]
            _ring(p, 0)

    if n % 2 or n // 2 < 4:
        return smooth(min(4096, max(64, n * n)))
    smooth(2)
    r = _residual(p, b)[1:-1, 1:-1]
    bc = torch.zeros(n // 2 + 2, n // 2 + 2, dtype=p.dtype, device=p.device)
    bc[1:-1, 1:-1] = r[::2, ::2] + r[::2, 1::2] + r[1::2, ::2] + r[1::2, 1::2]
    c = torch.zeros_like(bc)
    _v_cycle(c, bc)
    i = torch.arange(1, n + 1, device=p.device)
    near = (i + 1) // 2
    far = torch.where(i % 2 == 1, near - 1, near + 1)
    rows = 0.75 * c[near] + 0.25 * c[far]
    p[1:-1, 1:-1] += 0.75 * rows[:, near] + 0.25 * rows[:, far]
    _ring(p, 0)
    smooth(2)


def _exact_project(case, seed):
    u, v = (t.double() for t in _velocity_to_project(case, seed))
    n = case["n"]
    d, p = torch.zeros_like(u), torch.zeros_like(u)
    d[1:-1, 1:-1] = -0.5 / (n + 2) * (u[1:-1, 2:] - u[1:-1, :-2] + v[2:, 1:-1] - v[:-2, 1:-1])
    for _ in range(30):
        _v_cycle(p, d)
        if float(_residual(p, d).norm() / d.norm()) <= case["tol"]:
            break
    _subtract_gradient(u, v, p)
    return {"velocity": [u, v], "pressure": p, "sweeps": None}


def _convolve(x, w, b):
    """3 x 3 convolution of [N, H, W, Cin] by w [9, Cout, Cin] as nine products of matrices."""
    N, H, W, C = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    out = sum(p[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(-1, C) @ w[t].t() for t in range(9))
    return (out + b).reshape(N, H, W, -1)


def _network(params, d, prev):
    """The network's prediction (divided by each sample's scale) and the scales."""
    layers, at = [], 0
    for cin, cout in NET_LAYERS:
        w = params[at:at + 9 * cin * cout].reshape(9, cout, cin)
        at += 9 * cin * cout
        layers.append((w, params[at:at + cout]))
        at += cout
    rms = prev.square().mean((1, 2)).sqrt()
    rms_d = d.square().mean((1, 2)).sqrt()
    s = torch.where(rms > 0, rms, torch.where(rms_d > 0, rms_d, torch.ones_like(rms)))[:, None, None]
    x = torch.zeros(*d.shape, 16, dtype=d.dtype, device=d.device)
    x[..., 0], x[..., 1] = d / s, prev / s

    def conv(t, k):
        y = _convolve(t, *layers[k])
        return y if k == 14 else torch.relu(y)

    def pool(t):
        return 0.25 * (t[:, ::2, ::2] + t[:, ::2, 1::2] + t[:, 1::2, ::2] + t[:, 1::2, 1::2])

    def up(t):
        for dim in (1, 2):
            n = t.shape[dim]
            at = torch.arange(n, device=t.device)
            lo, hi = t.index_select(dim, (at - 1).clamp(min=0)), t.index_select(dim, (at + 1).clamp(max=n - 1))
            shape = list(t.shape)
            shape[dim] *= 2
            t = torch.stack([0.25 * lo + 0.75 * t, 0.75 * t + 0.25 * hi], dim + 1).reshape(shape)
        return t

    e1 = conv(conv(x, 0), 1)
    e2 = conv(conv(pool(e1), 2), 3)
    e3 = conv(conv(pool(e2), 4), 5)
    e4 = conv(conv(pool(e3), 6), 7)
    d3 = conv(conv(torch.cat([up(e4), e3], 3), 8), 9)
    d2 = conv(conv(torch.cat([up(d3), e2], 3), 10), 11)
    d1 = conv(conv(torch.cat([up(d2), e1], 3), 12), 13)
    return conv(d1, 14)[..., 0] + prev / s, s


def exact(case, seed):
    kind = case["kind"]
    if kind in ("steps", "solve"):
        return _exact_steps(case, seed)
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "project":
        return _exact_project(case, seed)
    d, prev, target = (t.double() for t in _net_fields(case, seed))
    if kind == "predict":
        with np.load(NET_PARAMS, allow_pickle=False) as z, torch.no_grad():
            pred, s = _network(torch.tensor(z["params"], device=DEVICE).double(), d, prev)
        return pred * s
    params = _net_start(seed).double().requires_grad_(True)
    pred, s = _network(params, d, prev)
    loss = (pred - target / s).square().mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grads": params.grad}
