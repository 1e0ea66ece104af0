"""The work that a program using this package has it do, as timed cases.

Every case goes through the package's public entry points, on inputs made
from a seed: the likelihood of one coefficient vector and of many, templates
built from isochrones in batches and one at a time, many uneven fits
evaluated together, the template network trained and evaluated, and a mock
population sampled, observed and binned.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import __graft_entry__

sfh = __graft_entry__.load_package()
from sfh_amd import mock, surrogate, synth  # noqa: E402


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one fg! as fit_templates' host optimiser calls it hundreds of times on
        # the 50-template grid (75 x 100 bins): host vectors in and out
        {"name": "fg_50x7500", "kind": "fg", "T": 50, "nx": 75, "ny": 100, "host": True},
        # one fg! of the largest grid on device buffers (a sampler on the GPU)
        {"name": "fg_700x60000", "kind": "fg", "T": 700, "nx": 200, "ny": 300, "host": False},
        # an ensemble of 4096 walkers, log-likelihood to FP64 accuracy and gradient
        {"name": "walkers_4096_f64", "kind": "walkers", "T": 700, "nx": 200, "ny": 300, "B": 4096,
         "precision": "f64", "grad": True},
        # a few dozen HMC chains stepped together
        {"name": "chains_24_f64", "kind": "walkers", "T": 700, "nx": 200, "ny": 300, "B": 24,
         "precision": "f64", "grad": True},
        # a middle-sized ensemble in the split-BF16 form, ragged in every size
        {"name": "walkers_384_bf16x2", "kind": "walkers", "T": 301, "nx": 117, "ny": 171, "B": 387,
         "precision": "bf16x2", "grad": True},
        # the 70 x 10 (age, metallicity) grid of templates, 200 x 300 bins, from
        # 2000-point isochrones with a colour-magnitude correlation
        {"name": "templates_700", "kind": "templates", "n": 700, "nx": 200, "ny": 300, "points": 2000,
         "correlation": 0.6, "filters": 2, "mmax": 120.0},
        # the 10 x 5 grid of templates, 75 x 100 bins, from 500-point isochrones
        {"name": "templates_50", "kind": "templates", "n": 50, "nx": 75, "ny": 100, "points": 500,
         "correlation": 0.0, "filters": 2, "mmax": 2.0},
        # one template with unresolved binaries through the one-template call
        {"name": "template_binary", "kind": "template", "nx": 100, "ny": 151, "points": 800, "fraction": 0.3},
        # fg! of many uneven fits in one launch (each optimiser step of a group)
        {"name": "fits_64", "kind": "fits", "fits": 64, "Tmin": 50, "Tmax": 700, "Nmin": 5000, "Nmax": 60000},
        # the template network: mini-batch training steps (BF16, batch 32)
        {"name": "train_24", "kind": "train", "steps": 24, "batch": 32, "rows": 192},
        # the template network: filling a grid of templates
        {"name": "predict_1000", "kind": "predict", "n": 1000},
        # a population of stars sampled, observed and binned
        {"name": "mock_2e6", "kind": "mock", "mass": 2.0e6, "nx": 200, "ny": 300, "fraction": 0.3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fg", "walkers", "walkers", "templates", "templates", "template", "fits", "train", "predict",
                       "mock"])
    nx, ny = rng.randint(60, 200), rng.randint(90, 300)
    if kind == "fg":
        return {"kind": kind, "T": _log(rng, 20, 1000), "nx": nx, "ny": ny, "host": rng.random() < 0.5}
    if kind == "walkers":
        return {"kind": kind, "T": _log(rng, 20, 700), "nx": nx, "ny": ny, "B": _log(rng, 2, 4000),
                "precision": rng.choice(["f64", "f64", "bf16x2", "fp32"]), "grad": rng.random() < 0.7}
    if kind == "templates":
        # three filters: the magnitude axis is not one of the colour's filters
        filters = rng.choice([2, 2, 3])
        return {"kind": kind, "n": _log(rng, 1, 400), "nx": nx, "ny": ny, "points": rng.randint(300, 2000),
                "correlation": rng.choice([0.0, 0.6]) if filters == 2 else 0.0, "filters": filters,
                "mmax": rng.choice([2.0, 120.0])}
    if kind == "template":
        return {"kind": kind, "nx": nx, "ny": ny, "points": rng.randint(300, 2000),
                "fraction": rng.choice([0.0, 0.3])}
    if kind == "fits":
        return {"kind": kind, "fits": _log(rng, 1, 64), "Tmin": 50, "Tmax": rng.randint(60, 1000), "Nmin": 5000,
                "Nmax": rng.randint(6000, 60000)}
    if kind == "train":
        return {"kind": kind, "steps": rng.randint(8, 24), "batch": rng.choice([8, 16, 32]),
                "rows": rng.randint(64, 256)}
    if kind == "predict":
        return {"kind": kind, "n": _log(rng, 1, 1000)}
    return {"kind": "mock", "mass": float(_log(rng, 10000, 2000000)), "nx": nx, "ny": ny,
            "fraction": rng.choice([0.0, 0.3])}


# --------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _cmd_templates(T, nx, ny, seed):
    """T smooth templates (T x nx ny FP32, colour bin fastest, unit sum): a
    ridge in the colour-magnitude plane that widens and is less complete
    towards the faint end, zero far from the ridge."""
    g = _gen(seed)
    r = torch.rand((T, 6), generator=g, device="cuda")
    y = (torch.arange(ny, device="cuda") + 0.5) / ny
    x = (torch.arange(nx, device="cuda") + 0.5) / nx
    sig = 0.012 + 0.25 * torch.exp(6.0 * (y - 1.0))
    c = (0.15 + 0.2 * r[:, 0:1] + (0.25 + 0.2 * r[:, 1:2]) * y + 0.06 * torch.sin(6.0 * y + 6.28 * r[:, 2:3])
         + 0.3 * (0.5 + r[:, 3:4]) * torch.clamp(0.45 - y, min=0.0))
    a = torch.exp(3.0 * y) * torch.sigmoid((0.9 - y) / 0.07) * torch.sigmoid((y - 0.5 * r[:, 4:5]) / 0.02)
    e = (x[None, None, :] - c[:, :, None]) / sig[None, :, None]
    t = torch.exp(-0.5 * e * e) * (a / sig)[:, :, None]
    t = torch.where(e.abs() < 7.5, t, torch.zeros_like(t)).reshape(T, ny * nx)
    return (t / t.double().sum(1, keepdim=True).float()).contiguous()


def _likelihood(T, nx, ny, seed, stars=1.0e6):
    """Templates, the coefficients that made the data, and Poisson data."""
    C = _cmd_templates(T, nx, ny, seed)
    x = torch.pow(10.0, 0.3 * torch.randn(T, generator=_gen(seed + 1), device="cuda", dtype=torch.float64))
    x *= stars / x.sum()
    m = torch.zeros(nx * ny, dtype=torch.float64, device="cuda")
    for t in range(0, T, 64):
        m += x[t:t + 64] @ C[t:t + 64].double()
    return C, x, torch.poisson(m, generator=_gen(seed + 2))


def _fits(case, seed):
    rng = np.random.default_rng(case["fits"] + case["Tmax"] + case["Nmax"])      # sizes belong to the case
    out = []
    for f in range(case["fits"]):
        T = int(rng.integers(case["Tmin"], case["Tmax"] + 1))
        N = int(rng.integers(case["Nmin"], case["Nmax"] + 1))
        nx = int(round(math.sqrt(N * 2.0 / 3.0)))
        out.append(_likelihood(T, nx, N // nx, seed + 10 * f, 10.0 ** rng.uniform(4.0, 6.0)))
    return out


def _isochrones(case, n, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(n):
        age = 6.6 + 3.5 * ((k + rng.uniform()) / n)
        m, mags = synth.isochrone(age, rng.uniform(-2.5, 0.0), case["points"], int(rng.integers(1 << 30)),
                                  mmax_imf=case.get("mmax", 120.0))
        if case.get("filters") == 3:          # a third filter, redder, as the magnitude axis
            mags = list(mags) + [mags[1] - 0.6 * (mags[0] - mags[1])]
        out.append((m, mags))
    return out


def _edges(case):
    return (sfh.edges_range(-0.5, 2.5, case["nx"] + 1), sfh.edges_range(18.0, 30.0, case["ny"] + 1))


def _parameters(n, seed):
    return surrogate.sample_parameters(n, seed=seed)


def _images(params, seed):
    """Log images of smooth templates that follow the parameters."""
    p = torch.from_numpy(surrogate.scale_params(params)).cuda()
    x = torch.linspace(-0.5, 2.5, surrogate.CROP_H, device="cuda")[None, :, None]
    y = torch.linspace(0.0, 1.0, surrogate.CROP_W, device="cuda")[None, None, :]
    q = p[:, :, None, None]
    ph = 6.28 * torch.rand((1, 2), generator=_gen(seed), device="cuda")
    c = 0.6 + 0.3 * q[:, 0] + 0.25 * q[:, 1] + 0.9 * y * (1 - y) + 0.05 * torch.sin(9.0 * y + ph[:, 0, None, None])
    s = (0.05 + 0.5 * torch.exp(4.0 * (y - 1.0))) * (1.0 + 0.4 * q[:, 3])
    lnT = -9.0 + 2.0 * y + q[:, 2] - 0.5 * ((x - c) / s) ** 2
    T = torch.exp(lnT) + surrogate.LOG_EPS
    return ((torch.log(T) - surrogate.LOG_OFFSET) / surrogate.LOG_SCALE).contiguous()


# ------------------------------------------------------------------- one pass

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("fg", "walkers"):
        T, N = case["T"], case["nx"] * case["ny"]
        C, x, n = _likelihood(T, case["nx"], case["ny"], seed)
        torch.cuda.synchronize()
        s["tpl"] = sfh.HIPTemplates(device_ptr=C.data_ptr(), shape=(N, T))
        s["data"] = sfh.HIPData(device_ptr=n.data_ptr(), nbins=N)
        s["tpl"].ctx.synchronize()
        B = case.get("B", 1)
        w = torch.randn((B, T), generator=_gen(seed + 3), device="cuda", dtype=torch.float64)
        s["X"] = (x * torch.pow(10.0, 0.3 * w)).contiguous()     # T x B column-major
        s["C"], s["n"] = C, n
        if case.get("host"):
            s["x"], s["G"] = s["X"][0].cpu().numpy(), np.empty(T)
        else:
            s["nll"] = torch.empty(B, dtype=torch.float64, device="cuda")
            s["G"] = torch.empty((B, T), dtype=torch.float64, device="cuda") if case.get("grad", True) else None
    elif kind == "templates":
        s["iso"] = sfh.IsochroneBatch.from_list(_isochrones(case, case["n"], seed))
        s["dmod"] = np.random.default_rng(seed + 5).uniform(23.8, 24.2, case["n"])
        s["imf"] = synth.Kroupa2001(0.08, case["mmax"])
    elif kind == "template":
        s["iso"] = _isochrones(case, 1, seed)[0]
        s["imf"] = synth.Kroupa2001(0.08, 120.0)
    elif kind == "fits":
        fits = _fits(case, seed)
        torch.cuda.synchronize()
        tpl = [sfh.HIPTemplates(device_ptr=C.data_ptr(), shape=(C.shape[1], C.shape[0])) for C, _, _ in fits]
        dat = [sfh.HIPData(device_ptr=n.data_ptr(), nbins=n.numel()) for _, _, n in fits]
        s["mf"] = sfh.MultiFit(tpl, dat)
        s["mf"].ctx.synchronize()
        X = [x * torch.pow(10.0, 0.3 * torch.randn(x.numel(), generator=_gen(seed + 7 + f), device="cuda",
                                                  dtype=torch.float64)) for f, (_, x, _) in enumerate(fits)]
        s["X"] = torch.cat(X)
        s["nll"] = torch.empty(len(fits), dtype=torch.float64, device="cuda")
        s["G"] = torch.empty_like(s["X"])
        s["keep"] = fits if case.get("keep") else None
    elif kind == "train":
        s["params"] = _parameters(case["rows"], seed)
        s["images"] = _images(s["params"], seed)
        s["net"] = surrogate.TemplateSurrogate(dtype="bf16", seed=seed, max_batch=case["batch"])
        s["w0"] = s["net"].flat.clone()
    elif kind == "predict":
        s["params"] = _parameters(case["n"], seed)
        s["net"] = surrogate.TemplateSurrogate(params=_trained(seed), dtype="bf16", max_batch=256)
    else:
        m, mags = synth.isochrone(8.5 + (seed % 97) / 97.0, -1.0, 2000, seed % 100003, mmax_imf=120.0)
        s["m"], s["mags"], s["seed"] = m, np.stack(mags, axis=1), seed
        s["imf"] = mock.Kroupa2001(0.08, 120.0)
    return s


def _trained(seed):
    """Network weights of the size that training leaves: the initial ones, with
    biases that put the outputs in the range of log templates."""
    w = surrogate.init_params(seed)
    off, rng = 0, np.random.default_rng(seed + 1)
    for name, shape, fan in surrogate.param_layout():
        n = int(np.prod(shape))
        if name == "bmap":
            w[off:off + n] = rng.uniform(0.5, 2.5, n)
        elif fan is None:
            w[off:off + n] = rng.normal(0.0, 0.05, n)
        else:
            w[off:off + n] *= 1.1
        off += n
    return w


def _template_args(case, s):
    err, comp = [synth.PHOTERR] * case.get("filters", 2), [synth.COMPLETENESS] * case.get("filters", 2)
    return err, 2 if case.get("filters") == 3 else 1, (0, 1), s["imf"], comp


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "fg":
        if case["host"]:
            return {"nll": sfh.fg_(True, s["G"], s["x"], s["tpl"], s["data"]), "G": s["G"]}
        sfh.fg_device(s["tpl"], s["data"], s["X"], s["nll"], s["G"])
        return {"nll": s["nll"], "G": s["G"]}
    if kind == "walkers":
        sfh.fg_batched_device(s["tpl"], s["data"], s["X"], case["B"], s["nll"], s["G"], precision=case["precision"])
        return {"nll": s["nll"], "G": s["G"]}
    if kind == "templates":
        err, y, col, imf, comp = _template_args(case, s)
        return sfh.partial_cmd_smooth_batch(s["iso"], err, y, col, imf, comp, dmod=s["dmod"], mean_mass=imf.mean(),
                                            correlation=case["correlation"], edges=_edges(case))
    if kind == "template":
        err, y, col, imf, comp = _template_args(case, s)
        m, mags = s["iso"]
        return sfh.partial_cmd_smooth(m, mags, err, y, col, imf, comp, dmod=24.0, mean_mass=imf.mean(),
                                      binary_model=sfh.RandomBinaryPairs(case["fraction"]),
                                      edges=_edges(case)).weights
    if kind == "fits":
        s["mf"].fg_device(s["X"], s["nll"], s["G"])
        return {"nll": s["nll"], "G": s["G"]}
    if kind == "train":
        net = s["net"]
        net.flat.copy_(s["w0"])              # from the same start on every pass
        net.m.zero_()
        net.v.zero_()
        net.step_count = 0
        hist = net.train(s["params"], s["images"], steps=case["steps"], batch=case["batch"],
                         log_every=case["steps"], warmup=case["steps"])
        return {"weights": net.flat, "grad": net.grad, "mse": hist[-1][1], "kl": hist[-1][2]}
    if kind == "predict":
        return s["net"].predict(s["params"])
    cat = sfh.generate_stars_mass(s["m"], s["mags"], ["B", "V"], case["mass"], s["imf"], dist_mod=24.0,
                                  binary_model=sfh.RandomBinaryPairs(case["fraction"]), seed=s["seed"], catalog=True)
    obs = sfh.model_cmd(cat, [synth.photerr] * 2, [synth.completeness] * 2, seed=s["seed"] + 1)
    h = mock.bin_cmd_catalog(obs, (0, 1), 1, _edges(case)).weights
    out = {"counts": h.astype(np.int64), "drawn": int(cat.sampled), "kept": int(cat.n), "observed": int(obs.n)}
    obs.close()
    cat.close()
    return out


# ------------------------------------------------------------ work, tolerance

_NET_MACS = 16 * 256 + 256 * 512 + 512 * 7904 + 247 * (1 + 4 + 16) * 512 * 32 + 247 * 64 * 512


def work(case):
    kind = case["kind"]
    if kind in ("fg", "walkers"):
        T, N, B = case["T"], case["nx"] * case["ny"], case.get("B", 1)
        g = case.get("grad", True)
        return {"bytes": 4.0 * T * N + 8.0 * N + 8.0 * B * (T * (2 if g else 1) + 1),
                "flops": B * N * (T * (4.0 if g else 2.0) + 8.0)}
    if kind in ("templates", "template"):
        n, nb, pts = case.get("n", 1), case["nx"] * case["ny"], case["points"]
        # a third of the bins lie in a point's kernel; one multiply and one add each
        pairs = n * nb * pts * 0.33 * (2.0 if case.get("fraction") else 1.0)
        return {"bytes": n * (4.0 * nb + 8.0 * pts * (1 + case.get("filters", 2))), "flops": 2.0 * pairs}
    if kind == "fits":
        TN = case["fits"] * 0.25 * (case["Tmin"] + case["Tmax"]) * (case["Nmin"] + case["Nmax"])
        return {"bytes": 4.0 * TN, "flops": 4.0 * TN}
    if kind == "train":
        k, nparam = case["steps"] * case["batch"], 4303680
        return {"bytes": case["steps"] * 28.0 * nparam + k * 4.0 * 60000 * 2, "flops": 6.0 * k * _NET_MACS}
    if kind == "predict":
        return {"bytes": case["n"] * 4.0 * 60000 + 4303680 * 4.0, "flops": 2.0 * case["n"] * _NET_MACS}
    systems = 1.33 * case["mass"]
    return {"bytes": systems * 41.0 + 4.0 * case["nx"] * case["ny"], "flops": systems * 200.0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("fg", "fits"):
        return {"rel": 1e-11, "max": 1e-8}            # FP64 sums in another order
    if kind == "walkers":
        if case["precision"] == "f64":                # FP64 log-likelihood, split-BF16 gradient
            return {"rel": 1e-6 if case["grad"] else 1e-12, "max": 1e-4 if case["grad"] else 1e-11}
        return {"rel": 2e-5, "max": 2e-3}
    if kind in ("templates", "template"):
        return {"rel": 3e-6, "max": 3e-5}              # FP32 kernels, FP64 sums over 64-point groups
    if kind == "train":
        return {"rel": 1e-2, "max": 0.5}               # BF16 operands through several steps
    if kind == "predict":
        return {"rel": 4e-3, "max": 0.1}               # BF16 operands, outputs exponentiated
    return "exact"                                    # whole counts


# ------------------------------------------------- the same results in 64 bits

def _exact_fg(C, n, X, eps=float(np.finfo(np.float64).eps), grad=True):
    """-logL and its gradient for each row of X (B x T)."""
    C = C.double()
    nll, G = [], []
    for b in range(0, X.shape[0], 1024):
        m = X[b:b + 1024] @ C
        c = torch.clamp(m, min=eps)
        safe = torch.where(n > 0, n, torch.ones_like(n))
        ll = torch.where(n > 0, n - c - n * torch.log(safe / c), -c).sum(1)
        nll.append(-ll)
        if grad:
            G.append((1.0 - n / c) @ C.T)
    return {"nll": torch.cat(nll), "G": torch.cat(G) if grad else None}


_GL = 0.7745966692414834


def _deposit_rows(out, pts, ex, ey, asym):
    """Adds pixel-integrated kernels (rows of pts: x, y, sx, sy, c, weight) to
    out (ny x nx), dense over the rows that the points' footprints span."""
    nx, ny = ex.length - 1, ey.length - 1
    x0, y0, sx, sy, c, A = (pts[:, k] for k in range(6))
    if asym:
        px, py = (x0 - ex.first) / ex.step + 1.0, (y0 - ey.first) / ey.step + 1.0
        sx, sy = sx / ex.step, sy / ey.step
        xp, yp = torch.round(px), torch.round(py)
        xo = torch.clamp(torch.floor(torch.ceil(10.0 * sx) / 2.0), min=1.0)
        yo = torch.clamp(torch.floor(torch.ceil(10.0 * sy) / 2.0), min=1.0)
    else:
        xp = torch.round((x0 - ex.first) / ex.step + 1.0)
        yp = torch.round((y0 - ey.first) / ey.step + 1.0)
        xo = torch.clamp(torch.round(15.0 * sx / ex.step / 2.0), min=1.0)
        yo = torch.clamp(torch.round(10.0 * sy / ey.step / 2.0), min=1.0)
    xa, xb = torch.clamp(xp - xo, min=1.0), torch.clamp(xp + xo, max=float(nx))
    ya, yb = torch.clamp(yp - yo, min=1.0), torch.clamp(yp + yo, max=float(ny))
    ok = (xb - xa >= 1) & (yb - ya >= 1)
    if not bool(ok.any()):
        return
    r0, r1 = int(ya[ok].min()), int(yb[ok].max())
    rows = torch.arange(r0, r1 + 1, dtype=torch.float64, device=pts.device)
    cols = torch.arange(1, nx + 1, dtype=torch.float64, device=pts.device)
    inx = (cols >= xa[:, None]) & (cols <= xb[:, None]) & ok[:, None]
    iny = (rows >= ya[:, None]) & (rows <= yb[:, None])
    if asym:
        f = lambda at, o, s: torch.special.erf((at + 0.5 - o) / (math.sqrt(2.0) * s))  # noqa: E731
        edge = torch.arange(1, nx + 2, dtype=torch.float64, device=pts.device) - 0.5
        fx = f(edge[None, :], px[:, None], sx[:, None]).diff(dim=1) * inx
        edge = torch.arange(r0, r1 + 2, dtype=torch.float64, device=pts.device) - 0.5
        fy = f(edge[None, :], py[:, None], sy[:, None]).diff(dim=1) * iny
        out[r0 - 1:r1] += (fy * (A / 4.0)[:, None]).T @ fx
        return
    hx, hy = ex.step / 2.0, ey.step / 2.0
    edge = (torch.arange(1, nx + 2, dtype=torch.float64, device=pts.device) - 0.5) * ex.step + ex.first - hx
    yc = (rows - 0.5) * ey.step + ey.first
    pref = A * hy / (2.0 * math.sqrt(2.0 * math.pi) * sy)
    for k, w in ((-1, 5.0 / 9.0), (0, 8.0 / 9.0), (1, 5.0 / 9.0)):
        t = (yc[None, :] + k * _GL * hy - y0[:, None]) / sy[:, None]                      # point x row
        u = ((edge[None, :] - x0[:, None])[:, None, :] + (c * sy)[:, None, None] * t[:, :, None])
        u = torch.special.erf(u / (math.sqrt(2.0) * sx)[:, None, None]).diff(dim=2)
        wy = pref[:, None] * w * torch.exp(-0.5 * t * t) * iny
        out[r0 - 1:r1] += torch.einsum("prc,pr->rc", u * inx[:, None, :], wy)


def _deposit(pts, ex, ey, asym):
    out = torch.zeros((ey.length - 1, ex.length - 1), dtype=torch.float64, device="cuda")
    pts = torch.from_numpy(np.stack([np.asarray(p, dtype=np.float64) for p in pts], axis=1)).cuda()
    for k in range(0, pts.shape[0], 192):
        _deposit_rows(out, pts[k:k + 192], ex, ey, asym)
    return out.reshape(-1)


def _sigma(m):
    return np.power(math.e, 0.6 * (m - 28.0)) + 0.01


def _complete(m):
    return 1.0 / (1.0 + np.exp((m - 28.0) / 0.7))


def _imf(m, mmax):
    hi = 0.5 * (0.5 ** -1.3 - mmax ** -1.3) / 1.3 if mmax > 0.5 else 0.0
    norm = 1.0 / ((0.08 ** -0.3 - min(mmax, 0.5) ** -0.3) / 0.3 + hi)
    return np.where((m >= 0.08) & (m <= mmax), np.where(m < 0.5, m ** -1.3, 0.5 * m ** -2.3) * norm, 0.0)


def _imf_mean(mmax):
    hi = 0.5 * (0.5 ** -0.3 - mmax ** -0.3) / 0.3 if mmax > 0.5 else 0.0
    above = 0.5 * (0.5 ** -1.3 - mmax ** -1.3) / 1.3 if mmax > 0.5 else 0.0
    norm = 1.0 / ((0.08 ** -0.3 - min(mmax, 0.5) ** -0.3) / 0.3 + above)
    return norm * ((min(mmax, 0.5) ** 0.7 - 0.08 ** 0.7) / 0.7 + hi)


def _mid(v):
    d = np.diff(v)
    if d.size and np.all(np.abs(d - d[0]) <= 1.4901161193847656e-08 * np.maximum(abs(d[0]), np.abs(d))):
        a, b, n = v[0] + d[0] / 2, v[-1] - d[0] / 2, v.size - 1
        return np.array([a]) if n == 1 else a + np.arange(n) * ((b - a) / (n - 1))
    return v[:-1] + d / 2


def _points(m, mags, case, dmod, mmax, ex, ey):
    """The kernel points of one isochrone and its resampled masses and magnitudes."""
    y = mags[2] if case.get("filters") == 3 else mags[1]
    d = np.hypot(np.diff(mags[0] - mags[1]), np.diff(y))
    step = min(ex.step, ey.step)
    k = np.where(d > step, np.ceil(d / step), 1.0).astype(int)
    new = [m[:1]]
    for i in range(d.size):
        new.append(m[i] + (m[i + 1] - m[i]) / k[i] * np.arange(1, k[i] + 1) if d[i] > step else m[i + 1:i + 2])
    new = np.concatenate(new)
    g = [np.interp(new, m, v) + dmod for v in mags]
    err = [_sigma(v) for v in g]
    comp = _complete(g[0]) * _complete(g[1])
    if case.get("filters") == 3:
        comp, cerr, yerr, yy, cov = comp * _complete(g[2]), np.hypot(err[0], err[1]), err[2], g[2], 0.0
    else:
        cerr, yerr, yy, cov = err[0], err[1], g[1], 1.0
    f = _imf(new, mmax)
    w = np.diff(new) * (f[:-1] + f[1:]) / 2 * comp[:-1] / _imf_mean(mmax)
    sx, sy = _mid(cerr), _mid(yerr)
    r = case.get("correlation", 0.0)
    c = -r / math.sqrt(1.0 - r * r) * sx / sy if r else np.full(w.size, cov)
    return (_mid(g[0] - g[1]), _mid(yy), sx, sy, c, w), new, g


def _exact_binary(m, g, ex, ey):
    """Pairs of an isochrone's intervals (summed fluxes), binned and smoothed."""
    f = _imf(m, 120.0)
    pre = 1.0 / _imf_mean(120.0) / 4.0 / float(np.sum(np.diff(m) * (f[1:] + f[:-1])) / 2)
    i, j = np.triu_indices(m.size - 1, 1)
    mag = [-2.5 * np.log10(10.0 ** (-0.4 * v[i]) + 10.0 ** (-0.4 * v[j])) for v in g]
    dm, s = np.diff(m), f[:-1] + f[1:]
    w = dm[i] * dm[j] * s[i] * s[j] * pre * _complete(mag[0]) * _complete(mag[1])
    nx, ny = ex.length - 1, ey.length - 1
    bx = np.floor((mag[0] - mag[1] - ex.first) / ex.step).astype(int)
    by = np.floor((mag[1] - ey.first) / ey.step).astype(int)
    ok = (bx >= 0) & (bx < nx) & (by >= 0) & (by < ny)
    h = np.bincount(by[ok] * nx + bx[ok], weights=w[ok], minlength=nx * ny)
    k = np.flatnonzero(h)
    # bin centres sit on a tie of the footprint's rounding: formed in the reference's order
    x, y = ex.first + (k % nx) * ex.step + ex.step / 2, ey.first + (k // nx) * ey.step + ey.step / 2
    return _deposit((x, y, _sigma(y + x), _sigma(y), np.ones(k.size), h[k]), ex, ey, False)


def _unpack(flat):
    out, off = {}, 0
    for name, shape, _ in surrogate.param_layout():
        n = int(np.prod(shape))
        out[name] = flat[off:off + n].view(*shape)
        off += n
    return out


def _up(a, K, B, H, W, co):
    """4 x 4 transposed convolution, stride 2, padding 1, of a (B H W x 32)."""
    cols = (a @ K.T).view(B, H * W, 16, co).permute(0, 3, 2, 1).reshape(B, co * 16, H * W)
    return torch.nn.functional.fold(cols, (2 * H, 2 * W), 4, padding=1, stride=2).permute(0, 2, 3, 1)


def _net(P, x):
    silu = torch.nn.functional.silu
    B = x.shape[0]
    x16 = torch.zeros((B, 16), dtype=torch.float64, device=x.device)
    x16[:, :4] = x
    a = x16
    for k in "012":
        a = silu(a @ P["W" + k].T + P["b" + k])
    H, W = surrogate.H0, surrogate.W0
    a = a.reshape(-1, 32)
    for k in "123":
        a = silu(_up(a, P["K" + k], B, H, W, 32) + P["c" + k]).reshape(-1, 32)
        H, W = 2 * H, 2 * W
    return _up(a, P["w4"], B, H, W, 1)[..., 0] + P["bmap"].view(2 * H, 2 * W)


def _exact_train(case, seed):
    params = _parameters(case["rows"], seed)
    images = _images(params, seed).double()
    xs = torch.from_numpy(surrogate.scale_params(params)).cuda().double()
    flat = torch.from_numpy(surrogate.init_params(seed)).cuda().double().requires_grad_(True)
    n, b, steps = case["rows"], case["batch"], case["steps"]
    rng = np.random.default_rng(0)
    per = n // b
    rows = np.concatenate([rng.permutation(n)[:per * b] for _ in range(-(-steps // per))])
    m, v = torch.zeros_like(flat), torch.zeros_like(flat)
    mse_sum = kl_sum = 0.0
    for k in range(steps):
        r = torch.from_numpy(rows[k * b:(k + 1) * b]).cuda()
        o = _net(_unpack(flat), xs[r])[:, :surrogate.CROP_H, :surrogate.CROP_W]
        t = images[r]
        ls, le = (torch.log_softmax((surrogate.LOG_SCALE * u + surrogate.LOG_OFFSET).reshape(b, -1), 1) for u in (o, t))
        mse, kl = ((o - t) ** 2).mean(), (torch.exp(le) * (le - ls)).sum(1).mean()
        g, = torch.autograd.grad(mse + kl, flat)
        mse_sum, kl_sum = mse_sum + float(mse.detach()), kl_sum + float(kl.detach())
        with torch.no_grad():
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            step = 1e-3 * (k + 1) / steps
            flat -= step * (m / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1 - 0.999 ** (k + 1))) + 1e-8)
    return {"weights": flat.detach(), "grad": g, "mse": mse_sum / steps, "kl": kl_sum / steps}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fg", "walkers"):
        s = prepare(case, seed)
        r = _exact_fg(s["C"], s["n"], s["X"], grad=case.get("grad", True))
        if case.get("host"):
            return {"nll": float(r["nll"][0]), "G": r["G"][0]}
        return r
    if kind == "fits":
        s = prepare({**case, "keep": True}, seed)
        at, nll, G = 0, [], []
        for C, x, n in s["keep"]:
            r = _exact_fg(C, n, s["X"][at:at + x.numel()][None])
            nll.append(r["nll"])
            G.append(r["G"][0])
            at += x.numel()
        return {"nll": torch.cat(nll), "G": torch.cat(G)}
    if kind == "templates":
        s, (ex, ey) = prepare(case, seed), _edges(case)
        iso, out = s["iso"], []
        for k in range(case["n"]):
            a, b = int(iso.offsets[k]), int(iso.offsets[k + 1])
            p, _, _ = _points(iso.m_ini[a:b], [v[a:b] for v in iso.mags], case, s["dmod"][k], case["mmax"], ex, ey)
            out.append(_deposit(p, ex, ey, case["filters"] == 3))
        return torch.stack(out)
    if kind == "template":
        (m, mags), (ex, ey) = _isochrones(case, 1, seed)[0], _edges(case)
        p, new, g = _points(m, mags, case, 24.0, 120.0, ex, ey)
        t = _deposit(p, ex, ey, False)
        if case["fraction"]:
            f = _imf(new, 120.0)
            b = 2 * case["fraction"] / (1 + case["fraction"]) * float(np.sum(np.diff(new) * (f[1:] + f[:-1])) / 2)
            t = t * (1 - b) + b * _exact_binary(new[::4], [v[::4] for v in g], ex, ey)
        return t.view(ey.length - 1, ex.length - 1).T
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "predict":
        P = _unpack(torch.from_numpy(_trained(seed)).cuda().double())
        x = torch.from_numpy(surrogate.scale_params(_parameters(case["n"], seed))).cuda().double()
        out = torch.empty((case["n"], 60000), dtype=torch.float64, device="cuda")
        for b in range(0, case["n"], 64):
            o = _net(P, x[b:b + 64])[:, :surrogate.CROP_H, :surrogate.CROP_W]
            t = torch.clamp(torch.exp(o * surrogate.LOG_SCALE + surrogate.LOG_OFFSET) - surrogate.LOG_EPS, min=0.0)
            out[b:b + 64] = t.permute(0, 2, 1).reshape(t.shape[0], -1)
        return out
    return None
