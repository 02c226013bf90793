"""The work that a user of this package has it do on the GPU, as measurable cases.

Each case is one pass through the public entry points: whole field runs in 2D,
3D and Nx2D (upload, trace, influence, download), a resident problem launched
again, batched sweeps, arrivals, ray paths, and the surrogate's training and
prediction. Sizes are those of the package's own workload builders, tests and
benchmark, or the small and ragged sizes between them.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call (problems, handles)
  run(state)           one pass; returns the outputs
  exact(case, seed)    the outputs in 64 bits by plain numpy, where that is quick
  work(case)           bytes and operations a pass cannot do without
  tolerance(case)      how far two correct runs may be apart
"""
import math

import numpy as np

import bellhopcuda_amd as bh
from bellhopcuda_amd import surrogate as sg
from bellhopcuda_amd.env import c2_env, munk_env, sweep_envs
from bellhopcuda_amd.env3d import c3_env


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # One small field at a time, as an interactive program or a fitting
        # loop runs them: latency of the whole call.
        dict(name="munk_small", kind="tl2d", beams=201, nrz=51, nrr=101, run="CG", ssp="C", bits=64),
        # The plain deep-water field with hat beams, at its usual size.
        dict(name="munk", kind="tl2d", beams=2001, nrz=201, nrr=1001, run="CG", ssp="C", bits=64),
        # Single precision, Gaussian beams, incoherent sum, a PCHIP profile and
        # ragged sizes: the quick-look setting.
        dict(name="munk_gauss_f32", kind="tl2d", beams=1501, nrz=153, nrr=777, run="IB", ssp="P", bits=32),
        # A large range-dependent field of ray-centred Gaussian beams, kept
        # resident and launched again.
        dict(name="seamount", kind="resident", beams=20001, nrz=501, nrr=5001, run="Cb", bits=64),
        # Arrivals (amplitudes and delays per receiver) for impulse responses.
        dict(name="arrivals", kind="arrivals", beams=2001, nrz=21, nrr=101, run="AG", narr=50, bits=64),
        # Ray paths for a plot.
        dict(name="rays", kind="rays", beams=101, points=1000, bits=64),
        # A sweep of unlike environments in one launch.
        dict(name="sweep", kind="sweep", problems=48, scale=0.5, set=0, bits=64),
        # A sweep over one environment family, as the surrogate is trained on.
        dict(name="family", kind="family", problems=128, beams=1001, nrz=51, nrr=201, bits=64),
        # The 3D shelf-canyon field of Gaussian beams at full size.
        dict(name="shelf3d", kind="field3d", alphas=1001, betas=181, thetas=36, nrz=101, nrr=1001, nxy=201,
             run="CB   3", bits=64),
        # The same sea in Nx2D: 2D rays on each receiver bearing.
        dict(name="shelf_nx2d", kind="field3d", alphas=501, betas=36, thetas=36, nrz=101, nrr=501, nxy=201,
             run="CB   2", bits=64),
        # The surrogate's training, a chunk of Adam steps at its default batch.
        dict(name="train", kind="train", members=4, batch=2048, outputs=128, steps=25),
        # The surrogate's prediction for a screened sweep's environments.
        dict(name="predict", kind="predict", members=4, points=1000, outputs=128),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tl2d", "tl2d", "resident", "arrivals", "rays", "sweep", "family", "field3d", "field3d",
                       "train", "predict"])
    bits = rng.choice([64, 64, 32])
    if kind == "tl2d":
        return dict(kind=kind, beams=_logint(rng, 101, 6001), nrz=_logint(rng, 21, 401), nrr=_logint(rng, 51, 2001),
                    run=rng.choice(["CG", "CB", "IB", "SG", "Cg", "Cb"]), ssp=rng.choice(["C", "P", "S", "N"]),
                    bits=bits)
    if kind == "resident":
        return dict(kind=kind, beams=_logint(rng, 1001, 15001), nrz=_logint(rng, 51, 501), nrr=_logint(rng, 301, 5001),
                    run=rng.choice(["Cb", "Cg", "CB", "CG"]), bits=bits)
    if kind == "arrivals":
        return dict(kind=kind, beams=_logint(rng, 201, 4001), nrz=_logint(rng, 3, 41), nrr=_logint(rng, 11, 201),
                    run=rng.choice(["AG", "AB", "Ag"]), narr=_logint(rng, 10, 80), bits=bits)
    if kind == "rays":
        return dict(kind=kind, beams=_logint(rng, 5, 400), points=1000, bits=bits)
    if kind == "sweep":
        return dict(kind=kind, problems=rng.randrange(5, 49), scale=rng.choice([0.1, 0.2, 0.35, 0.5]),
                    set=rng.randrange(1, 1000), bits=bits)
    if kind == "family":
        return dict(kind=kind, problems=_logint(rng, 16, 160), beams=_logint(rng, 251, 1201), nrz=_logint(rng, 21, 61),
                    nrr=_logint(rng, 101, 251), bits=64)
    if kind == "field3d":
        run = rng.choice(["CB   3", "CG   3", "IB   3", "CB   2", "CG   2"])
        three = run[5] == "3"
        thetas = rng.randrange(4, 37)
        return dict(kind=kind, alphas=_logint(rng, 51, 501), betas=_logint(rng, 31, 121) if three else thetas,
                    thetas=thetas, nrz=_logint(rng, 21, 101), nrr=_logint(rng, 101, 701), nxy=_logint(rng, 41, 201),
                    run=run, bits=64)
    if kind == "train":
        return dict(kind=kind, members=rng.randrange(1, 7), batch=32 * _logint(rng, 8, 64),
                    outputs=32 * rng.randrange(1, 9), steps=rng.randrange(5, 26))
    return dict(kind=kind, members=rng.randrange(1, 7), points=_logint(rng, 17, 3000), outputs=32 * rng.randrange(1, 9))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _munk(case, seed):
    """A deep-water environment around the Munk profile: source depth,
    frequency and a smooth profile perturbation from the seed."""
    rng = np.random.default_rng(seed)
    e = munk_env(nbeams=case["beams"], nrz=case.get("nrz", 11), nrr=case.get("nrr", 11),
                 precision=case["bits"], run_type=case.get("run", "RG"), ssp_type=case.get("ssp", "C"),
                 sd=float(rng.uniform(700.0, 1300.0)), freq=float(rng.uniform(45.0, 55.0)))
    z = e.ssp_z
    for k in range(1, 4):
        e.ssp_c = e.ssp_c + rng.uniform(-2.0, 2.0) / k * np.sin(k * np.pi * z / 5000.0)
    return e


def _sweep(case, seed):
    """Unlike environments: the set fixes their sizes, the seed their sources,
    frequencies and profiles."""
    rng = np.random.default_rng(seed)
    envs = sweep_envs(n=case["problems"], seed=20260004 + case["set"], precision=case["bits"], scale=case["scale"])
    for e in envs:
        e.Sz = (e.Sz * rng.uniform(0.9, 1.1)).astype(np.float32)
        e.freq0 *= float(rng.uniform(0.95, 1.05))
        e.ssp_c = e.ssp_c + rng.uniform(-2.0, 2.0) * np.sin(np.pi * e.ssp_z / e.ssp_z[-1])
    return envs


def _shelf(case, seed):
    rng = np.random.default_rng(seed)
    e = c3_env(seed=seed + 20260003, nalpha=case["alphas"], nbeta=case["betas"], ntheta=case["thetas"],
               nrz=case["nrz"], nrr=case["nrr"], nxy=case["nxy"], precision=case["bits"], run_type=case["run"])
    e.Sz = np.array([rng.uniform(80.0, 120.0)], np.float32)
    return e


def _net_params(case, seed):
    """Weights of an ensemble as a program loads them: He-uniform hidden
    layers, a small output layer."""
    rng = np.random.default_rng(seed)
    k = case["outputs"]
    parts = []
    for l in range(6):
        fan = 64 if l == 0 else 256
        a = math.sqrt(6.0 / fan)
        parts += [rng.uniform(-a, a, (case["members"], fan * 256)), rng.uniform(-0.05, 0.05, (case["members"], 256))]
    parts += [rng.uniform(-0.05, 0.05, (case["members"], 256 * k)), rng.uniform(-0.05, 0.05, (case["members"], k))]
    return np.concatenate(parts, axis=1).astype(np.float32)


def _net_inputs(case, seed, n):
    return sg.param_inputs(sg.draw_params(n, seed + 1, "global"))


class _Held:
    """Gives a device handle back when the state goes."""

    def __init__(self, h):
        self.h = h

    def __del__(self):
        self.h.release()


_CTX = []


def _ctx():
    """The program's one GPU context."""
    if not _CTX:
        _CTX.append(bh.Context(0))
    return _CTX[0]


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case, "kind": k}
    if k in ("tl2d", "arrivals", "rays"):
        s["prob"] = bh.Problem(_munk(case, seed))
        s["ctx"] = _ctx()
    elif k == "resident":
        e = c2_env(seed=seed + 20260002, nbeams=case["beams"], nrz=case["nrz"], nrr=case["nrr"],
                   precision=case["bits"], run_type=case["run"])
        s["held"] = _Held(bh.Resident(bh.Problem(e), _ctx()))
    elif k == "sweep":
        envs = _sweep(case, seed)
        s["sweep"] = bh.Sweep([bh.Problem(e) for e in envs], _ctx())
    elif k == "family":
        th = sg.draw_params(case["problems"], seed, "global")
        envs = [sg.environment(t, nbeams=case["beams"], nrz=case["nrz"], nrr=case["nrr"]) for t in th]
        s["sweep"] = bh.Sweep([bh.Problem(e) for e in envs], _ctx())
    elif k == "field3d":
        s["prob"] = bh.Problem3D(_shelf(case, seed))
        s["ctx"] = _ctx()
    elif k == "train":
        m = sg.Mlp(members=case["members"], max_batch=case["batch"], seed=3, sigma=0.05, n_out=case["outputs"], front=1)
        m.set_fourier(sg.fourier_matrix(11))
        m.set_params(_net_params(case, seed))
        n = 8192
        rng = np.random.default_rng(seed + 2)
        x = _net_inputs(case, seed, n)
        w = rng.normal(size=(16, case["outputs"])) / 4.0
        m.set_dataset(x, np.tanh(x @ w).astype(np.float32))
        s["mlp"], s["seed"] = m, seed
    else:
        m = sg.Mlp(members=case["members"], max_batch=2048, seed=3, sigma=0.05, n_out=case["outputs"], front=1)
        m.set_fourier(sg.fourier_matrix(11))
        m.set_params(_net_params(case, seed))
        s["mlp"], s["x"] = m, _net_inputs(case, seed, case["points"])
    return s


def run(state):
    k, case = state["kind"], state["case"]
    if k == "tl2d":
        return bh.field_run(state["prob"], ctx=state["ctx"]).field
    if k == "arrivals":
        r = bh.field_run(state["prob"], ctx=state["ctx"], max_narr=case["narr"])
        a = np.ctypeslib.as_array(r.arr).reshape(len(r.narr), case["narr"])
        a[np.arange(case["narr"]) >= r.narr[:, None]] = np.zeros((), a.dtype)   # slots no arrival was written to
        return {"narr": r.narr, **{f: a[f] for f in ("NTopBnc", "NBotBnc", "SrcDeclAngle", "RcvrDeclAngle", "a", "Phase",
                                                     "delay")}}
    if k == "rays":
        pts, nsteps, _ = bh.ray_run(state["prob"], ctx=state["ctx"], max_points=case["points"])
        return {"nsteps": nsteps, **{f: pts[f] for f in ("x", "t", "p", "q", "tau", "c", "Amp", "Phase", "NumTopBnc",
                                                         "NumBotBnc")}}
    if k == "resident":
        r = state["held"].h
        r.launch()
        return r.download().field
    if k == "sweep":
        sw = state["sweep"]
        sw.launch()
        return [sw.download(i).field for i in range(case["problems"])]
    if k == "family":
        sw = state["sweep"]
        sw.launch()
        return np.stack([sw.download(i).field for i in range(case["problems"])])
    if k == "field3d":
        return bh.field_run3d(state["prob"], ctx=state["ctx"]).field
    if k == "train":
        m = state["mlp"]
        loss = m.train(case["steps"], case["batch"], 1e-3, seed=state["seed"])
        return {"loss": loss, "params": m.params()[0]}
    return state["mlp"].predict(state["x"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Inputs read once, outputs written once; operations of the algorithm: so
    many per ray step and per contribution (each +, x, /, sqrt and function
    counted once), with the mean step and contribution counts of these
    environments; for the networks, the matrix products' multiplies and adds."""
    k = case["kind"]
    b = case.get("bits", 64) // 8
    if k in ("tl2d", "arrivals", "rays"):
        rays, steps = case["beams"], 485
        if k == "rays":
            return {"bytes": rays * steps * 112.0 + 8e3, "flops": rays * steps * 255.0}
        nrz, nrr = case["nrz"], case["nrr"]
        beams_over = 100e3 * math.radians(40.0) / rays * 2.0 / 5000.0   # a hat beam's share of the column, about
        contrib = rays * nrr * max(1.0, nrz * beams_over * 0.5)
        out = nrz * nrr * (8.0 if k == "tl2d" else 4.0 + 40.0 * case["narr"])
        return {"bytes": out + 8e3 + rays * 3 * b, "flops": rays * steps * 255.0 + contrib * 26.0}
    if k == "resident":
        rays = case["beams"]
        contrib = 3.53e9 * rays / 20001 * case["nrz"] / 501 * case["nrr"] / 5001
        return {"bytes": 8.0 * case["nrz"] * case["nrr"] + rays * 3 * b + 4e4,
                "flops": rays * 1825 * 326.0 + contrib * 30.0}
    if k == "sweep":
        n, sc = case["problems"], case["scale"]
        return {"bytes": n * (8.0 * 276 * 2600 * sc * sc + 1e4), "flops": n * sc * 10200 * (1950 * 298.0 + 1270 * 26.0)}
    if k == "family":
        n, rays = case["problems"], case["beams"]
        cells = case["nrz"] * case["nrr"]
        return {"bytes": n * (8.0 * cells + 1e4), "flops": n * rays * (700 * 260.0 + 0.08 * cells * 26.0)}
    if k == "field3d":
        cells = case["thetas"] * case["nrz"] * case["nrr"]
        rays = case["alphas"] * case["betas"]
        if case["run"][5] == "3":
            contrib = 1.377e9 * rays / 181181 * cells / 3.64e6
            fl = rays * 950 * 939.0 + contrib * 56.0
        else:
            fl = rays * 950 * 420.0 + rays * case["nrr"] * case["nrz"] * 0.05 * 26.0
        return {"bytes": 8.0 * cells + 8.0 * (case["nxy"] ** 2 + 21 * 21 * 50), "flops": fl}
    e, o = case["members"], case["outputs"]
    macs = 64 * 256 + 5 * 256 * 256 + 256 * o
    params = e * (macs + 6 * 256 + o) * 4.0
    if k == "train":
        n = case["batch"] * case["steps"]
        return {"bytes": n * 4.0 * (16 + o) + 2 * params, "flops": 2.0 * e * n * (3 * macs - 64 * 256)}
    n = case["points"]
    return {"bytes": params + 4.0 * n * 16 + 4.0 * e * n * o, "flops": 2.0 * e * n * macs}


def tolerance(case):
    """Fields are 32-bit sums added in no fixed order; arrivals and rays are
    computed one by one; the networks read 16-bit copies of the weights."""
    k = case["kind"]
    if k in ("arrivals", "rays"):
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if k == "train":
        return {"rel": 2e-3, "max": 0.2}
    if k == "predict":
        return {"rel": 1e-4, "max": 5e-3}
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits by plain numpy
# ---------------------------------------------------------------------------

def exact(case, seed):
    k = case["kind"]
    if k == "predict":
        return _exact_predict(case, seed)
    if (k == "tl2d" and case["bits"] == 64 and case["ssp"] == "C" and case["run"] in ("CG", "CB", "IB", "IG")
            and case["beams"] * case["nrr"] * case["nrz"] < 6e8):
        return _exact_munk(case, seed)
    return None


def _exact_predict(case, seed):
    P = _net_params(case, seed).astype(np.float64)
    x = _net_inputs(case, seed, case["points"]).astype(np.float64)
    B = sg.fourier_matrix(11).astype(np.float64)
    proj = 2.0 * np.pi * (x @ B.T[:, :24])
    f = np.empty((len(x), 64))
    f[:, :16] = x
    f[:, 16::2] = np.sin(proj)
    f[:, 17::2] = np.cos(proj)
    from torch.special import erf
    import torch
    out = []
    for p in P:
        h, o = torch.from_numpy(f), 0
        for fan, width, last in [(64, 256, False)] + [(256, 256, False)] * 5 + [(256, case["outputs"], True)]:
            w = torch.from_numpy(p[o:o + fan * width].reshape(fan, width))
            o += fan * width
            h = h @ w + torch.from_numpy(p[o:o + width])
            o += width
            if not last:
                h = 0.5 * h * (1.0 + erf(h * math.sqrt(0.5)))
        out.append(h.numpy())
    return np.stack(out)


def _caustic(q0, q1):
    return ((q1 <= 0.0) & (q0 > 0.0)) | ((q1 >= 0.0) & (q0 < 0.0))


def _exact_munk(case, seed):
    """The field of a depth-only c-linear ocean with a flat vacuum surface and
    a flat fluid halfspace bottom: all rays stepped together (second-order
    polygon steps cut at profile knots, boundaries and the box), then each
    step's beam added to the receiver columns it spans."""
    e = _munk(case, seed)
    z, cp = np.asarray(e.ssp_z), np.asarray(e.ssp_c)
    grad = np.diff(cp) / np.diff(z)
    D, deltas, rbox, zbox = 5000.0, 500.0, 1000.0 * e.box_r_km, e.box_z
    alpha = np.radians(e.alpha_deg)
    n = len(alpha)
    dalpha = (alpha[-1] - alpha[0]) / (n - 1)
    omega = 2.0 * np.pi * e.freq0
    cb = e.bot.alphaR
    cbot = cb + 1j * (e.bot.alphaI * e.freq0 / (8.6858896 * cb)) * cb * cb / omega
    Rz, Rr = np.asarray(e.Rz, np.float64), 1000.0 * np.asarray(e.Rr_km)
    gauss, coherent = e.run_type[1] == "B", e.run_type[0] == "C"
    zs = float(np.float32(e.Sz[0]))
    kmax = len(z) - 2

    def segment(x, tz):
        """Layer of depth x for a ray heading tz: a knot belongs to the layer ahead."""
        down = np.searchsorted(z, x, "right") - 1
        up = np.searchsorted(z, x, "left") - 1
        return np.clip(np.where(tz >= 0.0, down, up), 0, kmax)

    def speed(x, i):
        return cp[i] + (x - z[i]) * grad[i]

    def cut(h, x0r, x0z, ur, uz, i):
        """Step length h cut at the first knot, box side or boundary crossed."""
        x1r, x1z = x0r + h * ur, x0z + h * uz
        h2 = h
        with np.errstate(divide="ignore", invalid="ignore"):
            above, below = z[i] > x1z, z[i + 1] < x1z
            steep = np.abs(uz) > 2.2e-16
            h2 = np.where(steep & above, np.minimum(h2, (z[i] - x0z) / uz), h2)
            h2 = np.where(steep & ~above & below, np.minimum(h2, (z[i + 1] - x0z) / uz), h2)
            h2 = np.where(np.abs(x1r) >= rbox, np.minimum(h2, (rbox - np.abs(x0r)) / np.abs(ur)), h2)
            h2 = np.where(np.abs(x1z) >= zbox, np.minimum(h2, (zbox - np.abs(x0z)) / np.abs(uz)), h2)
            h2 = np.where(x1z <= 0.0, np.minimum(h2, -x0z / uz), h2)
            h2 = np.where(x1z >= D, np.minimum(h2, (D - x0z) / uz), h2)
        return np.maximum(h2, 1e-6 * deltas)

    field = np.zeros((len(Rz), len(Rr)), np.complex128)
    i0 = segment(np.full(n, zs), np.sin(alpha))
    c0 = speed(np.full(n, zs), i0)
    ray = dict(r=np.zeros(n), z=np.full(n, zs), tr=np.cos(alpha) / c0, tz=np.sin(alpha) / c0, p=np.ones(n),
               q=np.zeros(n), tau=np.zeros(n), amp=np.ones(n), ph=np.zeros(n), c=c0, i=i0, caus=np.zeros(n),
               qold=np.zeros(n), ratio=np.sqrt(np.cos(alpha)) / (math.sqrt(2.0 * np.pi) if gauss else 1.0),
               rq=dalpha / c0)
    first = 1 if Rr[0] <= 0.0 else 0
    for _ in range(4000):
        if not len(ray["r"]):
            break
        R = ray
        c0, g0 = R["c"], grad[R["i"]]
        ur, uz = c0 * R["tr"], c0 * R["tz"]
        h = cut(np.full(len(c0), deltas), R["r"], R["z"], ur, uz, R["i"])
        half = 0.5 * h
        zm, tzm = R["z"] + half * uz, R["tz"] - half * g0 / c0 ** 2
        im = segment(zm, tzm)
        c1, g1 = speed(zm, im), grad[im]
        p1 = R["p"]                                    # no curvature inside a linear layer
        u1r, u1z = c1 * R["tr"], c1 * tzm
        h1 = cut(h, R["r"], R["z"], u1r, u1z, R["i"])
        w1 = h1 / (2.0 * half)
        w0 = 1.0 - w1
        u2r, u2z = w0 * ur + w1 * u1r, w0 * uz + w1 * u1z
        h2 = cut(h1, R["r"], R["z"], u2r, u2z, R["i"])
        rn, zn = R["r"] + h2 * u2r, R["z"] + h2 * u2z
        for level in (z[R["i"]], z[R["i"] + 1]):       # end on the knot exactly
            zn = np.where(np.abs(zn - level) < 1e-7, level, zn)
        top, bot = zn <= 1e-7, zn >= D - 1e-7
        rn = np.where(np.abs(rn - rbox) < 1e-6, rbox, rn)
        a, b = h2 * w0, h2 * w1
        tz2 = R["tz"] - a * g0 / c0 ** 2 - b * g1 / c1 ** 2
        N = dict(R, r=rn, z=zn, tz=tz2, tau=R["tau"] + a / c0 + b / c1, q=R["q"] + a * c0 * R["p"] + b * c1 * p1)
        N["i"] = segment(zn, tz2)
        N["c"] = speed(zn, N["i"])
        moved = N["i"] != R["i"]
        jump = grad[N["i"]] - g0
        with np.errstate(divide="ignore", invalid="ignore"):
            rm = R["tr"] / tz2
            kick = rm * (2.0 * jump * R["tr"] - rm * jump * tz2) / N["c"]
        N["p"] = np.where(moved, R["p"] - N["q"] * kick, R["p"])
        _exact_beam(field, R, N, Rz, Rr, first, omega, gauss, coherent, e.freq0)
        # boundary reflection: flat surfaces, so only the profile's gradient bends the beam
        hit = top | bot
        tz3 = np.where(hit, -tz2, tz2)
        g = grad[N["i"]]
        with np.errstate(divide="ignore", invalid="ignore"):
            nz = np.where(top, -1.0, 1.0)              # outward normal
            Th = nz * tz2
            Tg = R["tr"]
            cnj = -(g * (-N["c"] * R["tr"] - N["c"] * R["tr"]))
            csj = -(g * (N["c"] * tz3 - N["c"] * tz2))
            cnj = np.where(top, -cnj, cnj)
            rmr = Tg / Th
            bend = rmr * (2.0 * cnj - rmr * csj) / N["c"] ** 2
        N["p"] = np.where(hit, N["p"] + N["q"] * bend, N["p"])
        kx, kz = omega * Tg, omega * Th
        kzp = np.sqrt((kx * kx).astype(np.complex128) - (omega / cbot) ** 2)
        refl = -(kzp - 1j * kz * e.bot.rho) / (kzp + 1j * kz * e.bot.rho)
        N["ph"] = np.where(top & ~bot, N["ph"] + np.pi, np.where(bot, N["ph"] + np.angle(refl), N["ph"]))
        N["amp"] = np.where(bot, N["amp"] * np.abs(refl), N["amp"])
        N["tz"] = tz3
        N["i"] = segment(zn, np.where(hit, tz3, tz2))
        N["c"] = speed(zn, N["i"])
        keep = (np.abs(rn) < rbox) & (np.abs(zn) < zbox) & (N["amp"] >= 0.005)
        ray = {f: v[keep] for f, v in N.items()}
    return field[None]


def _exact_beam(field, R, N, Rz, Rr, first, omega, gauss, coherent, freq):
    """One step of every ray: its beam at the receiver columns in [r0, r1)."""
    tr, tz = N["r"] - R["r"], N["z"] - R["z"]
    L = np.hypot(tr, tz)
    N["caus"] = R["caus"] + np.where(_caustic(R["qold"], R["q"]), 0.5 * np.pi, 0.0)
    N["qold"] = R["q"]
    with np.errstate(divide="ignore", invalid="ignore"):
        tr, tz = tr / L, tz / L
    lo, hi = np.minimum(R["r"], N["r"]), np.maximum(R["r"], N["r"])
    j0 = np.maximum(np.searchsorted(Rr, lo, "left"), first)
    j1 = np.searchsorted(Rr, hi, "left")
    reach = np.maximum(np.abs(R["q"]), np.abs(N["q"])) * R["rq"] / np.abs(tr)
    floor = np.minimum(0.2 * freq * N["tau"], np.pi * R["c"] / freq) if gauss else np.zeros(len(L))
    reach = np.maximum(reach, floor) * (4.0 if gauss else 1.0)
    flat = np.abs(tr) > 0.50001
    zlo = np.where(flat, np.minimum(R["z"], N["z"]) - reach, -np.inf)
    zhi = np.where(flat, np.maximum(R["z"], N["z"]) + reach, np.inf)
    k0, k1 = np.searchsorted(Rz, zlo, "left"), np.searchsorted(Rz, zhi, "right")
    cols = np.maximum(j1 - j0, 0)
    who = np.repeat(np.arange(len(L)), cols)
    j = np.arange(len(who)) - np.repeat(np.cumsum(cols) - cols, cols) + j0[who]
    rows = np.maximum(k1 - k0, 0)[who]
    pair = np.repeat(np.arange(len(who)), rows)
    iz = np.arange(len(pair)) - np.repeat(np.cumsum(rows) - rows, rows) + k0[who][pair]
    w, ir = who[pair], j[pair]
    dr, dz = Rr[ir] - R["r"][w], Rz[iz] - R["z"][w]
    s = (dr * tr[w] + dz * tz[w]) / L[w]
    d = np.abs(-dr * tz[w] + dz * tr[w])
    q = R["q"][w] + s * (N["q"] - R["q"])[w]
    sig0 = np.abs(q * R["rq"][w])
    sig = np.maximum(sig0, floor[w]) if gauss else sig0
    ok = d < sig * (4.0 if gauss else 1.0)
    w, ir, iz, s, d, q, sig, sig0 = (v[ok] for v in (w, ir, iz, s, d, q, sig, sig0))
    amp = R["ratio"][w] * np.sqrt(N["c"][w]) * R["amp"][w] / np.sqrt(np.abs(q))
    wt = np.exp(-0.5 * (d / sig) ** 2) * (sig0 / sig) if gauss else (sig - d) / sig
    tau = R["tau"][w] + s * (N["tau"] - R["tau"])[w]
    if coherent:
        ph = np.where(_caustic(R["q"][w], q), N["caus"][w] + 0.5 * np.pi, R["ph"][w] + N["caus"][w])
        v = amp * wt * np.exp(-1j * (omega * tau - ph))
    else:
        v = amp * amp * wt * (math.sqrt(2.0 * np.pi) if gauss else 1.0) + 0j
    np.add.at(field, (iz, ir), v)
