"""The work that users of this framework have it do, as timed cases.

Each case is one pass through the public Python view of the C ABI
(`asteroid_amd.api.Context`): chi^2 of candidate models, the -plot curves, the
simplex searches and reoptimisations, RMSD confidence intervals, batches of
light curves and the serving loop.  Sizes are those of the benchmark
workloads, the reference's own launch shapes (256 simplexes per block, 224
blocks, 20000 plotting points) and ragged ones between them.
"""
import math

import numpy as np
import torch

from asteroid_amd import abi, api, flops, synth, variants

PREC = {"fp64": abi.PREC_FP64, "f32simplex": abi.PREC_F32SIMPLEX, "mixed": abi.PREC_MIXED}

# name -> (variant, TIME_STEP in days)
VARIANTS = {
    "ls_torque": (variants.ls_torque, 1e-2),
    "ls": (lambda p, ts: variants.make_variant(False, precision=p, time_step=ts), 1e-2),
    "bc": (variants.bc_free, 5e-3),
    "bc_torque": (lambda p, ts: variants.make_variant(True, True, precision=p, time_step=ts), 1e-2),
    "bw_torque": (variants.bw_ball_torque, 1e-2),
    "trend_torque": (variants.ls_torque_trend, 1e-2),
    "torque2": (variants.ls_torque2, 1e-2),
    "bc_rotate": (variants.bc_rotate, 1e-2),
    "rect": (variants.rect, 1e-2),
    "nudge_torque": (variants.ls_torque_nudge, 1e-2),
    "segment3": (variants.ls_segments, 1e-2),
}


def listed():
    return [
        # One model's chi^2 on a short night's curve: the driver's and an
        # outer optimiser's single evaluation, all latency.
        dict(name="chi2_one", kind="chi2", variant="ls_torque", precision="fp64", n_obs=57, span=1.0, filters=1,
             models=1, noalloc=False),
        # A candidate list screened inside a loop that may not allocate.
        dict(name="chi2_list_noalloc", kind="chi2", variant="bc", precision="mixed", n_obs=818, span=5.0, filters=3,
             models=999, noalloc=True),
        # A grid of candidates: the evaluator at full width, FP64.
        dict(name="chi2_grid", kind="chi2", variant="ls_torque", precision="fp64", n_obs=400, span=3.0, filters=1,
             models=131072, noalloc=False),
        # The driver's -plot: one best model on the reference's 20000 points,
        # then the periodogram of its minima.
        dict(name="plot_one", kind="plot", variant="ls_torque", precision="f32simplex", n_obs=400, span=3.0,
             filters=1, models=1, points=20000),
        # Curves of a set of accepted models, to draw a band around a fit.
        dict(name="plot_band", kind="plot", variant="bc", precision="fp64", n_obs=818, span=5.0, filters=3,
             models=257, points=4001),
        # The small FP64 search: 4096 random starts.
        dict(name="search_small", kind="fit", variant="ls_torque", precision="fp64", n_obs=400, span=3.0, filters=1,
             groups=16, group_size=256, nstages=1, budget=80, reopt=False),
        # The reference's own launch: 224 blocks of 256, float simplex, two
        # stages (a random search and its reseeded second stage).
        dict(name="search_two_stage", kind="fit", variant="ls_torque", precision="f32simplex", n_obs=400, span=3.0,
             filters=1, groups=224, group_size=256, nstages=2, budget=50, reopt=False),
        # The Stage One random search with the chip full, mixed form.
        dict(name="search_full", kind="fit", variant="ls_torque", precision="mixed", n_obs=400, span=3.0, filters=1,
             groups=1024, group_size=256, nstages=1, budget=100, reopt=False),
        # Stage Two: reoptimisation of one start, relaxed brightness ellipsoid.
        dict(name="reopt_bc", kind="fit", variant="bc", precision="mixed", n_obs=818, span=5.0, filters=3,
             groups=13, group_size=256, nstages=1, budget=80, reopt=True),
        # Confidence intervals around a solution.
        dict(name="rmsd", kind="rmsd", variant="ls_torque", precision="f32simplex", n_obs=400, span=3.0, filters=1,
             groups=512, group_size=256, samples=6),
        # A night's batch of uneven curves: 60/30/10% LS+torque, BC, ball, and
        # a Stage Three (NUDGE) reoptimisation among them.
        dict(name="batch_uneven", kind="jobs", precision="mixed", jobs=11, fits=512, budget=80, least=50, most=1200,
             serve=False),
        # Requests that arrive together at a serving context.
        dict(name="serve_requests", kind="jobs", precision="mixed", jobs=8, fits=1024, budget=50, least=50, most=800,
             serve=True),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


# Model-points of the largest listed case, and the longest serial walk of one
# lane (its observations times the evaluations it does one after another).
MOST_POINTS = 1024 * 256 * 100 * 400
MOST_SERIAL = 70000


def draw(rng):
    kind = rng.choice(["chi2", "chi2", "plot", "fit", "fit", "rmsd", "jobs"])
    if kind == "jobs":
        return dict(kind="jobs", precision=rng.choice(["mixed", "fp64", "f32simplex"]), jobs=rng.randint(3, 11),
                    fits=256 * rng.randint(1, 4), budget=rng.randint(30, 80), least=50, most=_log(rng, 300, 1200),
                    serve=rng.random() < 0.3)
    name = rng.choice(["ls_torque", "ls_torque", "ls_torque", "bc", "bc", *VARIANTS])
    precision = rng.choice(list(PREC))
    if name == "nudge_torque" and precision == "mixed":  # refused: NUDGE has no mixed form
        precision = "fp64"
    if kind == "rmsd" and name == "segment3":  # refused: SEGMENT has no RMSD
        name = "ls_torque"
    n_obs = _log(rng, 50, 2000)
    case = dict(kind=kind, variant=name, precision=precision, n_obs=n_obs, span=round(rng.uniform(1.0, 8.0), 3),
                filters=rng.randint(1, 4))
    if kind == "chi2":
        case["models"] = _log(rng, 1, min(131072, 131072 * 400 // n_obs))
        case["noalloc"] = case["models"] <= abi_noalloc() and rng.random() < 0.3
    elif kind == "plot":
        case["models"], case["points"] = _log(rng, 1, 300), _log(rng, 1000, 20000)
    elif kind == "rmsd":
        case["group_size"] = rng.choice([64, 256, 256, 1024])
        case["samples"] = rng.randint(1, 8)
        case["groups"] = _log(rng, 1, 131072 // case["group_size"])
        case["groups"] = max(1, min(case["groups"], MOST_POINTS // 10 // (n_obs * case["samples"] * case["group_size"])))
    else:
        case["group_size"] = rng.choice([64, 128, 256, 256, 256, 1024])
        case["nstages"], case["reopt"] = rng.randint(1, 2), rng.random() < 0.4
        case["budget"] = max(20, min(rng.randint(20, 100), MOST_SERIAL // (n_obs * case["nstages"])))
        evals = case["budget"] * case["nstages"] * case["group_size"]
        case["groups"] = max(1, min(_log(rng, 1, 262144 // case["group_size"]), MOST_POINTS // (2 * n_obs * evals)))
    return case


def abi_noalloc():
    return 16384  # AST_NOALLOC_MAX_MODELS


# ---------------------------------------------------------------- inputs
def _variant(name, precision):
    make, time_step = VARIANTS[name]
    return make(PREC[precision], time_step)


def _curve(name, precision, seed, n_obs, span, filters):
    """Variant, curve, truth and what the variant needs beside them: a seeded
    ground truth's magnitudes with noise of 0.05 to 0.3 mag."""
    v = _variant(name, precision)
    extra = {}
    if v.n_seg > 1:  # the plain curve cut in thirds; each part starts a little away from the first
        one = variants.make_variant(False, precision=PREC[precision], time_step=v.time_step)
        curve, t1 = synth.make_curve(seed, one, n_obs, span, n_filters=filters)
        at, off = variants.param_positions(one), np.random.default_rng(seed + 1)
        truth = np.array([t1[at[k.split(":")[0]]] + (off.uniform(-0.2, 0.2) if ":" in k else 0.0)
                          for k in variants.param_positions(v)])
        extra["t_segments"] = curve.mjd[0] + (curve.mjd[-1] - curve.mjd[0]) * np.arange(v.n_seg) / v.n_seg
    else:
        curve, truth = synth.make_curve(seed, v, n_obs, span, n_filters=filters)
    if v.nudge:  # four of the truth's brightness minima
        vm = synth.truth_vmod(v, truth, curve.mjd, curve.E, curve.S)
        at = [i - 1 for i in range(2, len(vm)) if vm[i - 1] > vm[i - 2] and vm[i - 1] >= vm[i]] or [len(vm) // 2]
        at = at[::max(1, len(at) // 4)][:4]
        extra["minima"] = (curve.mjd[at].astype(np.float32), vm[at].astype(np.float32))
    return v, curve, truth, extra


def _near(truth, n, seed):
    """n candidate models around a fit, the first the fit itself."""
    r = np.random.default_rng(seed).standard_normal((n, len(truth)))
    r[0] = 0.0
    return truth * (1.0 + 1e-3 * r)


def _job_specs(case, seed):
    rng = np.random.default_rng(seed)
    names = ["ls_torque"] * 6 + ["bc"] * 3 + ["bw_torque", "nudge_torque"]
    for k in range(case["jobs"]):
        name = names[(3 * k) % len(names)]
        precision = case["precision"]
        if name == "nudge_torque" and precision == "mixed":
            precision = "f32simplex"
        n_obs = int(round(math.exp(math.log(case["least"]) + (math.log(case["most"]) - math.log(case["least"]))
                                   * (k + rng.uniform()) / case["jobs"])))
        fits = case["fits"] if not case["serve"] else 256 * (1 + (5 * k) % (case["fits"] // 128))
        yield dict(name=name, precision=precision, n_obs=n_obs, filters=1 + k % 4, span=float(rng.uniform(1.0, 8.0)),
                   seed=int(rng.integers(1 << 30)), fits=fits)


def _jobs(case, seed):
    jobs = []
    for k, s in enumerate(_job_specs(case, seed)):
        v, curve, truth, extra = _curve(s["name"], s["precision"], s["seed"], s["n_obs"], s["span"], s["filters"])
        reopt = int(bool(v.nudge))
        if reopt:
            extra["params0"] = truth * (1.0 + np.random.default_rng(s["seed"] + 2).uniform(-0.02, 0.02, truth.shape))
        jobs.append(dict(space=variants.default_model_space(v, reopt=reopt), curve=curve, n_fits=s["fits"],
                         eval_budget=case["budget"], size_min=1e-10, seed=s["seed"] + 3, tag=k, **extra))
    return jobs


def prepare(case, seed):
    if case["kind"] == "jobs":
        jobs = _jobs(case, seed)
        ctx = api.Context(jobs[0]["space"].variant)
        if case["serve"]:
            ctx.serve_start(max_resident_fits=1 << 16)
        return dict(case=case, ctx=ctx, jobs=jobs)
    v, curve, truth, extra = _curve(case["variant"], case["precision"], seed, case["n_obs"], case["span"],
                                    case["filters"])
    reopt = bool(case.get("reopt")) or case["kind"] == "rmsd"
    ctx = api.Context(v)
    ctx.set_model_space(variants.default_model_space(v, reopt=int(reopt)))
    if "t_segments" in extra:
        ctx.set_segments(extra["t_segments"])
    ctx.upload_curve(curve)
    if "minima" in extra:
        ctx.set_minima(*extra["minima"])
    state = dict(case=case, ctx=ctx, seed=seed)
    if case["kind"] in ("chi2", "plot"):
        state["models"] = _near(truth, case["models"], seed + 4)
    if case["kind"] == "rmsd":
        ctx.set_start(truth)
    elif reopt:
        ctx.set_start(truth * (1.0 + np.random.default_rng(seed + 5).uniform(-0.02, 0.02, truth.shape)))
    return state


# ------------------------------------------------------------------- pass
def _answers(results):
    """The jobs' answers in the jobs' order: best chi^2, best group, best
    parameters and delta_V (one job after another), evaluations and status."""
    rs = sorted(results, key=lambda r: r["tag"])
    return (np.array([r["best_f"] for r in rs]), np.array([r["best_group"] for r in rs]),
            np.concatenate([r["best_params"] for r in rs]), np.concatenate([r["best_dV"] for r in rs]),
            np.array([r["n_evals"] for r in rs]), np.array([r["status"] for r in rs]))


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "chi2":
        return (ctx.chi2_batch_noalloc if case["noalloc"] else ctx.chi2_batch)(state["models"])
    if case["kind"] == "plot":
        t, vmod, chi2, dv = ctx.model_curve(state["models"], n_plot=case["points"])
        fr, height, n_minima = ctx.periodogram(t, vmod[0])
        return t, vmod, chi2, dv, fr, height, n_minima
    if case["kind"] == "rmsd":
        ctx.rng_seed(state["seed"])
        return ctx.rmsd(case["groups"], case["group_size"], case["samples"], dx=0.003)
    if case["kind"] == "fit":
        ctx.rng_seed(state["seed"])
        ctx.run(case["groups"], case["group_size"], nstages=case["nstages"], eval_budget=case["budget"],
                size_min=1e-10)
        return (*ctx.fetch(), *ctx.fetch_lanes())
    if case["serve"]:
        return _answers(ctx.wait_all([ctx.submit(**j) for j in state["jobs"]]).values())
    return _answers(ctx.run_jobs(state["jobs"]))


# ------------------------------------------------------------------- work
def _one(name, precision, n_obs, span, filters):
    """FLOPs of one evaluation on a curve of that size (evenly spaced times
    stand for the drawn ones) and the bytes of its observations."""
    v = _variant(name, precision)
    t = np.arange(n_obs) * (span / n_obs)
    seg = span * np.arange(v.n_seg) / v.n_seg if v.n_seg > 1 else None
    return flops.eval_flops(v, t, seg_t=seg), 96 * n_obs, abi.type_ids(v)["n_params"]


def work(case):
    if case["kind"] == "jobs":
        f = b = 0
        for s in _job_specs(case, 1):
            one, curve, n = _one(s["name"], s["precision"], s["n_obs"], s["span"], s["filters"])
            f += one * s["fits"] * case["budget"]
            b += curve + 8 * (n + s["filters"])
        return dict(bytes=b, flops=f)
    one, curve, n = _one(case["variant"], case["precision"], case["n_obs"], case["span"], case["filters"])
    out = 1 + case["filters"]
    if case["kind"] == "chi2":
        return dict(bytes=curve + 8 * case["models"] * (n + out), flops=one * case["models"])
    if case["kind"] == "plot":
        grid, _, _ = _one(case["variant"], case["precision"], case["points"], case["span"], 1)
        return dict(bytes=curve + 8 * case["points"] + 8 * case["models"] * (n + out + case["points"]),
                    flops=(one + grid) * case["models"])
    if case["kind"] == "rmsd":
        lanes = case["groups"] * case["group_size"]
        return dict(bytes=curve + 8 * case["groups"] * n, flops=one * lanes * case["samples"])
    fits = case["groups"] * case["group_size"]
    return dict(bytes=curve + 8 * case["groups"] * (n + out) + 24 * fits,
                flops=one * fits * case["budget"] * case["nstages"])


# ------------------------------------------------------------------ exact
def _rk4(y, h, rhs):
    k1 = rhs(y)
    k2 = rhs([a + 0.5 * h * k for a, k in zip(y, k1)])
    k3 = rhs([a + 0.5 * h * k for a, k in zip(y, k2)])
    k4 = rhs([a + h * k for a, k in zip(y, k3)])
    return [a + h / 6.0 * (p + 2.0 * q + 2.0 * r + s) for a, p, q, r, s in zip(y, k1, k2, k3, k4)]


def _walk(v, p, t):
    """Euler angles (phi, theta, psi), each (models, points), of the models p
    (dict of (models,) tensors) at the times t: classical RK4 with the
    framework's steps (int(dt / TIME_STEP + 1) equal ones per interval)."""
    bt, ct = p["b_tumb"], p["c_tumb"]
    i_s = (1.0 + bt * bt) / (bt * bt + ct * ct)
    i_i = (1.0 + ct * ct) / (bt * bt + ct * ct)
    psi, spin = p["psi_0"], p["L"]
    theta = torch.asin(torch.sqrt((p["Es"] - 1.0) / (torch.sin(psi) ** 2 * (1.0 / i_i - 1.0 / i_s) + 1.0 / i_s - 1.0)))
    if v.torque or v.torque2:
        m0, m1, m2 = (i_s - 1.0) / i_i, (1.0 - i_i) / i_s, i_i - i_s

        def rhs(torque):
            def f(y):
                wi, ws, wl, _, th, ps = y
                sp, cp = torch.sin(ps), torch.cos(ps)
                dphi = (wi * sp + ws * cp) / torch.sin(th)
                return [m0 * ws * wl + torque[0], m1 * wl * wi + torque[1], m2 * wi * ws + torque[2], dphi,
                        wi * cp - ws * sp, wl - dphi * torch.cos(th)]
            return f

        y = [spin / i_i * torch.sin(theta) * torch.sin(psi), spin / i_s * torch.sin(theta) * torch.cos(psi),
             spin * torch.cos(theta), p["phi_0"], theta, psi]
        f = rhs((p["Ti"], p["Ts"], p["Tl"]))
        pick = (3, 4, 5)
    else:
        a, b = 0.5 * (1.0 / i_i + 1.0 / i_s), 0.5 * (1.0 / i_i - 1.0 / i_s)

        def f(y):
            dphi = spin * (a - b * torch.cos(2.0 * y[2]))
            return [dphi, spin * b * torch.sin(y[1]) * torch.sin(2.0 * y[2]), torch.cos(y[1]) * (spin - dphi)]

        y = [p["phi_0"], theta, psi]
        pick = (0, 1, 2)
    seen = [[y[k]] for k in pick]
    for t1, t2 in zip(t[:-1], t[1:]):
        steps = int((t2 - t1) / v.time_step + 1)
        for _ in range(steps):
            y = _rk4(y, float(t2 - t1) / steps, f)
        for s, k in zip(seen, pick):
            s.append(y[k])
    return [torch.stack(s, 1) for s in seen]


def _magnitudes(v, p, t, e, s):
    """Magnitudes (models, points) of LS-ellipsoid models (with or without
    torque and photometric b, c)."""
    phi, theta, psi = _walk(v, p, t)
    col = {k: x[:, None] for k, x in p.items()}
    mx, my, mz = (torch.sin(col["theta_M"]) * torch.cos(col["phi_M"]),
                  torch.sin(col["theta_M"]) * torch.sin(col["phi_M"]), torch.cos(col["theta_M"]))
    r = torch.sqrt(mx * mx + mz * mz)
    axes = [(mz / r, 0.0 * r, -mx / r), (-my * mx / r, r, -my * mz / r), (mx, my, mz)]  # x, y, z of the spin frame
    cf, sf, ct, st, cp, sp = (torch.cos(phi), torch.sin(phi), torch.cos(theta), torch.sin(theta), torch.cos(psi),
                              torch.sin(psi))

    def body(w):  # components of the unit vectors w along the body's b, c, a
        x, y, z = (sum(a[k] * w[:, k] for k in range(3)) for a in axes)
        return ((cf * cp - sf * ct * sp) * x + (sf * cp + cf * ct * sp) * y + st * sp * z,
                (-cf * sp - sf * ct * cp) * x + (-sf * sp + cf * ct * cp) * y + st * cp * z,
                sf * st * x - cf * st * y + ct * z)

    b, c = (col["b"], col["c"]) if v.bc else (col["b_tumb"], col["c_tumb"])
    eb, ec, ea = body(e)
    sb, sc, sa = body(s)
    eb, ec, sb, sc = eb / b, ec / c, sb / b, sc / c
    s_s, s_e = torch.sqrt(sb * sb + sc * sc + sa * sa), torch.sqrt(eb * eb + ec * ec + ea * ea)
    cos_al = (sb * eb + sc * ec + sa * ea) / (s_s * s_e)
    sin_al = torch.sqrt(1.0 - cos_al * cos_al)
    both = torch.sqrt(s_s * s_s + s_e * s_e + 2.0 * s_s * s_e * cos_al)
    cl, sl = (s_s + s_e * cos_al) / both, s_e * sin_al / both
    cd, sd = cl * cos_al + sl * sin_al, sl * cos_al - cl * sin_al  # of lambda' - alpha'
    f = cd + cl + sl * sd * torch.log((1.0 + cl) * (1.0 + cd) / (sl * -sd))
    return -2.5 * torch.log10(b * c * s_s * s_e / both * f)


def exact(case, seed):
    if case["kind"] not in ("chi2", "plot") or case["variant"] not in ("ls_torque", "ls", "bc", "bc_torque"):
        return None  # a search follows its own random stream; the rarer brightness forms are left to the tests
    v, curve, truth, _ = _curve(case["variant"], case["precision"], seed, case["n_obs"], case["span"],
                                case["filters"])
    if case["models"] * flops.rk4_steps(curve.mjd, v.time_step) > 1e8:
        return None
    names = variants.param_positions(v)
    models = torch.from_numpy(_near(truth, case["models"], seed + 4))
    dof = case["n_obs"] - len(names) - case["filters"]
    e, s = (torch.from_numpy(np.ascontiguousarray(x)) for x in (curve.E, curve.S))
    mag, w = (torch.from_numpy(np.asarray(x, np.float64)) for x in (curve.V, curve.w))
    chi2, dv = np.zeros(case["models"]), np.zeros((case["models"], case["filters"]))
    for a in range(0, case["models"], 16384):
        part = slice(a, min(a + 16384, case["models"]))
        res = mag - _magnitudes(v, {k: models[part, i] for k, i in names.items()}, curve.mjd, e, s)
        total = 0.0
        for m in range(case["filters"]):
            at = torch.from_numpy(curve.filter == m)
            r, wm = res[:, at], w[at]
            d = (r * wm).sum(1) / wm.sum()
            total = total + (((r - d[:, None]) ** 2) * wm).sum(1)
            dv[part, m] = d.numpy()
        chi2[part] = (total / dof).numpy()
    if case["kind"] == "chi2":
        return chi2, dv
    t = np.linspace(curve.mjd[0], curve.mjd[-1], case["points"])
    e, s = (torch.from_numpy(x / np.linalg.norm(x, axis=1, keepdims=True)) for x in synth.quad_interp(curve.eph, t))
    vmod = _magnitudes(v, {k: models[:, i] for k, i in names.items()}, t, e, s).numpy() + dv[:, :1]
    return t, vmod, chi2, dv, None, None, None
