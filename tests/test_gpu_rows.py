"""The evaluator with several lanes per model (ast_rows.h) against the oracle,
bit for bit: chi^2 batches and fits at the sizes where the number of lanes per
model or the use of teams changes (1024, 4096, 8192 and 16384 models), curves
whose length leaves every kind of remainder in a batch of 16 or 4 points or in a
team's chunk of steps, curves on short grids, and a run whose groups end their
stages in separate launches."""
import numpy as np
import pytest

import oracle
from asteroid_amd import abi, api, synth, variants

pytestmark = pytest.mark.gpu

PRECS = {"fp64": abi.PREC_FP64, "f32simplex": abi.PREC_F32SIMPLEX}


def _problem(make, prec, n_obs, filters, span=1.5, seed=5):
    v = make(PRECS[prec])
    curve, truth = synth.make_curve(seed, v, n_obs, span, n_filters=filters)
    space = variants.default_model_space(v)
    return v, curve, truth, space, oracle.Problem(space, curve)


def _models(pb, n):
    x = np.random.default_rng(2).uniform(0.0, 1.0, (2 * n + 64, pb.space.n_params))
    p, rc = pb.x2params(x)
    return p[rc == 0][:n]


def _ctx(v, space, curve):
    ctx = api.Context(v)
    ctx.set_model_space(space)
    ctx.upload_curve(curve)
    return ctx


def _same(got, want):
    np.testing.assert_array_equal(np.asarray(got), np.asarray(want))  # NaN equal to NaN


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4096, 4097, 16384, 16387])
def test_chi2_where_the_lanes_per_model_change(n):
    v, curve, _, space, pb = _problem(variants.ls_torque, "fp64", 21, 2)
    p = _models(pb, n)
    with _ctx(v, space, curve) as ctx:
        got = ctx.chi2_batch(p)
    for g, w in zip(got, pb.chi2(p)):
        _same(g, w)


@pytest.mark.parametrize("make", [variants.ls_torque, variants.bc_free, variants.ls_torque2], ids=["tq", "bc", "tq2"])
@pytest.mark.parametrize("n_obs,filters", [(19, 1), (20, 1), (32, 3), (33, 4), (47, 6)])
def test_curve_length_remainders(make, n_obs, filters):
    v, curve, _, space, pb = _problem(make, "f32simplex", n_obs, filters)
    p = _models(pb, 4200)
    want = pb.chi2(p)
    with _ctx(v, space, curve) as ctx:
        for n in (70, 4200):  # 16 and 4 lanes per model
            got = ctx.chi2_batch(p[:n])
            _same(got[0], want[0][:n])
            _same(got[1], want[1][:n])
        for n_plot in (2, 17, 31):
            for g, w in zip(ctx.model_curve(p[:5], n_plot=n_plot), pb.model_curve(p[:5], n_plot=n_plot)):
                _same(g, w)


@pytest.mark.parametrize("prec", list(PRECS))
@pytest.mark.parametrize("groups,group_size,nstages", [(1, 64, 1), (3, 64, 3), (16, 256, 1), (17, 256, 2),
                                                       (16, 1024, 1), (65, 256, 2)])
def test_fits_where_the_lanes_per_model_change(prec, groups, group_size, nstages):
    v, curve, _, space, pb = _problem(variants.ls_torque, prec, 21, 1)
    run = dict(nstages=nstages, n_steps=12, eval_budget=24)
    with _ctx(v, space, curve) as ctx:
        ctx.rng_seed(4)
        ctx.run(groups, group_size, ticks_per_launch=7 if nstages == 3 else 0, **run)
        got = ctx.fetch() + ctx.fetch_lanes()
    want = pb.run(groups, group_size, seed=4, form=oracle.CANON, n_threads=8, **run)
    for g, k in zip(got, ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")):
        _same(g, want[k])


def test_refilled_fits_on_few_lanes():
    v, curve, _, space, pb = _problem(variants.ls_torque, "fp64", 21, 1)
    run = dict(nstages=1, n_steps=12, eval_budget=24)
    with _ctx(v, space, curve) as ctx:
        ctx.rng_seed(4)
        ctx.run(7, 64, resident_groups=2, **run)
        got = ctx.fetch() + ctx.fetch_lanes()
    want = pb.run(7, 64, seed=4, form=oracle.CANON, n_threads=8, **run)
    for g, k in zip(got, ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")):
        _same(g, want[k])


BUILDS = {
    "ls": lambda p: variants.make_variant(False, precision=p),
    "bc": variants.bc_free,
    "bc_torque": lambda p: variants.make_variant(True, True, precision=p),
    "bw": lambda p: variants.make_variant(False, False, True, precision=p),
    "bw_torque": variants.bw_ball_torque,
    "trend": variants.ls_torque_trend,
    "torque2": variants.ls_torque2,
    "bc_rotate": variants.bc_rotate,
    "bc_rotate_torque": lambda p: variants.bc_rotate(p, torque=True),
    "rect": variants.rect,
    "rect_torque": lambda p: variants.rect(p, torque=True),
    "nudge": variants.ls_torque_nudge,
    "nudge_bc": lambda p: variants.ls_torque_nudge(p, bc=True),
    **{f"seg{n}{'_onele' if le else ''}{'_torque' if tq else ''}{'_bc' if bc else ''}":
       (lambda p, n=n, le=le, tq=tq, bc=bc: variants.ls_segments(p, n_seg=n, one_le=le, torque=tq, bc=bc))
       for n in (3, 4) for le in (True, False) for tq in (False, True) for bc in (False, True)},
}


@pytest.mark.parametrize("groups", [20, 65])  # 5120 fits: 4 lanes per model; 16640: one
@pytest.mark.parametrize("name", list(BUILDS))
def test_every_build_on_four_lanes_and_one(name, groups):
    v = BUILDS[name](abi.PREC_FP64)
    base = variants.make_variant(bool(v.torque), bool(v.bc), precision=abi.PREC_FP64) if v.n_seg > 1 else v
    curve, truth = synth.make_curve(7, base, 56, 1.5, n_filters=2)
    space = variants.default_model_space(v)
    keep = {}
    with api.Context(v) as ctx:
        ctx.set_model_space(space)
        if v.n_seg > 1:
            keep["t_start"] = curve.mjd[0] - 0.01 + 1.5 * np.arange(v.n_seg) / v.n_seg
            ctx.set_segments(keep["t_start"])
        ctx.upload_curve(curve)
        if v.nudge:
            keep["minima"] = (curve.mjd[[9, 30]].astype(np.float32), curve.V[[9, 30]])
            ctx.set_minima(*keep["minima"])
        pb = oracle.Problem(space, curve, **keep)
        run = dict(nstages=1, n_steps=4, eval_budget=space.n_params + 6)
        ctx.rng_seed(8)
        ctx.run(groups, 256, **run)
        got = ctx.fetch() + ctx.fetch_lanes()
        p = _models(pb, 200)
        chi2 = ctx.chi2_batch(np.resize(p, (groups * 256, p.shape[1])))
    want = pb.run(groups, 256, seed=8, form=oracle.CANON, n_threads=8, **run)
    for g, k in zip(got, ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")):
        _same(g, want[k])
    want = pb.chi2(p)
    n = len(want[0])
    for a in (0, (groups * 256 // n - 1) * n):
        _same(chi2[0][a:a + n], want[0])
        if not v.nudge:  # delta_V of a failed NUDGE model is the caller's
            _same(chi2[1][a:a + n], want[1])


@pytest.mark.parametrize("fits,group_size", [(256, 64), (2048, 256), (5120, 256)])  # 16 lanes, teams of 4, 4 or teams
@pytest.mark.parametrize("name", list(BUILDS))
def test_every_build_on_few_models(name, fits, group_size):
    v = BUILDS[name](abi.PREC_FP64)
    base = variants.make_variant(bool(v.torque), bool(v.bc), precision=abi.PREC_FP64) if v.n_seg > 1 else v
    curve, truth = synth.make_curve(7, base, 61, 1.5, n_filters=2)
    space = variants.default_model_space(v)
    keep = {}
    with api.Context(v) as ctx:
        ctx.set_model_space(space)
        if v.n_seg > 1:
            keep["t_start"] = curve.mjd[0] - 0.01 + 1.5 * np.arange(v.n_seg) / v.n_seg
            ctx.set_segments(keep["t_start"])
        ctx.upload_curve(curve)
        if v.nudge:
            keep["minima"] = (curve.mjd[[9, 30]].astype(np.float32), curve.V[[9, 30]])
            ctx.set_minima(*keep["minima"])
        pb = oracle.Problem(space, curve, **keep)
        run = dict(nstages=1, n_steps=4, eval_budget=space.n_params + 6)
        ctx.rng_seed(8)
        ctx.run(fits // group_size, group_size, **run)
        got = ctx.fetch() + ctx.fetch_lanes()
        p = _models(pb, 70)
        n = len(p)
        chi2 = ctx.chi2_batch(np.resize(p, (fits + n, p.shape[1])))
        plots = [(n, 37, ctx.model_curve(p, n_plot=37))]
        if v.n_seg > 1:  # a grid without a point in every segment is refused
            with pytest.raises(api.AsteroidError):
                ctx.model_curve(p[:3], n_plot=2)
        else:
            plots.append((3, 2, ctx.model_curve(p[:3], n_plot=2)))
        many = ctx.model_curve(np.resize(p, (1024 + n, p.shape[1])), n_plot=19)
    want = pb.run(fits // group_size, group_size, seed=8, form=oracle.CANON, n_threads=8, **run)
    for g, k in zip(got, ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")):
        _same(g, want[k])
    want = pb.chi2(p)
    last = (fits // n) * n
    for a, m in ((0, n), (last - n, n), (last, fits + n - last)):
        m = min(m, n)
        _same(chi2[0][a:a + m], want[0][:m])
        if not v.nudge:  # delta_V of a failed NUDGE model is the caller's
            _same(chi2[1][a:a + m], want[1][:m])
    a = (1024 // n) * n
    plots += [(n, 19, [many[0]] + [g[k:k + n] for g in many[1:]]) for k in (0, a)]
    for m, n_plot, got in plots:
        t, vmod, f, dv = pb.model_curve(p[:m], n_plot=n_plot)
        _same(got[0], t)
        _same(got[2], f)
        ok = f < 1e29  # a failed NUDGE model has no delta_V
        _same(got[1][ok], vmod[ok])
        _same(got[3][ok], dv[ok])


@pytest.mark.parametrize("make", [variants.ls_torque, variants.bc_free], ids=["tq", "bc"])
@pytest.mark.parametrize("n", [1023, 1024, 1025, 4095, 4096, 4097, 8192, 8193])
def test_chi2_where_teams_begin_and_end(make, n):
    v, curve, _, space, pb = _problem(make, "f32simplex", 18, 3, span=2.5)
    p = _models(pb, 300)
    with _ctx(v, space, curve) as ctx:
        got = ctx.chi2_batch(np.resize(p, (n, p.shape[1])))
    want = pb.chi2(p)
    for g, w in zip(got, want):
        _same(g, np.resize(w, (n,) + w.shape[1:]))


@pytest.mark.parametrize("make", [variants.ls_torque, variants.bc_free], ids=["tq", "bc"])
@pytest.mark.parametrize("groups,group_size,resident", [(30, 64, 3), (9, 256, 4), (30, 256, 8), (40, 256, 24)])
def test_refilled_fits_on_teams(make, groups, group_size, resident):
    v, curve, _, space, pb = _problem(make, "f32simplex", 18, 3, span=2.5)
    run = dict(nstages=1, n_steps=12, eval_budget=24)
    with _ctx(v, space, curve) as ctx:
        ctx.rng_seed(4)
        ctx.run(groups, group_size, resident_groups=resident, **run)
        got = ctx.fetch() + ctx.fetch_lanes()
    want = pb.run(groups, group_size, seed=4, form=oracle.CANON, n_threads=8, **run)
    for g, k in zip(got, ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")):
        _same(g, want[k])


@pytest.mark.parametrize("n", [65536, 65537, 131071])  # in one launch, in two halves
def test_chi2_batches_in_halves(n):
    v, curve, _, space, pb = _problem(variants.ls_torque, "fp64", 18, 2)
    p = _models(pb, 301)
    with _ctx(v, space, curve) as ctx:
        got = ctx.chi2_batch(np.resize(p, (n, p.shape[1])))
    for g, w in zip(got, pb.chi2(p)):
        _same(g, np.resize(w, (n,) + w.shape[1:]))
