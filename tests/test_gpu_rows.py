"""The evaluator with several lanes per model (ast_rows.h) against the oracle,
bit for bit: chi^2 batches and fits at the sizes where the number of lanes per
model changes (16 up to 4096 models, 4 up to 16384, then one), curves whose
length leaves every kind of remainder in a batch of 16 or 4 points, curves on
short grids, and a run whose groups end their stages in separate launches."""
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
