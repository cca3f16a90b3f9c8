"""The one-lane kernels, which launches of more than 16384 fits (models) or 4096
curves run, in the forms that smaller launches no longer reach: register
budgets, refill, replayed cycles, group sizes from 64 to 1024, the mixed form,
more than 65536 fits, and batches.  A fit's trajectory depends on its own index
only, so the oracle's run of the first and last groups, or a run of a few groups
on several lanes per fit, gives what the same fits of a large run must be, bit
for bit."""
import numpy as np
import pytest

import oracle
from asteroid_amd import abi, api, synth, variants

from .test_gpu_rows import BUILDS, _models, _same

pytestmark = pytest.mark.gpu

PRECS = {"fp64": abi.PREC_FP64, "f32simplex": abi.PREC_F32SIMPLEX, "mixed": abi.PREC_MIXED}
NAMES = ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")


def _problem(make, prec, n_obs=21, filters=1):
    v = make(PRECS[prec])
    curve, _ = synth.make_curve(5, v, n_obs, 1.5, n_filters=filters)
    return v, curve, variants.default_model_space(v)


def _run(v, curve, space, groups, group_size, waves=None, **run):
    with api.Context(v) as ctx:
        if waves:
            ctx.set_waves(v, curve.n_filters, waves)
        ctx.set_model_space(space)
        ctx.upload_curve(curve)
        ctx.rng_seed(4)
        ctx.run(groups, group_size, **run)
        return ctx.fetch() + ctx.fetch_lanes()


def _first(got, groups, group_size):
    return [g[:groups] for g in got[:3]] + [g[:groups * group_size] for g in got[3:]]


def _oracle(curve, space, groups, group_size, **run):
    want = oracle.Problem(space, curve).run(groups, group_size, seed=4, form=oracle.CANON, n_threads=8, **run)
    return [want[k] for k in NAMES]


def _equal(got, want):
    for g, w in zip(got, want):
        _same(g, w)


@pytest.mark.parametrize("waves", [4, 3, 2])
@pytest.mark.parametrize("prec", list(PRECS))
@pytest.mark.parametrize("groups,nstages,graphs", [(65, 1, False), (65, 2, True), (257, 1, False)])
def test_register_budgets(waves, prec, groups, nstages, graphs):
    v, curve, space = _problem(variants.ls_torque, prec)
    run = dict(nstages=nstages, n_steps=12, eval_budget=24)
    got = _run(v, curve, space, groups, 256, waves=waves, use_graphs=graphs, ticks_per_launch=11, **run)
    if prec == "mixed":  # no oracle: the same fits with 16 and with 4 lanes each
        _equal(_first(got, 3, 256), _run(v, curve, space, 3, 256, **run))
        _equal(_first(got, 20, 256), _run(v, curve, space, 20, 256, **run))
    else:
        _equal(_first(got, 20, 256), _oracle(curve, space, 20, 256, **run))


@pytest.mark.parametrize("waves", [4, 2])
@pytest.mark.parametrize("prec", list(PRECS))
@pytest.mark.parametrize("groups,resident,graphs", [(72, 65, False), (150, 65, True), (300, 260, False)])
def test_refill(waves, prec, groups, resident, graphs):
    v, curve, space = _problem(variants.ls_torque, prec, n_obs=18, filters=3)
    run = dict(nstages=1, n_steps=12, eval_budget=24)
    got = _run(v, curve, space, groups, 256, waves=waves, resident_groups=resident, use_graphs=graphs,
               ticks_per_launch=9, **run)
    if prec == "mixed":
        _equal(got, _run(v, curve, space, groups, 256, **run))  # without refill
        _equal(_first(got, 16, 256), _run(v, curve, space, 16, 256, **run))  # on several lanes
    elif groups == 72:
        _equal(got, _oracle(curve, space, groups, 256, **run))
    else:
        _equal(got, _run(v, curve, space, groups, 256, **run))
        _equal(_first(got, 16, 256), _oracle(curve, space, 16, 256, **run))


@pytest.mark.parametrize("prec", list(PRECS))
@pytest.mark.parametrize("groups,group_size", [(257, 64), (129, 128), (33, 512), (17, 1024), (65, 1024)])
def test_group_sizes(prec, groups, group_size):
    v, curve, space = _problem(variants.bc_free, prec, n_obs=20, filters=2)
    for nstages in (1, 3):
        run = dict(nstages=nstages, n_steps=10, eval_budget=20)
        got = _run(v, curve, space, groups, group_size, **run)
        few = max(1, 2048 // group_size)
        small = _run(v, curve, space, few, group_size, **run)
        _equal(_first(got, few, group_size), small)
        if prec != "mixed":
            _equal(small, _oracle(curve, space, few, group_size, **run))


@pytest.mark.parametrize("prec", ["f32simplex", "mixed"])
@pytest.mark.parametrize("name", list(BUILDS))
def test_every_build_in_float(name, prec):
    v = BUILDS[name](PRECS[prec])
    if v.nudge and prec == "mixed":
        pytest.skip("NUDGE has no mixed form")
    base = variants.make_variant(bool(v.torque), bool(v.bc), precision=PRECS[prec]) if v.n_seg > 1 else v
    curve, _ = synth.make_curve(7, base, 56, 1.5, n_filters=2)
    space = variants.default_model_space(v)
    run = dict(nstages=1, n_steps=4, eval_budget=space.n_params + 6)
    keep, got = {}, {}
    with api.Context(v) as ctx:
        ctx.set_model_space(space)
        if v.n_seg > 1:
            keep["t_start"] = curve.mjd[0] - 0.01 + 1.5 * np.arange(v.n_seg) / v.n_seg
            ctx.set_segments(keep["t_start"])
        ctx.upload_curve(curve)
        if v.nudge:
            keep["minima"] = (curve.mjd[[9, 30]].astype(np.float32), curve.V[[9, 30]])
            ctx.set_minima(*keep["minima"])
        for groups in (1, 20, 65):  # 16 lanes per model, 4, one
            ctx.rng_seed(8)
            ctx.run(groups, 256, **run)
            got[groups] = _first(ctx.fetch() + ctx.fetch_lanes(), 1, 256)
    _equal(got[20], got[1])
    _equal(got[65], got[1])
    if prec == "f32simplex":
        want = oracle.Problem(space, curve, **keep).run(1, 256, seed=8, form=oracle.CANON, n_threads=8, **run)
        _equal(got[1], [want[k] for k in NAMES])


def test_batch_of_many_fits_equals_each_job_alone():
    jobs = []
    for k, (make, prec, filters) in enumerate([(variants.ls_torque, "fp64", 1), (variants.bc_free, "mixed", 3),
                                               (variants.bw_ball_torque, "f32simplex", 2),
                                               (variants.ls_torque, "mixed", 1), (variants.bc_free, "mixed", 1)]):
        v, curve, space = _problem(make, prec, n_obs=22 + k, filters=filters)
        jobs.append(dict(space=space, curve=curve, n_fits=4096 + 256 * k, nstages=1 + k % 2, n_steps=12, eval_budget=24,
                         seed=9 + k))
    with api.Context(variants.ls_torque()) as ctx:
        alone = [ctx.run_jobs([j])[0] for j in jobs]  # several lanes per fit
        for waves in (4, 2):
            for j in jobs:
                ctx.set_waves(j["space"].variant, j["curve"].n_filters, waves)
            for a, b in zip(alone, ctx.run_jobs(jobs)):
                assert a["best_f"] == b["best_f"] and a["n_evals"] == b["n_evals"]
                _same(b["best_params"], a["best_params"])
                _same(b["best_dV"], a["best_dV"])


@pytest.mark.parametrize("prec", ["fp64", "f32simplex"])
@pytest.mark.parametrize("name", ["ls", "bc", "bw_torque", "torque2", "bc_rotate", "rect_torque", "nudge", "trend",
                                  "seg3", "seg4_onele_torque_bc"])
def test_more_curves_than_rows_take(name, prec):
    v = BUILDS[name](PRECS[prec])
    base = variants.make_variant(bool(v.torque), bool(v.bc), precision=PRECS[prec]) if v.n_seg > 1 else v
    curve, _ = synth.make_curve(7, base, 61, 1.5, n_filters=2)
    space = variants.default_model_space(v)
    keep = {}
    with api.Context(v) as ctx:
        ctx.set_model_space(space)
        if v.n_seg > 1:
            keep["t_start"] = curve.mjd[0] + 0.2 + 1.3 * np.arange(v.n_seg) / v.n_seg  # grid points before the first
            ctx.set_segments(keep["t_start"])
        ctx.upload_curve(curve)
        if v.nudge:
            keep["minima"] = (curve.mjd[[9, 30]].astype(np.float32), curve.V[[9, 30]])
            ctx.set_minima(*keep["minima"])
        pb = oracle.Problem(space, curve, **keep)
        p = _models(pb, 70)
        n = len(p)
        got = {m: ctx.model_curve(np.resize(p, (m, p.shape[1])), n_plot=37) for m in (4096, 4097, 4400)}
    t, vmod, f, dv = pb.model_curve(p, n_plot=37)
    ok = f < 1e29  # a failed NUDGE model has no delta_V
    for m, g in got.items():
        _same(g[0], t)
        for a in (0, (m // n - 1) * n):
            _same(g[2][a:a + n], f)
            _same(g[1][a:a + n][ok], vmod[ok])
            _same(g[3][a:a + n][ok], dv[ok])
        rest = m - (m // n) * n
        _same(g[2][m - rest:], f[:rest])
        _same(g[1][m - rest:][ok[:rest]], vmod[:rest][ok[:rest]])
