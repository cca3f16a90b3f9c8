"""Runs of several stages whose launches hold more evaluation rounds than a
stage needs: with several lanes per model a stage ends between launches, so
the run takes one launch per stage at least.  Each equals the oracle's run bit
for bit, alone and as a job of a batch."""
import numpy as np
import pytest

import oracle
from asteroid_amd import abi, api, synth, variants

pytestmark = pytest.mark.gpu


def _problem(make, n_obs=50):
    v = make(abi.PREC_FP64)
    curve, _ = synth.make_curve(5, v, n_obs, 1.0)
    return v, curve, variants.default_model_space(v)


def _ls(p):
    return variants.make_variant(False, precision=p)


@pytest.mark.parametrize("make", [variants.ls_torque, _ls], ids=["torque", "ls"])
@pytest.mark.parametrize("groups,group_size", [(1, 64), (17, 256), (65, 256)])  # 16 lanes, 4 lanes, one
def test_more_stages_than_launches_of_evaluations(make, groups, group_size):
    v, curve, space = _problem(make)
    run = dict(nstages=12, n_steps=3)
    with api.Context(v) as ctx:
        ctx.set_model_space(space)
        ctx.upload_curve(curve)
        ctx.rng_seed(6)
        ctx.run(groups, group_size, ticks_per_launch=4096, **run)
        got = ctx.fetch() + ctx.fetch_lanes()
    want = oracle.Problem(space, curve).run(groups, group_size, seed=6, form=oracle.CANON, n_threads=8, **run)
    for g, k in zip(got, ("f", "params", "dV", "lane_f", "lane_nev", "lane_steps")):
        np.testing.assert_array_equal(g, want[k])


@pytest.mark.parametrize("schedule", [0, 1])
def test_batch_of_more_stages_than_launches(schedule):
    probs = [_problem(_ls), _problem(variants.ls_torque)]
    run = dict(nstages=12, n_steps=2)
    jobs = [dict(space=space, curve=curve, n_fits=512, seed=3 + k, **run) for k, (_, curve, space) in enumerate(probs)]
    with api.Context(probs[0][0]) as ctx:
        res = ctx.run_jobs(jobs, schedule=schedule)
    for j, r in zip(jobs, res):
        want = oracle.Problem(j["space"], j["curve"]).run(2, 256, seed=j["seed"], n_threads=8, **run)
        g = int(np.argmin(want["f"]))
        assert r["status"] == 0 and r["best_f"] == want["f"][g] and r["n_evals"] == want["lane_nev"].sum()
        np.testing.assert_array_equal(r["best_params"], want["params"][g])
