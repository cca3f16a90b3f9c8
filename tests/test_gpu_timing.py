"""ast_last_timing of the calls that launch more than one kernel: every launch
is reported, and the kernels' time is no more than the call's."""
import time

import numpy as np
import pytest

from asteroid_amd import abi, api, synth, variants

pytestmark = pytest.mark.gpu


def test_launches_and_kernel_time_of_every_route():
    v = variants.ls_torque(abi.PREC_FP64)
    curve, truth = synth.make_curve(7, v, 40, 1.0)
    with api.Context(v) as ctx:
        ctx.set_model_space(variants.default_model_space(v))
        ctx.upload_curve(curve)

        def timed(call):
            t0 = time.perf_counter()
            out = call()
            wall = (time.perf_counter() - t0) * 1e3
            ms, launches = ctx.last_timing()
            print(f"{launches} launches, {ms:.3f} of {wall:.3f} ms")
            assert 0 < ms < wall
            return out, launches

        models = np.repeat(truth[None], 70000, axis=0)
        for n, want in ((1, 1), (20000, 1), (65536, 1), (65537, 2)):
            assert timed(lambda: ctx.chi2_batch(models[:n]))[1] == want
        for n, want in ((1, 2), (4096, 2), (4097, 1)):  # observations and grid, or both in one
            out, launches = timed(lambda: ctx.model_curve(models[:n], n_plot=300))
            assert launches == want
        t = np.linspace(0.0, 5.0, 2000)
        assert timed(lambda: ctx.periodogram(t, np.sin(40 * t)))[1] == 2  # pairs and their sum
        ctx.periodogram(t, t)  # no minima
        assert ctx.last_timing()[1] == 0
