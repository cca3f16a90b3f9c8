"""A refused ast_model_curve leaves the caller's arrays as they were."""
import ctypes as C

import numpy as np
import pytest

from asteroid_amd import abi, api, synth, variants

pytestmark = pytest.mark.gpu


def test_refused_model_curve_writes_nothing():
    v = variants.ls_segments(abi.PREC_FP64)
    curve, _ = synth.make_curve(7, variants.make_variant(bool(v.torque), False, precision=abi.PREC_FP64), 60, 1.5)
    space = variants.default_model_space(v)
    with api.Context(v) as ctx:
        ctx.set_model_space(space)
        ctx.set_segments(curve.mjd[0] - 0.01 + 1.5 * np.arange(v.n_seg) / v.n_seg)
        ctx.upload_curve(curve)
        dp = C.POINTER(C.c_double)
        params = np.full((3, space.n_params), 0.5)
        out = [np.full(n, 7.25) for n in (2, 3 * 2, 3, 3 * curve.n_filters)]  # t, vmod, chi2, dV
        eph = curve.ephem3()
        # a grid of two points has none in the middle segment
        rc = ctx.lib.ast_model_curve(ctx.h, params.ctypes.data_as(dp), 3, C.byref(eph), 2,
                                     *[a.ctypes.data_as(dp) for a in out])
        assert rc == -5  # AST_E_DATA
        for a in out:
            assert np.all(a == 7.25)
        assert len(ctx.chi2_batch(params)[0]) == 3  # the context is as before
