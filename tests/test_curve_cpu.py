"""Curve.obs_array: the observations as the C ABI takes them, one of each of
the curve's times; longer columns are cut to the times, shorter ones refused."""
import numpy as np
import pytest

from asteroid_amd import abi, synth, variants


def _curve(n=9):
    return synth.make_curve(3, variants.ls_torque(abi.PREC_FP64), n, 1.0, n_filters=2)[0]


def _values(obs):
    return [(o.mjd, o.V, o.w, o.filter, list(o.E), list(o.S)) for o in obs]


def test_columns_in_their_places():
    c = _curve()
    for k, o in enumerate(c.obs_array()):
        assert (o.mjd, o.V, o.w, o.filter) == (c.mjd[k], c.V[k], c.w[k], c.filter[k])
        assert list(o.E) == list(c.E[k]) and list(o.S) == list(c.S[k])
    assert len(synth.Curve([], [], [], [], 1, np.zeros((0, 3)), np.zeros((0, 3))).obs_array()) == 0


def test_longer_columns_are_cut():
    c = _curve()
    want = _values(c.obs_array())[:5]
    c.mjd = c.mjd[:5]
    assert c.n_data == 5 and _values(c.obs_array()) == want
    c.E = np.hstack([c.E, c.E])
    c.V = list(c.V)
    assert _values(c.obs_array()) == want


@pytest.mark.parametrize("name", ["V", "w", "filter", "E", "S"])
@pytest.mark.parametrize("n", [0, 1, 8])
def test_shorter_columns_are_refused(name, n):
    c = _curve()
    setattr(c, name, getattr(c, name)[:n])
    with pytest.raises(IndexError):
        c.obs_array()
