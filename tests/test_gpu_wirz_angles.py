"""The Wirz pusher's rotation by any angle a step: below 0.75 its sine and cosine
take no argument reduction.  Half angles (the predictor) and whole ones on both
sides of that line, bit for bit the oracle's."""
import numpy as np
import pytest

from test_particle_amd import abi
from test_particle_amd.particles import init_particles

pytestmark = pytest.mark.gpu


# uniform field of 1: the angle is dt / gamma, gamma in 1 .. 1.4; ABC: B from
# near 0 to 1.7, the lanes of a wavefront on both sides
@pytest.mark.parametrize("field", ["test", "abc"])
@pytest.mark.parametrize("dt", [0.01, 0.75, 0.9, 1.6, 2.2, 7.0, 1e3])
def test_angles(oracle_tp, field, dt):
    from test_particle_amd.gpu import Tracker
    hi = (2 * np.pi,) * 3
    n = 17000                             # beyond the four-lane form in the ABC field
    p = init_particles(n, (0, 0, 0), hi, 0.5, seed=91, kind="loguniform", vmax=0.7)
    prm = abi.make_params(dt=dt, estep=4, lo=(0, 0, 0), hi=hi, pusher=abi.TP_PUSH_WIRZ,
                          dcoeff_interval=4)
    with Tracker(0) as t:
        if field == "test":
            t.set_field_test()
            f = oracle_tp.Field.test()
        else:
            t.set_field_abc(1.0, 1.0, 1.0)
            f = oracle_tp.Field.abc(1.0, 1.0, 1.0)
        r = t.track_fixed(prm, p)["ptl"]
    pick = np.random.default_rng(92).choice(n, 2000, replace=False)
    ref = oracle_tp.track_fixed(f, prm, p[pick])["ptl"]
    assert np.array_equal(r[pick], ref, equal_nan=True)
