"""Fixed-step runs in the ABC field with four lanes to a particle (up to 16,384
particles) and with one, around the edges of wavefronts and blocks and on both
sides of the rule.  Both do the oracle's operations in its order, so all but the
diffusion sums is compared bit for bit; those are sums of n terms in another
order (1e-12 relative, n u = 2e-12 at worst and its square root in practice;
D_ee and D_mumu can be rounding noise, hence 1e-15 absolute)."""
import numpy as np
import pytest

from test_particle_amd import abi
from test_particle_amd.particles import init_particles

pytestmark = pytest.mark.gpu

LO, HI = (0.0, 0.0, 0.0), (2 * np.pi,) * 3


@pytest.fixture(scope="module")
def gpu():
    from test_particle_amd.gpu import Tracker
    t = Tracker(0)
    yield t
    t.close()


def compare(r, ref):
    for k in ("ptl", "nsteps", "espect", "espect_escape", "remain"):
        assert np.array_equal(r[k], ref[k], equal_nan=k == "ptl"), k
    assert (np.abs(r["dcoeff"] - ref["dcoeff"]) <= 1e-12 * np.abs(ref["dcoeff"]) + 1e-15).all()


def params(pusher, bc, steps, **kw):
    kw = {"nt_out": 3, "nbins": 40, "emin": 1e-3, "emax": 10.0, **kw}
    return abi.make_params(dt=0.05, estep=steps, lo=LO, hi=HI, pusher=pusher, bc_flag=bc,
                           precision=abi.TP_FP64, **kw)


@pytest.mark.parametrize("pusher", [abi.TP_PUSH_WIRZ, abi.TP_PUSH_BORIS])
@pytest.mark.parametrize("bc", [0, 1, abi.TP_BC_NONE])
@pytest.mark.parametrize("n,steps", [(1, 130), (15, 130), (16, 130), (17, 130), (65, 301),
                                     (16384, 60), (16385, 60), (65281, 25)])
def test_against_oracle(gpu, oracle_tp, pusher, bc, n, steps):
    p = init_particles(n, LO, HI, 0.7, seed=81 + n)
    prm = params(pusher, bc, steps, dcoeff_interval=20, einterval_t=10)
    gpu.set_field_abc(1.0, 0.7, -0.4)
    r = gpu.track_fixed(prm, p)
    compare(r, oracle_tp.track_fixed(oracle_tp.Field.abc(1.0, 0.7, -0.4), prm, p, nthreads=1))
    if bc == 1 and n > 1:
        assert (r["nsteps"] < steps + 1).any()      # some left before the end


@pytest.mark.parametrize("pusher", [abi.TP_PUSH_WIRZ, abi.TP_PUSH_BORIS])
def test_unusual_states(gpu, oracle_tp, pusher):
    """At rest, outside the box, far away (both forms of the sine's reduction),
    with infinities and NaN: a lane's neighbours in the quad and the wavefront
    are not touched by it."""
    p = init_particles(40, LO, HI, 0.5, seed=83)
    p[3, 4:7] = 0.0
    p[4, 0] = 1e3
    p[7, 1] = -1e9
    p[9, 2] = 3e15
    p[17, 0] = np.inf
    p[21, 5] = np.nan
    prm = params(pusher, abi.TP_BC_NONE, 50)
    gpu.set_field_abc(1.0, 1.0, 1.0)
    r = gpu.track_fixed(prm, p)
    ref = oracle_tp.track_fixed(oracle_tp.Field.abc(1.0, 1.0, 1.0), prm, p, nthreads=1)
    assert np.array_equal(r["ptl"], ref["ptl"], equal_nan=True)
    assert np.array_equal(r["nsteps"], ref["nsteps"])


@pytest.mark.parametrize("n", [65536, 65537, 70001, 130816, 130817])
def test_block_sizes(gpu, oracle_tp, n):
    """Blocks of 256, 128 and 64 lanes and the lines between them."""
    p = init_particles(n, LO, HI, 0.7, seed=84)
    prm = params(abi.TP_PUSH_BORIS, 0, 10, dcoeff_interval=5)
    gpu.set_field_abc(1.0, 0.7, -0.4)
    r = gpu.track_fixed(prm, p)
    compare(r, oracle_tp.track_fixed(oracle_tp.Field.abc(1.0, 0.7, -0.4), prm, p, nthreads=1))
