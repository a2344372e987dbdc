"""The adaptive kernels' mode sum on the matrix cores (groups of 16 points,
four modes at a time) at the edges of its groups and tables: bit for bit the
oracle's sum, whatever share of a wavefront is active."""
import numpy as np
import pytest

from test_particle_amd import abi
from test_particle_amd.fields import mode_table
from test_particle_amd.particles import init_particles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from test_particle_amd.gpu import Tracker
    t = Tracker(0)
    yield t
    t.close()


def _ptl(n):
    return init_particles(n, (0, 0, 0), (10, 10, 10), 0.1, seed=61, kind="loguniform", vmax=0.9)


# 1008 modes are the last that fit the copy in LDS; 1009 are read from memory
@pytest.mark.parametrize("modes", [1, 3, 16, 17, 63, 1008, 1009])
def test_tables(gpu, oracle_tp, modes):
    rows = mode_table(modes, kmin=0.3, kmax=30.0, rms=0.5, seed=62)
    prm = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=0.2, b_ref=1.0)
    gpu.set_field_modes(rows, 1.0)
    p = _ptl(40)
    r = gpu.track_adaptive(prm, p)
    ref = oracle_tp.bs_track(oracle_tp.Field.modes(rows, 1.0), prm, p)
    assert np.array_equal(r["ptl"], ref["ptl"]) and np.array_equal(r["nsteps"], ref["nsteps"])


# one to four groups of 16 points, with ragged last groups
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 49, 64, 65])
@pytest.mark.parametrize("block,wpc", [(64, 1), (256, 4)])
def test_groups(gpu, oracle_tp, n, block, wpc):
    rows = mode_table(30, kmin=0.3, kmax=30.0, rms=0.5, seed=63)
    prm = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=0.5, b_ref=1.0, block=block,
                             waves_per_cu=wpc)
    gpu.set_field_modes(rows, 1.0)
    p = _ptl(n)
    r = gpu.track_adaptive(prm, p)
    ref = oracle_tp.bs_track(oracle_tp.Field.modes(rows, 1.0), prm, p)
    assert np.array_equal(r["ptl"], ref["ptl"]) and np.array_equal(r["nsteps"], ref["nsteps"])


# 16, 32 and 64 particles to a wavefront (256 compute units, four wavefronts
# each), more particles than lanes in the last
@pytest.mark.parametrize("n", [16384, 16385, 32768, 32769, 70001])
@pytest.mark.parametrize("dense", [False, True])
def test_lanes_per_wavefront(gpu, oracle_tp, n, dense):
    rows = mode_table(20, kmin=0.3, kmax=10.0, rms=0.5, seed=64)
    f = oracle_tp.Field.modes(rows, 1.0)
    gpu.set_field_modes(rows, 1.0)
    p = _ptl(n)
    pick = np.random.default_rng(65).choice(n, 200, replace=False)
    if dense:
        bs = abi.make_bs_params(rtol=1e-8, atol=1e-10)
        prm = abi.make_params(dt=0.05, estep=20, lo=(0, 0, 0), hi=(10, 10, 10), nbins=52,
                              nt_out=2, einterval_t=10, dcoeff_interval=10, emin=1e-4, emax=10.0)
        r = gpu.track_adaptive_diag(bs, prm, p)
        ref = oracle_tp.bs_track_diag(f, bs, prm, p[pick])
        assert r["espect"].sum() == 2 * n
    else:
        bs = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=0.05, b_ref=1.0)
        r = gpu.track_adaptive(bs, p)
        ref = oracle_tp.bs_track(f, bs, p[pick])
    assert np.array_equal(r["ptl"][pick], ref["ptl"])
    assert np.array_equal(r["nsteps"][pick], ref["nsteps"])


def test_far_phases(gpu, oracle_tp):
    """Phases beyond the range in which the sum that rounds them keeps their
    parity (7e15): the probe, and both adaptive forms' sum with near and far
    points in one wavefront, bit for bit the oracle's."""
    rows = mode_table(40, kmin=0.3, kmax=30.0, rms=0.5, seed=66)
    f = oracle_tp.Field.modes(rows, 1.0)
    gpu.set_field_modes(rows, 1.0)
    rng = np.random.default_rng(67)
    pts = np.exp(rng.uniform(np.log(1e12), np.log(1e16), (500, 4))) * rng.choice([-1, 1], (500, 4))
    pts[7] = [np.nan, 0, 0, 0]
    pts[8] = [0, np.inf, 0, 0]
    b = gpu.eval_field(pts)
    assert np.array_equal(b, oracle_tp.eval_field(f, pts), equal_nan=True)
    assert np.isnan(b[7:9, :3]).all() and np.isfinite(b[9:]).all()
    p = _ptl(100)
    p[::3, 0] = 2.0 ** 49 + 1000.0 * np.arange(34)      # phases of up to 1.4e16
    p[1::3, 1] = -2.0 ** 49
    bs = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=0.2, b_ref=1.0)
    r = gpu.track_adaptive(bs, p)
    ref = oracle_tp.bs_track(f, bs, p)
    assert np.array_equal(r["ptl"], ref["ptl"]) and np.array_equal(r["nsteps"], ref["nsteps"])
    rows[5, 6] = 1e16                                    # a phase that is far by itself
    f = oracle_tp.Field.modes(rows, 1.0)
    gpu.set_field_modes(rows, 1.0)
    p = _ptl(100)
    bs = abi.make_bs_params(rtol=1e-8, atol=1e-10)
    prm = abi.make_params(dt=0.05, estep=20, lo=(0, 0, 0), hi=(10, 10, 10), nbins=52, nt_out=2,
                          einterval_t=10, dcoeff_interval=10, emin=1e-4, emax=10.0)
    r = gpu.track_adaptive_diag(bs, prm, p)
    ref = oracle_tp.bs_track_diag(f, bs, prm, p)
    for k in ("ptl", "nsteps", "espect"):
        assert np.array_equal(r[k], ref[k]), k


def test_empty_table(oracle_tp):
    """No modes at all: the uniform guide field, through both forms and the
    launch-shape trials."""
    from test_particle_amd.gpu import Tracker
    rows = np.zeros((0, 7))
    f = oracle_tp.Field.modes(rows, 0.8)
    p = _ptl(70)
    with Tracker(0) as t:
        t.set_field_modes(rows, 0.8)
        bs = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=0.5, b_ref=0.8)
        r = t.track_adaptive(bs, p)
        ref = oracle_tp.bs_track(f, bs, p)
        assert np.array_equal(r["ptl"], ref["ptl"]) and np.array_equal(r["nsteps"], ref["nsteps"])
        t.tune_adaptive(bs)
        r = t.track_adaptive(bs, p)
        assert np.array_equal(r["ptl"], ref["ptl"]) and np.array_equal(r["nsteps"], ref["nsteps"])
        bs = abi.make_bs_params(rtol=1e-8, atol=1e-10)
        prm = abi.make_params(dt=0.05, estep=20, lo=(0, 0, 0), hi=(10, 10, 10), nbins=52,
                              nt_out=2, einterval_t=10, dcoeff_interval=10, emin=1e-4, emax=10.0)
        r = t.track_adaptive_diag(bs, prm, p)
        ref = oracle_tp.bs_track_diag(f, bs, prm, p)
        for k in ("ptl", "nsteps", "espect"):
            assert np.array_equal(r[k], ref[k]), k
