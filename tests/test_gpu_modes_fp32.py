"""The FP32 mode sum of a wavefront on the matrix cores against 64 bits: one
Boris step in a field of B alone turns u by an angle of |B| h, so the momentum
after a step gives the field the step used.  Table and wavefront edges, and
both sides of the rule that chooses it (80 modes)."""
import numpy as np
import pytest

from test_particle_amd import abi
from test_particle_amd.fields import eval_modes_numpy, mode_table
from test_particle_amd.particles import init_particles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from test_particle_amd.gpu import Tracker
    t = Tracker(0)
    yield t
    t.close()


@pytest.mark.parametrize("modes", [79, 80, 81, 96, 97, 1000])
@pytest.mark.parametrize("n", [1, 63, 64, 257])
def test_one_step(gpu, modes, n):
    rows = mode_table(modes, kmin=0.05, kmax=50.0, rms=0.5, seed=71)
    p = init_particles(n, (0, 0, 0), (100, 100, 100), 0.5, seed=72)
    dt = 0.2
    prm = abi.make_params(dt=dt, estep=1, lo=(0, 0, 0), hi=(100, 100, 100),
                          pusher=abi.TP_PUSH_BORIS, precision=abi.TP_FP32_MIXED,
                          bc_flag=abi.TP_BC_NONE)
    gpu.set_field_modes(rows, 1.0)
    r = gpu.track_fixed(prm, p)["ptl"]
    b = eval_modes_numpy(rows, p[:, :3], 1.0)
    u = p[:, 4:7]
    g = np.sqrt(1 + (u * u).sum(1, keepdims=True))
    t = 0.5 * dt / g * b
    s = 2 * t / (1 + (t * t).sum(1, keepdims=True))
    un = u + np.cross(u + np.cross(u, t), s)
    # momentum rounding: 2^-24 in each of some 10 operations; field: float
    # positions up to 100 (ulp 2^-17) shift the phases of kmax = 50 by up to
    # 50 * 3 * 2^-18 = 6e-4, times the amplitude of those modes (k^-5/3: below
    # 1e-3 of rms) -- 1e-6 of |B| in all, times |u| dt / g
    assert np.abs(r[:, 4:7] - un).max() < 3e-6
    x = p[:, :3] + un * dt / np.sqrt(1 + (un * un).sum(1, keepdims=True))
    assert np.abs(r[:, :3] - x).max() < 3e-6


def test_open_boundary_and_short_wavefronts(gpu):
    """Particles that leave stop; those that stay do not depend on which others
    share their wavefront."""
    rows = mode_table(100, kmin=0.1, kmax=10.0, rms=0.5, seed=73)
    lo, hi = (0, 0, 0), (4, 4, 4)
    p = init_particles(300, lo, hi, 0.6, seed=74)
    prm = abi.make_params(dt=0.1, estep=200, lo=lo, hi=hi, pusher=abi.TP_PUSH_BORIS,
                          precision=abi.TP_FP32_MIXED, bc_flag=abi.TP_BC_OPEN, nt_out=2,
                          emin=1e-4, emax=10.0)
    gpu.set_field_modes(rows, 1.0)
    r = gpu.track_fixed(prm, p)
    out = r["nsteps"] < 201
    # nsteps counts from 1: a particle that leaves at step j has j + 1
    assert out.any() and r["remain"][-1] == 300 - (r["nsteps"] <= 101).sum()
    perm = np.random.default_rng(75).permutation(300)[:77]
    q = gpu.track_fixed(prm, p[perm])
    assert np.array_equal(q["ptl"], r["ptl"][perm])
    assert np.array_equal(q["nsteps"], r["nsteps"][perm])


@pytest.mark.parametrize("bins", [14336, 14337, 16000])
def test_large_histograms(gpu, bins):
    """Histograms that leave no LDS for the wavefront sum take the other kernel:
    the same field to FP32 rounding, every particle counted."""
    rows = mode_table(96, kmin=0.1, kmax=10.0, rms=0.5, seed=76)
    p = init_particles(65, (0, 0, 0), (4, 4, 4), 0.6, seed=77)
    kw = dict(dt=0.1, estep=10, lo=(0, 0, 0), hi=(4, 4, 4), pusher=abi.TP_PUSH_BORIS,
              precision=abi.TP_FP32_MIXED, bc_flag=abi.TP_BC_NONE, nt_out=1, einterval_t=10,
              emin=1e-4, emax=10.0)
    gpu.set_field_modes(rows, 1.0)
    a = gpu.track_fixed(abi.make_params(nbins=40, **kw), p)
    b = gpu.track_fixed(abi.make_params(nbins=bins, **kw), p)
    assert a["espect"].sum() == b["espect"].sum()
    # ten steps of rounding in field and momentum (see above)
    assert np.abs(a["ptl"] - b["ptl"]).max() < 3e-5


@pytest.mark.parametrize("modes", [1, 79, 80, 1000])
def test_probe_is_the_steps_field(gpu, modes):
    """eval_field in FP32 returns the step's field, bit for bit.  With |u| =
    2^-13 (gamma rounds to 1) along one axis and qm dt / 2 = 2^-30, a step
    turns the momentum by 2 t x u with t = 2^-30 B, all exact scalings by
    powers of two: the terms left out are 2^-30 |B|^2 / B_c of what is kept,
    below half a unit in the last place for |B_c| > |B|^2 / 32."""
    rows = mode_table(modes, kmin=0.05, kmax=50.0, rms=0.5, seed=78)
    n, w, hf = 333, 2.0 ** -13, 2.0 ** -30
    p = init_particles(n, (0, 0, 0), (1000, 1000, 1000), 0.5, seed=79)
    gpu.set_field_modes(rows, 1.0)
    b = gpu.eval_field(np.c_[p[:, :3], np.zeros(n)], abi.TP_FP32_MIXED)[:, :3]
    prm = abi.make_params(dt=2 * hf, estep=1, lo=(0, 0, 0), hi=(1000, 1000, 1000), qm=1.0,
                          pusher=abi.TP_PUSH_BORIS, precision=abi.TP_FP32_MIXED,
                          bc_flag=abi.TP_BC_NONE)
    size = np.sqrt((b * b).sum(1))
    for c in range(3):
        a = (c + 1) % 3                      # u along a: component d gets 2 w hf B_c, up to sign
        d = 3 - a - c
        p[:, 4:7] = 0.0
        p[:, 4 + a] = w
        u = gpu.track_fixed(prm, p)["ptl"][:, 4:7]
        ok = np.abs(b[:, c]) > size ** 2 / 32
        assert ok.sum() > n // 2
        sign = 1.0 if (a, c, d) in ((0, 1, 2), (1, 2, 0), (2, 0, 1)) else -1.0
        assert np.array_equal(u[ok, d], sign * 2 * w * hf * b[ok, c]), c


@pytest.mark.parametrize("modes,box,rms", [(100, 130, 3.9e-7), (300, 130, 3.9e-7),
                                           (1000, 130, 3.9e-7), (1000, 1000, 1.9e-6)])
def test_field_error(gpu, modes, box, rms):
    """The step's field (the probe returns its bits) against 64 bits at points
    that are floats, where nothing but the sum errs.

    rms: phases of up to kmax box / 2 pi = 1000 revolutions (8000) rounded at
    2^-14 (2^-11), 1.9e-4 rad (1.5e-3) for the largest k, which hold 1e-3 of the
    field's square; amplitude, cosine and sum, 2^-24 each and growing with the
    partial sums.  Measured 2.3e-7 to 3.0e-7 (1.5e-6); FP32 FMAs a point to a
    lane 4.0e-7 to 8.4e-7 (2.1e-6), twice the error.

    Along the field: errors of either sign average out, but for the rounding of
    the few largest amplitudes, up to 1.5e-8 a table and 5e-9 over eight of them;
    the hardware cosine's own gain error of 3.2e-8 would show."""
    gain = []
    for seed in range(81, 89):
        rows = mode_table(modes, kmin=0.05, kmax=48.0, rms=0.5, seed=seed)
        x = np.random.default_rng(seed).uniform(0, box, (20000, 3))
        pts = np.c_[x.astype(np.float32).astype(np.float64), np.zeros(len(x))]
        gpu.set_field_modes(rows, 0.0)
        b = gpu.eval_field(pts, abi.TP_FP32_MIXED)[:, :3]
        e = gpu.eval_field(pts, abi.TP_FP64)[:, :3]      # the oracle's to 1e-14
        n2 = (e * e).sum(1).mean()
        assert np.sqrt(((b - e) ** 2).sum(1).mean() / n2) < rms
        gain.append(((b - e) * e).sum(1).mean() / n2)
    assert abs(np.mean(gain)) < 1.5e-8
