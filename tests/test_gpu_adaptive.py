"""GPU adaptive Bulirsch-Stoer (persistent work-queue kernel) against the
oracle's sequential implementation of the same algorithm: trajectories,
per-particle accepted steps and the accepted/rejected/RHS totals are
identical (bit for bit), with and without the captured graph."""
import os

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


def _same(a, b, what):
    a = np.asarray(a)
    b = np.asarray(b)
    diff = ~((a == b) | (np.isnan(a) & np.isnan(b)))
    assert not diff.any(), f"{what}: {diff.sum()} differ, first {np.argwhere(diff)[0]}"


def _compare(r, ref, what):
    _same(r["ptl"], ref["ptl"], what + " particles")
    _same(r["nsteps"], ref["nsteps"], what + " accepted steps")
    for k in ("accepted", "rejected", "rhs", "failed"):
        assert r[k] == ref[k], f"{what} {k}: {r[k]} vs {ref[k]}"


def test_bs_modes_bitwise(gpu, oracle_tp):
    """64 modes over 2 decades, 300 particles with |v| log-uniform in
    [0.1, 0.9]c (uneven step counts), 3 gyroperiods, rtol 1e-8."""
    print("[case] bs modes n=300", flush=True)
    rows = mode_table(64, kmin=0.3, kmax=30.0, rms=0.5, seed=51)
    p = init_particles(300, (0, 0, 0), (10, 10, 10), 0.1, seed=52, kind="loguniform",
                       vmax=0.9)
    prm = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=3.0, b_ref=1.0)
    gpu.set_field_modes(rows, 1.0)
    r = gpu.track_adaptive(prm, p)
    ref = oracle_tp.bs_track(oracle_tp.Field.modes(rows, 1.0), prm, p)
    _compare(r, ref, "modes")
    assert r["nsteps"].min() < r["nsteps"].max()        # uneven work
    assert r["failed"] == 0


def test_bs_uniform_field_and_launch_shapes(gpu, oracle_tp):
    p = init_particles(200, (0, 0, 0), (1, 1, 1), 0.6, seed=53)
    gpu.set_field_test()
    ref = oracle_tp.bs_track(oracle_tp.Field.test(),
                             abi.make_bs_params(rtol=1e-9, atol=1e-12, t_end_gyro=5.0), p)
    for block, wpc, graph in ((64, 1, 1), (128, 4, 0), (256, 2, 1)):
        prm = abi.make_bs_params(rtol=1e-9, atol=1e-12, t_end_gyro=5.0, block=block,
                                 waves_per_cu=wpc, use_graph=graph)
        _compare(gpu.track_adaptive(prm, p), ref, f"uniform {block}/{wpc}/{graph}")


def test_bs_graph_replay_and_attempt_cap(gpu, oracle_tp):
    """The captured graph replayed on reloaded particles gives the same
    result each time; an attempt cap stops particles at their last accepted
    state, as the oracle does."""
    rows = mode_table(32, kmin=0.5, kmax=10.0, rms=0.5, seed=54)
    p = init_particles(128, (0, 0, 0), (5, 5, 5), 0.5, seed=55)
    gpu.set_field_modes(rows, 1.0)
    prm = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=2.0, use_graph=1)
    outs = []
    for _ in range(3):
        gpu.load(p)
        st = gpu.run_adaptive(prm)
        q, ns = gpu.store()
        outs.append((q, ns, st["rhs"]))
    for q, ns, rhs in outs[1:]:
        _same(q, outs[0][0], "replay particles")
        assert rhs == outs[0][2]
    capped = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=2.0, max_attempts=5)
    r = gpu.track_adaptive(capped, p)
    ref = oracle_tp.bs_track(oracle_tp.Field.modes(rows, 1.0), capped, p)
    _compare(r, ref, "capped")
    assert r["failed"] > 0


def test_bs_autotuner_cache(gpu, tmp_path):
    rows = mode_table(16, kmin=0.5, kmax=10.0, rms=0.5, seed=56)
    p = init_particles(2048, (0, 0, 0), (5, 5, 5), 0.5, seed=57)
    gpu.set_field_modes(rows, 1.0)
    gpu.load(p)
    prm = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=1.0)
    cache = str(tmp_path / "tune.txt")
    b, w = gpu.tune_adaptive(prm, cache)
    assert b in (64, 128, 256) and w > 0
    assert os.path.exists(cache) and len(open(cache).read().splitlines()) == 1
    assert gpu.tune_adaptive(prm, cache) == (b, w)          # read back, not re-run
    assert len(open(cache).read().splitlines()) == 1
    # the tuner leaves the resident particles untouched
    q, _ = gpu.store()
    assert np.array_equal(q, p)


def test_bs_autotuner_keys(gpu, tmp_path):
    """A choice counts for the kernels and the ensemble class it was timed for:
    entries without them (older files) and of another class are not taken."""
    rows = mode_table(16, kmin=0.5, kmax=10.0, rms=0.5, seed=56)
    gpu.set_field_modes(rows, 1.0)
    prm = abi.make_bs_params(rtol=1e-8, atol=1e-10, t_end_gyro=1.0)
    cu = gpu.device_info()[1]
    cache = tmp_path / "tune.txt"
    cache.write_text(f"192 1 1e9 fk=5 modes=16 rtol=1e-08 kmax={prm.kmax} cu={cu}\n")
    gpu.load(init_particles(2048, (0, 0, 0), (5, 5, 5), 0.5, seed=57))
    b, _ = gpu.tune_adaptive(prm, str(cache))
    lines = cache.read_text().splitlines()
    assert b != 192 and len(lines) == 2
    gpu.load(init_particles(70000, (0, 0, 0), (5, 5, 5), 0.5, seed=57))
    gpu.tune_adaptive(prm, str(cache))
    lines = cache.read_text().splitlines()
    assert len(lines) == 3 and lines[1].split(None, 3)[3] != lines[2].split(None, 3)[3]
    gpu.tune_adaptive(prm, str(cache))
    assert cache.read_text().splitlines() == lines
