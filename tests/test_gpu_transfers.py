"""Particles to the GPU and back, whole bytes: around the size from which host
threads copy them out in chunks (8 MiB, 95,325.09 particles) and from which the
chunks are larger (16 MiB, 190,650.2), with
ragged last chunks, into pageable and pinned memory, and from several threads."""
import ctypes
import threading

import numpy as np
import pytest

from test_particle_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from test_particle_amd.gpu import Tracker
    t = Tracker(0)
    t.set_field_abc(1.0, 1.0, 1.0)
    yield t
    t.close()


def particles(n, seed):
    return np.random.default_rng(seed).standard_normal((n, 11))


@pytest.mark.parametrize("n", [1, 95325, 95326, 107240, 190650, 190651, 700001])
@pytest.mark.parametrize("pinned", [False, True])
def test_round_trip(gpu, n, pinned):
    from hipmem import hip
    from test_particle_amd.gpu import lib
    p = particles(n, 91)
    mem = ctypes.c_void_p()
    if pinned:
        hip().hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t,
                                        ctypes.c_uint]
        hip().hipHostFree.argtypes = [ctypes.c_void_p]
        assert hip().hipHostMalloc(ctypes.byref(mem), p.nbytes, 0) == 0
        out = np.ctypeslib.as_array(ctypes.cast(mem, ctypes.POINTER(ctypes.c_double)), p.shape)
    else:
        out = np.empty(p.shape)
    gpu.load(p)
    for _ in range(2):                  # the slots are used again
        out[:] = -1.0
        assert lib().tp_gpu_store_particles(gpu._ctx, abi.dptr(out), None) == 0
        assert np.array_equal(out, p)
    if pinned:
        assert hip().hipHostFree(mem) == 0
    got, nsteps = gpu.store()
    assert np.array_equal(got, p)
    assert (nsteps == 1).all()


def test_start_given_or_not(gpu):
    """Without ptl_init the start is the particles themselves, with it the D
    sums are taken against that; the caller's arrays stay as they were."""
    p = particles(300, 92)
    p0 = p.copy()
    prm = abi.make_params(dt=0.01, estep=40, lo=(-9,) * 3, hi=(9,) * 3, dcoeff_interval=20,
                          pusher=abi.TP_PUSH_BORIS, nt_out=1, emin=1e-3, emax=10.0)
    a = gpu.track_fixed(prm, p)
    b = gpu.track_fixed(prm, p, p.copy())
    q = p + 0.5
    c = gpu.track_fixed(prm, p, q)
    assert np.array_equal(p, p0)
    for k in a:
        assert np.array_equal(a[k], b[k]), k
    assert np.array_equal(a["ptl"], c["ptl"])
    assert not np.array_equal(a["dcoeff"], c["dcoeff"])


def test_two_contexts_two_threads():
    from test_particle_amd.gpu import Tracker
    bad = []

    def run(seed):
        t = Tracker(0)
        t.set_field_abc(1.0, 1.0, 1.0)
        p = particles(150000 + seed, seed)
        for _ in range(3):
            t.load(p)
            if not np.array_equal(t.store()[0], p):
                bad.append(seed)
        t.close()

    th = [threading.Thread(target=run, args=(s,)) for s in (93, 94)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not bad
