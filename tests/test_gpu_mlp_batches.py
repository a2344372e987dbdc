"""Loss and gradient of the surrogate at the edges of the training kernels'
tiles (64 samples) and of rows and gradient chunks (256), against the oracle
with the GPU's rounding points;
the sum over samples must not depend on how they are cut."""
import numpy as np
import pytest

from test_particle_amd import abi, surrogate

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from test_particle_amd.gpu import Tracker
    t = Tracker(0)
    yield t
    t.close()


def _set(gpu):
    period = 10.0
    q = surrogate.fourier_frequencies(period, seed=3)
    p = surrogate.init_params(seed=4)
    gpu.mlp_set(q, p, 0.7)
    return q, p, period


def _data(n, period):
    rng = np.random.default_rng(n)
    return (rng.uniform(0.0, period, (n, 3)).astype(np.float32),
            rng.normal(0.0, 1.0, (n, 3)).astype(np.float32))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257])
def test_tiles(gpu, n):
    from oracle import tpref
    q, p, period = _set(gpu)
    x, y = _data(n, period)
    loss, g = gpu.mlp_loss_grad(x, y)
    lref, gref = tpref.mlp_loss_grad(p.astype(np.float64), q.astype(np.float64),
                                     x.astype(np.float64), y.astype(np.float64), emulate=True)
    assert abs(loss - lref) < 1e-3 * lref
    o = 0
    for fin, fout in surrogate.LAYERS:
        for size in (fin * fout, fout):
            a, b = g[o:o + size].astype(np.float64), gref[o:o + size]
            # 1 % of the block's norm, as for 300 samples (bf16 flips); a
            # single sample's flips do not average out: 2^-8 a flip, some of
            # 128 units in three layers
            assert np.linalg.norm(a - b) < (1e-2 if n > 1 else 3e-2) * np.linalg.norm(b), (o, n)
            o += size
    assert o == abi.TP_MLP_NPARAMS


@pytest.mark.parametrize("n", [8192, 8193, 16384, 16700])
def test_chunks(gpu, n):
    """The gradient of the whole set is the sample-weighted mean of its
    parts', which are one chunk each: FP32 sums of n terms in another order,
    at most sqrt(n) roundings of 2^-24 of the largest partial sum -- 1e-5 of
    the norm -- and dL/dout rounded to bf16 after another scale factor 2/(3n),
    a power of two apart only for the first part: 2^-9 a term, averaged."""
    _, _, period = _set(gpu)
    x, y = _data(n, period)
    loss, g = gpu.mlp_loss_grad(x, y)
    want, lw = 0.0, 0.0
    for a in range(0, n, 256):
        m = min(256, n - a)
        lp, gp = gpu.mlp_loss_grad(x[a:a + m], y[a:a + m])
        want = want + gp.astype(np.float64) * (m / n)
        lw += lp * m / n
    assert abs(loss - lw) < 1e-6 * lw
    assert np.linalg.norm(g - want) < 2.0 ** -9 * np.linalg.norm(want)
