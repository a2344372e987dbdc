"""The order of the training kernels' sums, which fixes the gradient's bits:
the network's outputs are the evaluation's; the sums over samples run in
chunks of 256 samples, one sample after another within a chunk for the biases,
and one chunk after another.  Adam normalises the gradient and the bfloat16
weights round, so a change of this order shows up in a trained network by
orders of magnitude more than in the gradient.

All comparisons are bit for bit.  The gradient of n samples holds the factor
2/(3n), rounded once; for n a power of two times another number of samples the
factors, and with them every term and partial sum, differ by exactly that
power (no term is near the smallest float)."""
import numpy as np
import pytest

from test_particle_amd import abi, surrogate

pytestmark = pytest.mark.gpu

CHUNK = 256


@pytest.fixture(scope="module")
def gpu():
    from test_particle_amd.gpu import Tracker
    t = Tracker(0)
    t.mlp_set(surrogate.fourier_frequencies(10.0, seed=3), surrogate.init_params(seed=4), 0.7)
    yield t
    t.close()


def _data(n, seed=0):
    rng = np.random.default_rng(1000 * seed + n)
    return (rng.uniform(0.0, 10.0, (n, 3)).astype(np.float32),
            rng.normal(0.0, 1.0, (n, 3)).astype(np.float32))


def _slices():
    out, o = [], 0
    for fin, fout in surrogate.LAYERS:
        out += [slice(o, o + fin * fout), slice(o + fin * fout, o + fin * fout + fout)]
        o += fin * fout + fout
    assert o == abi.TP_MLP_NPARAMS
    return out


def _in_order(terms):
    s = np.zeros_like(terms[0])
    for t in terms:
        s = s + t
    return s


@pytest.mark.parametrize("n", [1, 64, 200, 256])
def test_outputs_are_the_evaluations(gpu, n):
    """The output bias's gradient is the sum of dL/dout = 2 (o - y) / 3n, in
    sample order, with the evaluation's outputs o; the loss the sum of the
    squared differences in double."""
    x, y = _data(n)
    loss, g = gpu.mlp_loss_grad(x, y)
    o = gpu.mlp_forward(x.astype(np.float64))
    e = o.astype(np.float32) - y
    assert np.array_equal(o.astype(np.float32).astype(np.float64), o)
    d = np.float32(2.0) * e * np.float32(1.0 / (3.0 * n))
    assert np.array_equal(g[-3:], _in_order(list(d)))
    # any order of n <= 256 double sums: 256 roundings of 2^-53
    want = np.sum(e.astype(np.float64) ** 2) / (3.0 * n)
    assert abs(loss - want) <= 256 * 2.0 ** -53 * want


def test_biases_within_a_chunk(gpu):
    x, y = _data(CHUNK)
    _, g = gpu.mlp_loss_grad(x, y)
    one = [gpu.mlp_loss_grad(x[s:s + 1], y[s:s + 1])[1] for s in range(CHUNK)]
    f = np.float32(1.0 / CHUNK)
    for k in (1, 3, 5, 7):
        sl = _slices()[k]
        assert np.array_equal(g[sl], _in_order([f * t[sl] for t in one])), k


@pytest.mark.parametrize("n", [512, 1024, 16384, 32768])
def test_chunks_in_order(gpu, n):
    x, y = _data(n)
    loss, g = gpu.mlp_loss_grad(x, y)
    parts = [gpu.mlp_loss_grad(x[a:a + CHUNK], y[a:a + CHUNK]) for a in range(0, n, CHUNK)]
    f = np.float32(CHUNK / n)
    want = _in_order([f * p[1] for p in parts])
    for k, sl in enumerate(_slices()):
        assert np.array_equal(g[sl], want[sl]), k
    # the chunks' sums of squares: 3 CHUNK loss, exact up to two roundings each
    lw = sum(3.0 * CHUNK * p[0] for p in parts) / (3.0 * n)
    assert abs(loss - lw) <= (n // CHUNK + 4) * 2.0 ** -53 * lw
