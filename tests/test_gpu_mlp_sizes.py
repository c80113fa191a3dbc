"""The predictor network's kernels at the edges of their sizes (fribo_mlp.hip:
8 samples per workgroup, at most 128 gradient parts, sets of up to 16384
floats predicted through pinned memory) against the FP64 oracle.

Bars: a gradient component is a sum over the samples and, backwards, over at
most 64 + 16 terms per layer in FP32; with all terms of one sign its relative
error is at most (n/8 + 8 + 3 * 64 + ni) * 2^-24, taken of the largest
component.  An output of the BF16 inference moves by at most 2^-8 |W3| for
every hidden activation that rounds the other way."""
import numpy as np
import pytest

import mlp_oracle as M

pytestmark = pytest.mark.gpu


def _net(ni, no, seed):
    from fribois2d_amd.gpu import Mlp
    net = Mlp(ni, no, seed=seed)
    return net, net.params()


@pytest.mark.parametrize("ni,no,n", [(1, 1, 1), (2, 16, 7), (45, 3, 8), (45, 3, 9), (64, 1, 63), (255, 16, 65),
                                     (256, 5, 130), (9, 2, 1031)])
def test_gradient_sizes(ni, no, n):
    net, p = _net(ni, no, 5)
    rng = np.random.default_rng([ni, no, n])
    X = (rng.standard_normal((n, ni)) / np.sqrt(ni)).astype(np.float32)
    T = rng.standard_normal((n, no)).astype(np.float32)
    g, loss = net.grad(X, T)
    gr = M.grad(p.astype(np.float64), X, T)
    bar = (n / 8 + 8 + 3 * 64 + ni) * 2.0 ** -24
    assert np.abs(g - gr).max() <= bar * np.abs(gr).max()
    assert abs(loss - M.loss(p.astype(np.float64), X, T)) <= bar * loss
    assert np.array_equal(net.params(), p)     # no update
    net.close()


def test_training_with_a_short_last_minibatch():
    """Three epochs over 100 samples in minibatches of 64 and 36 against the
    same Adam steps of the oracle (the bar of five steps on one minibatch)."""
    net, p = _net(12, 2, 6)
    rng = np.random.default_rng(8)
    X = rng.standard_normal((100, 12)).astype(np.float32)
    T = rng.standard_normal((100, 2)).astype(np.float32)
    loss = net.train(X, T, 3, 64, 1e-3)
    q = p.astype(np.float64)
    m, v, t = np.zeros_like(q), np.zeros_like(q), 0
    for _ in range(3):
        for a, b in ((0, 64), (64, 100)):
            t += 1
            last = M.loss(q, X[a:b], T[a:b])
            q, m, v = M.adam(q, M.grad(q, X[a:b], T[a:b]), m, v, t, 1e-3)
    assert np.abs(net.params() - q).max() <= 1e-4
    assert abs(loss - last) <= 1e-4 * last
    net.close()


# 16384 / (9 + 2) = 1489 samples are the most that go through pinned memory
@pytest.mark.parametrize("ni,no,n", [(1, 1, 1), (45, 3, 1), (45, 3, 8), (256, 16, 9), (9, 2, 1489), (9, 2, 1490)])
def test_inference_sizes(ni, no, n):
    net, p = _net(ni, no, 7)
    rng = np.random.default_rng([n, ni])
    X = (rng.standard_normal((n, ni)) / np.sqrt(ni)).astype(np.float32)
    Y = net.predict(X)
    w3 = p[-(no * 64 + no):-no].reshape(no, 64)
    assert (np.abs(Y - M.forward_bf16(p, X, no)) <= 2.0 ** -8 * np.abs(w3).sum(axis=1)).all()
    assert np.array_equal(Y, net.predict(X))
    net.close()
