"""The network kernels at the edges of their tiles and dispatch: hidden widths
below, at and above one column tile per wavefront (128), widths that leave
half a 32 x 32 gradient block empty, feature rows from one tile to above the
register path's limit, batches below a tile, ragged, over one gradient split
and in 32-row tiles (8,192 rows on), and the epoch chunks of the training's
permutation uploads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# FP32 sums of at most 1,024 products in a random-walk error model: sqrt(1024)
# * 6e-8 = 2e-6 a layer, six layers on the way there and back: 1.2e-5
TOL = 2e-5


@pytest.mark.parametrize("n_freq,hidden,n", [
    (1, 16, 1), (1, 48, 63), (3, 64, 65), (4, 128, 4096), (4, 128, 8193), (22, 112, 300),
    (4, 144, 4100), (24, 272, 200), (2, 512, 8200), (64, 1024, 130)])
def test_network_kernels_at_tile_edges(n_freq, hidden, n):
    import mlp as M
    from mepinterp_amd import capi
    rng = np.random.default_rng(hidden + n)
    k = rng.uniform(-0.5, 0.5, size=(3, n))
    t = rng.normal(size=n).astype(np.float32) + np.float32(3.0)  # errors of order one
    with capi.MLP(n_freq=n_freq, hidden=hidden, seed=3) as net:
        p = net.params.astype(np.float64)
        y, yo = net.predict(k), M.forward(p, k, n_freq, hidden)
        assert np.max(np.abs(y - yo)) < TOL * max(1.0, np.max(np.abs(yo)))
        g, loss = net.grad(k, t)
        go, lo = M.grad(p, k, t, n_freq, hidden), M.loss(p, k, t, n_freq, hidden)
        assert abs(loss - lo) < TOL * lo
        assert np.max(np.abs(g - go)) < TOL * np.max(np.abs(go))
        # a smaller call on the larger buffers, bit for bit as on its own
        if n > 64:
            g2, l2 = net.grad(k[:, :64], t[:64])
            with capi.MLP(n_freq=n_freq, hidden=hidden, seed=3) as own:
                g3, l3 = own.grad(k[:, :64], t[:64])
            np.testing.assert_array_equal(g2, g3)
            assert l2 == l3


@pytest.mark.parametrize("epochs", [1, 2, 3, 7, 8])
def test_training_over_permutation_chunks(epochs):
    """One batch an epoch: the order of the rows does not matter, so the
    weights follow a plain FP64 Adam run.  A step moves a weight by at most
    lr; the FP32 gradients (TOL of the largest) perturb the normalised steps
    of all but the smallest gradients by about that much."""
    import mlp as M
    from mepinterp_amd import capi
    rng = np.random.default_rng(epochs)
    k = rng.uniform(-0.5, 0.5, size=(3, 500))
    t = rng.normal(size=500).astype(np.float32)
    lr = 2e-3
    with capi.MLP(n_freq=3, hidden=64, seed=9) as net:
        p = net.params.astype(np.float64)
        loss = net.train(k, t, epochs=epochs, batch=512, lr=lr, seed=4)
        got = net.params
    m, v = np.zeros_like(p), np.zeros_like(p)
    for s in range(1, epochs + 1):
        lo = M.loss(p, k, t, 3, 64)
        g = M.grad(p, k, t, 3, 64)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1 - 0.9 ** s)) / (np.sqrt(v / (1 - 0.999 ** s)) + 1e-8)
    assert abs(loss - lo) < 1e-4 * lo
    assert np.linalg.norm(got - p) < 1e-3 * lr * np.sqrt(epochs * p.size)


def test_training_chunks_of_a_data_set_after_a_larger_one():
    """The permutation buffers serve any smaller data set: 200 epochs of 700
    points after 140,000 points, equal to the same run on its own."""
    from mepinterp_amd import capi
    rng = np.random.default_rng(12)
    k = rng.uniform(-0.5, 0.5, size=(3, 140000))
    t = rng.normal(size=140000).astype(np.float32)
    out = []
    for first in (True, False):
        with capi.MLP(n_freq=2, hidden=32, seed=2) as net:
            p0 = net.params
            if first:
                net.predict(k)
                net.train(k, t, epochs=1, batch=8192, lr=1e-7, seed=1)
            else:
                net.train(k[:, :700], t[:700], epochs=1, batch=128, lr=1e-7, seed=1)
            net.params = p0
            a = net.grad(k[:, :700], t[:700])
            net.train(k[:, :700], t[:700], epochs=200, batch=128, lr=1e-3, seed=1)
            out.append((a, net.params))
    np.testing.assert_array_equal(out[0][0][0], out[1][0][0])
    # the Adam moments of the first calls differ, the fits do not by much
    assert np.linalg.norm(out[0][1] - out[1][1]) < 0.5 * np.linalg.norm(out[1][1])


@pytest.mark.parametrize("n,epochs", [(700, 200), (1000, 131), (140000, 3)])
def test_chunks_of_epochs_equal_single_epochs(n, epochs):
    """Epoch e of a run with seed s is shuffled from s + (e + 1) times a constant,
    so single-epoch calls whose seeds step by it see the same rows in the same
    batches: the same bits, whichever part of the index buffers a chunk of epochs
    went through (1, 2, 4, ... epochs, up to 131,072 points), and whether the
    buffers were made for this data set or for a larger one."""
    from mepinterp_amd import capi
    rng = np.random.default_rng(n)
    k = rng.uniform(-0.5, 0.5, size=(3, n))
    t = rng.normal(size=n).astype(np.float32)
    big = rng.uniform(-0.5, 0.5, size=(3, 200000))
    kw = dict(batch=8192 if n > 8192 else 128, lr=1e-3)
    out = []
    for first in (False, True):
        with capi.MLP(n_freq=2, hidden=32, seed=2) as net:
            if first:
                net.predict(big)
            out.append((net.train(k, t, epochs=epochs, seed=1, **kw), net.params))
    with capi.MLP(n_freq=2, hidden=32, seed=2) as net:
        for e in range(epochs):
            loss = net.train(k, t, epochs=1, seed=(1 + 0x9e3779b97f4a7c15 * e) % 2 ** 64, **kw)
        out.append((loss, net.params))
    for loss, p in out[1:]:
        assert loss == out[0][0]
        np.testing.assert_array_equal(p, out[0][1])
