"""The learned proposal's network on the matrix cores against the oracle
(oracle/guide.py): forward outputs and mixtures, the loss and its gradient
with respect to all 21,808 parameters, the Adam update, and that online
training fits a known directional distribution."""
import numpy as np
import pytest

from oracle import guide as G

pytestmark = pytest.mark.gpu


def _inputs(seed, n):
    rng = np.random.default_rng(seed)
    pos = rng.random((n, 3))
    wo = rng.normal(size=(n, 3))
    wo /= np.linalg.norm(wo, axis=1, keepdims=True)
    nn = rng.normal(size=(n, 3))
    nn /= np.linalg.norm(nn, axis=1, keepdims=True)
    return G.features(pos, wo, nn, rng.random(n)), rng


def _theta(seed):
    th = G.init_params(seed)
    th = th + np.random.default_rng(seed + 1).normal(scale=0.05, size=th.size).astype(np.float32)
    return th.astype(np.float32)


def _close(got, ref, q=0.999, tol=2e-2):
    scale = np.sqrt(np.mean(ref ** 2)) + 1e-12
    err = np.abs(got - ref) / (np.abs(ref) + 0.05 * scale)
    return float(np.quantile(err, q)) < tol and float(err.max()) < 0.5, float(np.quantile(err, q)), float(err.max())


def test_forward_matches_oracle(backend):
    th = _theta(11)
    x, _ = _inputs(12, 1000)            # not a multiple of the 64-row tile
    backend.guide_init(params=th)
    out, mix = backend.guide_eval(x)
    ref = G.forward(th, x)
    ok, q, mx = _close(out, ref)
    print("forward rel err q999 %.3e max %.3e" % (q, mx), flush=True)
    assert ok
    w, k, mu, _, _ = G.decode(out.astype(np.float64))
    m = mix.reshape(-1, 8, 5)
    assert np.allclose(m[:, :, 0], w, rtol=1e-5, atol=1e-7)
    assert np.allclose(m[:, :, 1], k, rtol=1e-5)
    assert np.allclose(m[:, :, 2:5], mu, atol=1e-6)


def test_gradient_matches_oracle(backend):
    th = _theta(21)
    x, rng = _inputs(22, 4096)
    d = rng.normal(size=(4096, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    c = rng.random(4096) * 3
    backend.guide_init(params=th)
    loss = backend.guide_train_step(x, d, c, apply=False)
    _, g = backend.guide_params()
    rl, rg = G.loss_and_grad(th, x, d, c)
    print("loss gpu %.6f oracle %.6f" % (loss, rl), flush=True)
    assert loss == pytest.approx(rl, rel=2e-3)
    cos = float(np.dot(g, rg) / (np.linalg.norm(g) * np.linalg.norm(rg)))
    print("gradient cosine %.6f" % cos, flush=True)
    assert cos > 0.999
    k = 0
    for i, o in G.LAYERS:
        for size in (o * i, o):
            a, b = g[k:k + size], rg[k:k + size]
            rel = np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12)
            assert rel < 0.05, (i, o, size, rel)
            k += size


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 32767, 32769, 70001])
def test_gradient_at_tile_edges(backend, n):
    """Rows short of a wave's 16, of a block's 64 and of one tile per block,
    and blocks with several tiles.  Each of the rows on either side of those
    edges carries 98 % of the weight in turn, so that a row lost or counted
    twice takes or doubles nearly all of the loss and the gradient.  The
    matrix products read bfloat16 (2^-9 relative per operand): through ten of
    them the gradient of a layer keeps its norm to 5 % over a large batch, and
    for a single row, whose gradient hangs on a few lobes' concentrations (exp
    of a rounded output), to 10 %; the loss to 2 %."""
    th = _theta(41)
    x, rng = _inputs(42, n)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    c = rng.random(n) + 0.1
    # of the first tile, of the first block (of 512, each of consecutive tiles
    # of 64 rows) and of the last tile
    tiles = (n + 63) // 64
    share = -(-tiles // 512)
    edges = {0, 15, 16, 63, 64, 64 * share - 1, 64 * share, 64 * (tiles - 1) - 1, 64 * (tiles - 1), n - 1}
    edges = sorted(e for e in edges if 0 <= e < n)
    c[edges] = 0.0
    rest = c.sum()
    rest_loss, rest_grad = G.loss_and_grad(th, x, d, c) if rest > 0 else (0.0, np.zeros(len(th)))
    backend.guide_init(params=th)
    for e in edges:
        w = c.copy()
        w[e] = max(1.0, 49.0 * rest)
        one_loss, one_grad = G.loss_and_grad(th, x[e:e + 1], d[e:e + 1], w[e:e + 1])
        share_e = w[e] / (w[e] + rest)
        rl = share_e * one_loss + (1.0 - share_e) * rest_loss
        rg = share_e * one_grad + (1.0 - share_e) * rest_grad
        before = backend.guide_params()[1]  # gradients add up until a step applies them
        loss = backend.guide_train_step(x, d, w, apply=False)
        g = backend.guide_params()[1] - before
        assert loss == pytest.approx(rl, rel=2e-2), e
        k = 0
        for i, o in G.LAYERS:
            for size in (o * i, o):
                a, b = g[k:k + size], rg[k:k + size]
                rel = np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12)
                assert rel < 0.10, (e, i, o, size, rel)
                k += size


def test_adam_step_matches_oracle(backend):
    th = _theta(31)
    x, rng = _inputs(32, 2048)
    d = rng.normal(size=(2048, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    c = rng.random(2048)
    backend.guide_init(params=th, lr=1e-2)
    backend.guide_train_step(x, d, c, apply=True)
    th1, gres = backend.guide_params()
    assert not gres.any()                 # gradient buffer cleared by the update
    _, rg = G.loss_and_grad(th, x, d, c)
    ref = G.Adam(th.size, lr=1e-2).step(th, rg)
    moved = np.abs(rg) > 1e-6
    agree = np.isclose(th1, ref, atol=2e-4)
    print("adam agreement %.5f" % agree[moved].mean(), flush=True)
    assert agree[moved].mean() > 0.99


def test_training_fits_known_distribution(backend):
    """Directions drawn from a vMF whose mean depends on position: online
    training must raise the likelihood of held-out samples well above the
    uniform density 1/(4 pi)."""
    rng = np.random.default_rng(41)

    def batch(n):
        pos = rng.random((n, 3))
        mu = np.stack([np.cos(2 * np.pi * pos[:, 0]), np.sin(2 * np.pi * pos[:, 0]), np.zeros(n)], 1)
        x = G.features(pos, np.tile([0, 0, 1.0], (n, 1)), np.tile([0, 1.0, 0], (n, 1)), np.full(n, 0.5))
        d = G.vmf_sample(np.full(n, 20.0), mu, rng.random(n), rng.random(n))
        return x, d
    backend.guide_init(seed=5, lr=1e-2)
    losses = []
    for it in range(300):
        x, d = batch(4096)
        losses.append(backend.guide_train_step(x, d, np.ones(4096)))
    xt, dt = batch(4096)
    _, mix = backend.guide_eval(xt)
    m = mix.reshape(-1, 8, 5).astype(np.float64)
    q = G.mixture_pdf(m[:, :, 0], m[:, :, 1], m[:, :, 2:5], dt)
    print("loss first %.3f last %.3f  mean held-out log q %.3f" % (losses[0], losses[-1], np.log(q).mean()),
          flush=True)
    assert losses[-1] < losses[0] - 1.0
    assert np.log(q).mean() > np.log(1 / (4 * np.pi)) + 1.5
