"""Head gradient of the learned-proposal network against FP64 sums of the
logits' gradient, taken from the network's own FP32 logits.

Tolerance, per channel, relative to the sum of magnitudes: a value is a few
FP32 operations and library functions of its logits (below 16 units of 2^-24
together) and the longest chain of the FP32 sums has some 100 terms, so
1e-5 > 120 x 2^-24. Losses are FP64 sums of FP32 terms: 1e-5 likewise."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("nbin", [1, 5, 63, 64, 65, 76])
@pytest.mark.parametrize("offsets", [True, False])
def test_head_bias_gradient(nbin, offsets):
    from tom_amd import api
    print("head gradient", nbin, offsets, flush=True)
    rng = np.random.default_rng(nbin)
    nz, ny, nx = shape = (8, 12, 20)
    V = nz * ny * nx
    vol = rng.standard_normal(shape).astype(np.float32)
    tprob = rng.random(shape).astype(np.float32)
    tbin = np.where(rng.random(shape) < 0.1, rng.integers(0, nbin, shape), -1).astype(np.int32)
    tbin[0, 0, 0], tbin[-1, -1, -1] = nbin - 1, 0
    toff = np.zeros(shape + (4,), np.float32)
    toff[..., :3] = rng.uniform(-1.5, 1.5, shape + (3,))
    toff[..., 3] = rng.random(shape) < 0.1
    f = lambda a: a.transpose(2, 1, 0)  # noqa: E731
    with api.Unet((nx, ny, nz), nbin=nbin, seed=7, train=True) as net:
        net.forward(f(vol))
        L = np.asarray(net.logits(), np.float64).reshape(V, 80)
        loss = net.backward(f(tprob), f(tbin), 3.0, toff=toff.transpose(3, 2, 1, 0) if offsets else None)
        got = net.get_grads()[-80:].astype(np.float64)
    z, t, b = L[:, 0], tprob.reshape(-1).astype(np.float64), tbin.reshape(-1)
    p = 1 / (1 + np.exp(-z))
    G = np.zeros((V, 80))
    G[:, 0] = (3 * t * (p - 1) + (1 - t) * p) / V
    sel = np.flatnonzero(b >= 0)
    e = np.exp(L[sel, 1:1 + nbin] - L[sel, 1:1 + nbin].max(1, keepdims=True))
    soft = e / e.sum(1, keepdims=True)
    ce = -np.log(soft[np.arange(len(sel)), b[sel]]).mean()
    soft[np.arange(len(sel)), b[sel]] -= 1
    G[sel, 1:1 + nbin] = soft / len(sel)
    bce = (-(3 * t * np.log(p) + (1 - t) * np.log1p(-p))).mean()
    want = [bce, ce, 0.0]
    if offsets:
        o = toff.reshape(V, 4).astype(np.float64)
        on = np.flatnonzero(o[:, 3] > 0)
        d = L[on, 1 + nbin:4 + nbin] - o[on, :3]
        G[on, 1 + nbin:4 + nbin] = 2 * d / len(on)
        want[2] = (d ** 2).sum() / len(on)
    # near zero a difference of logit and target keeps the rounding of both
    slack = 1e-5 * np.abs(G).sum(0) + 1e-9
    assert (np.abs(got - G.sum(0)) <= slack).all(), np.abs(got - G.sum(0)) / slack
    for a, w in zip(loss, want):
        assert abs(a - w) <= 1e-5 * abs(w) + 1e-9
