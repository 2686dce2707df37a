"""Gradients of the learned-proposal network at sizes where the kernels' tiles
do not fit: rows shorter than 16 voxels, remainders in x and y, several units
of rows. Tolerance: that of the regular size (BF16 operands, FP32 sums)."""
import numpy as np
import pytest

from oracle import unet_ref as U
from test_unet import NBIN, _offsets, _targets, _theta


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 20, 36), (12, 40, 20), (8, 36, 100)])
def test_gradients_at_ragged_sizes(shape):
    from tom_amd import api
    print("unet gradients", shape, flush=True)
    rng = np.random.default_rng(sum(shape))
    vol = rng.standard_normal(shape).astype(np.float32)
    theta = _theta(rng).astype(np.float32)
    tprob, tbin = _targets(rng, shape)
    tprob[0, 0, 0], tbin[0, 0, 0] = 1.0, NBIN - 1
    toff = _offsets(rng, shape)
    f = lambda a: a.transpose(2, 1, 0)  # noqa: E731
    with api.Unet(shape[::-1], nbin=NBIN, seed=1, train=True) as net:
        net.set_params(theta)
        net.forward(f(vol))
        loss = net.backward(f(tprob), f(tbin), 4.0, toff=toff.transpose(3, 2, 1, 0))
        g = net.get_grads()
        again = net.backward(f(tprob), f(tbin), 4.0, toff=toff.transpose(3, 2, 1, 0))
        g2 = net.get_grads()
    *ref, rg = U.gradients(vol, theta.astype(np.float64), tprob, tbin, NBIN, 4.0, bf16=True, toff=toff)
    for a, b, c in zip(loss, again, ref):
        assert abs(a - c) <= 1e-3 * abs(c) and abs(a - b) <= 1e-6 * abs(a)
    at = 0
    for li, (ci, co, t, _) in enumerate(U.SPEC):
        n = t * co * ci
        a, b = g[at:at + n + co].astype(np.float64), rg[at:at + n + co]
        cos = a @ b / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-300)
        rel = np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-300)
        print(f"  layer {li}: cos {cos:.5f} rel {rel:.3e}", flush=True)
        assert cos >= 0.9999 and rel <= 1e-2, li
        # the weights' sums are taken in one fixed order
        assert np.array_equal(g[at:at + n], g2[at:at + n]), li
        at += n + co
