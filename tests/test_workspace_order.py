"""A workspace that is given back while its stream still has work queued, and
taken by a call on another stream: both calls return what they return alone
(the same kernels: the same bits)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_workspace_returned_while_its_stream_is_busy():
    import torch

    from tom_amd import api
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(4)
    n, first, more = 24, 40, 400
    V = torch.from_numpy(rng.standard_normal((64, 64, 64)).astype(np.float32)).to(dev)
    T = np.asfortranarray(rng.standard_normal((n, n, n)), np.float32)
    M = np.ones((n, n, n), np.float32, order="F")
    W = np.asfortranarray(rng.uniform(0, 1, (n, n, n)), np.float32)
    tn, mu, sg = api.prepare_template(T, M, W)
    ang = rng.uniform(0, 360, (first + more, 3)).astype(np.float32)
    box = torch.from_numpy(rng.standard_normal((n, n, n)).astype(np.float32)).to(dev)
    other = rng.uniform(0, 360, (first, 3)).astype(np.float32)  # a list of the length of the first one
    a = torch.randn((2048, 2048), device=dev)
    torch.cuda.synchronize()
    with api.SearchPlan(V, (n, n, n), M, batch=8) as p:
        p.set_template(tn, W, mu, sg)
        p.run(ang, 0)
        ref = [t.clone() for t in p.finalize()]
    ref_rot = api.tom_rotate_batch(box, other).clone()
    torch.cuda.synchronize()
    ctxs = [api.Context(0), api.Context(0)]
    try:
        side = [torch.cuda.Stream(device=dev) for _ in range(2)]
        with torch.cuda.stream(side[0]):
            p = api.SearchPlan(V, (n, n, n), M, batch=8, ctx=ctxs[0])
            p.set_template(tn, W, mu, sg)
            for _ in range(40):
                a = torch.tanh(a @ a * (1.0 / 64.0))
            p.run(ang[:first], 0)
            p.run(ang[first:], first)  # a longer list: the first one's memory goes back
        with torch.cuda.stream(side[1]):
            rot = api.tom_rotate_batch(box, other, ctx=ctxs[1])
        with torch.cuda.stream(side[0]):
            got = p.finalize()
        torch.cuda.synchronize()
        assert torch.equal(rot, ref_rot)
        assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])
        p.close()
    finally:
        for c in ctxs:
            c.close()
