"""The two-kernel inverse of large batches where it runs in earnest: through
the captured graph's replays, with its angles in groups, and in the rule that
selects it. Reference: the separate passes of a z-chunk of the whole volume,
launched eagerly; the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(X, Y, Z, n, A):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(X + 3 * Y + 5 * Z)
    V = torch.randn((Z, Y, X), generator=g, device="cuda") + 0.5
    rng = np.random.default_rng(Z + A)
    T = np.asfortranarray(rng.standard_normal((n, n, n)), np.float32)
    M = np.asfortranarray(rng.uniform(0.1, 1.0, (n, n, n)), np.float32)
    W = np.asfortranarray(rng.uniform(0.0, 1.0, (n, n, n)), np.float32)
    return V, T, M, W, rng.uniform(0, 360, (A, 3)).astype(np.float32)


def _run(api, ctx, V, T, M, W, ang, batch, zchunk, graph):
    tn, mu, sg = api.prepare_template(T, M, W)
    with api.SearchPlan(V, T.shape, M, batch=batch, ctx=ctx) as p:
        p.set_graph(graph)
        p.set_zchunk(zchunk)
        p.set_template(tn, W, mu, sg)
        p.run(ang, 0)
        first = [t.clone() for t in p.finalize()]
        # the graph again, on another list and with other first indices
        p.run(ang[::-1].copy(), len(ang))
        return first + [t.clone() for t in p.finalize()]


def _y_launches(api, V, T, M, ang, batch):
    tn, mu, sg = api.prepare_template(T, M, None)
    with api.SearchPlan(V, T.shape, M, batch=batch) as p:
        p.set_template(tn, None, mu, sg)
        p.profile(True)
        p.run(ang[:batch], 0)
        return int(p.profile(False)[1][4])


# every z length; classes of y taken in pairs of planes and singly; one group of
# angles and two; full batches for the graph and a last one that is not
CASES = [(512, 192, 32, 16), (512, 512, 32, 8), (256, 512, 64, 8), (384, 128, 64, 16), (256, 96, 128, 16),
         (512, 128, 128, 7), (128, 240, 128, 16), (256, 256, 192, 8), (512, 64, 256, 6), (128, 512, 256, 5)]


@pytest.mark.parametrize("X,Y,Z,batch", CASES)
def test_replay_equals_separate_passes(X, Y, Z, batch):
    import torch

    from tom_amd import api
    print("fused replay", X, Y, Z, batch, flush=True)
    A = 3 * batch + 2
    assert A // batch >= 2  # what a plan replays
    V, T, M, W, ang = _inputs(X, Y, Z, 24, A)
    assert _y_launches(api, V, T, M, ang, batch) == 0
    ref = _run(api, None, V, T, M, W, ang, batch, Z, False)
    ctx = api.Context(0)  # no twiddle list made before the capture
    try:
        got = _run(api, ctx, V, T, M, W, ang, batch, 0, True)
    finally:
        ctx.close()
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("X,Y,Z,batch", [(512, 384, 256, 1), (512, 192, 256, 2), (512, 96, 192, 6), (384, 96, 192, 8),
                                         (192, 240, 192, 6), (320, 384, 256, 2)])
def test_batches_that_lose_take_the_separate_passes(X, Y, Z, batch):
    """Batches that measured 6 to 20 % slower in the two kernels."""
    from tom_amd import api
    V, T, M, _, ang = _inputs(X, Y, Z, 16, batch)
    assert _y_launches(api, V, T, M, ang, batch) > 0
