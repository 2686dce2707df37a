"""The two-kernel inverse of large search batches (fused.hip) against the
separate z, y and x passes, which a z-chunk of the whole volume selects: the
same bits at every length it is built for, and FP64 direct sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from tom_amd import api as a
    return a


@pytest.fixture(scope="module")
def oracle():
    from oracle import tom_oracle as o
    return o


def _run(api, V, T, M, W, ang, batch, zchunk, graph):
    tn, mu, sg = api.prepare_template(T, M, W)
    with api.SearchPlan(V, T.shape, M, batch=batch) as p:
        p.set_graph(graph)
        p.set_zchunk(zchunk)
        p.set_template(tn, W, mu, sg)
        p.profile(True)
        p.run(ang[:batch], 0)
        _, n = p.profile(False)
        p.run(ang[batch:], batch)
        sc, an = p.finalize()
    return sc, an, int(n[4])


# X, Y, Z, box, batch, orientations: every length, smallest and largest
# template extents, batches that are not full, both kinds of plane groups
CASES = [
    (256, 96, 128, (24, 24, 24), 16, 37), (512, 192, 32, (64, 64, 32), 16, 32), (192, 128, 192, (48, 31, 64), 16, 35),
    (128, 240, 128, (33, 9, 17), 16, 34), (320, 384, 64, (16, 16, 16), 8, 17), (384, 320, 64, (1, 1, 1), 8, 16),
    (256, 512, 64, (40, 40, 40), 8, 20), (512, 64, 256, (64, 64, 64), 12, 25), (256, 480, 64, (8, 64, 5), 8, 9),
    (320, 160, 256, (32, 32, 32), 5, 10), (384, 256, 32, (24, 2, 32), 16, 33), (512, 512, 64, (48, 48, 48), 4, 7),
]


@pytest.mark.parametrize("X,Y,Z,box,batch,A", CASES)
def test_fused_equals_separate_passes(api, X, Y, Z, box, batch, A):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(X + Y + Z)
    V = torch.randn((Z, Y, X), generator=g, device="cuda") + 0.5
    rng = np.random.default_rng(Z)
    T = np.asfortranarray(rng.standard_normal(box), np.float32)
    M = np.asfortranarray(rng.uniform(0.1, 1.0, box), np.float32)
    ang = rng.uniform(0, 360, (A, 3)).astype(np.float32)
    ref = _run(api, V, T, M, None, ang, batch, Z, False)
    assert ref[2] > 0  # a y pass of its own
    for graph in (False, True):
        got = _run(api, V, T, M, None, ang, batch, 0, graph)
        assert got[2] == 0
        assert torch.equal(got[1], ref[1])
        assert torch.equal(got[0], ref[0])


def test_fused_matches_direct_sums(api, oracle):
    """Scores at sampled voxels, borders included, within the 1e-4 of the
    search's FP64 comparisons; weighted template."""
    import torch
    X, Y, Z, n, A = 256, 96, 128, 24, 16
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    V = torch.randn((Z, Y, X), generator=g, device="cuda")
    rng = np.random.default_rng(3)
    T = np.asfortranarray(rng.standard_normal((n, n, n)), np.float32)
    M = oracle.sphere_mask_binary(n, 10)
    W = oracle.wedge((n, n, n), 30).astype(np.float32)
    ang = rng.uniform(0, 360, (A, 3)).astype(np.float32)
    sc, an, y_launches = _run(api, V, T, M, W, ang, 16, 0, False)
    assert y_launches == 0
    vox = np.stack([rng.integers(0, N, 200) for N in (X, Y, Z)], 1)
    vox[:8] = [(x, y, z) for x in (0, X - 1) for y in (0, Y - 1) for z in (0, Z - 1)]
    Tn, mu, sg = oracle.prepare_template(T, M, W)
    ref = oracle.flcf_at_voxels(V.cpu().numpy().transpose(2, 1, 0), Tn, M, mu, sg, ang, vox, W=W)
    got = sc.cpu().numpy()[vox[:, 2], vox[:, 1], vox[:, 0]]
    assert np.abs(got - ref.max(1)).max() < 1e-4
    best = an.cpu().numpy()[vox[:, 2], vox[:, 1], vox[:, 0]]
    top = np.sort(ref, 1)
    clear = top[:, -1] - top[:, -2] > 1e-4
    assert np.array_equal(best[clear], ref.argmax(1)[clear])
