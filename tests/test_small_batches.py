"""Small searches: where a batch has too few blocks, its orientations are
spread over groups of blocks and the groups' maxima merged in order. The maps
are the same bits as one orientation at a time (which has no groups), with the
first of equal maxima."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(V, T, M, ang, batch, tiles=(16, 16), graph=False, zchunk=0):
    from tom_amd import api
    tn, mu, sg = api.prepare_template(T, M, None)
    with api.SearchPlan(V, T.shape, M, batch=batch) as p:
        p.set_tiles(*tiles)
        p.set_graph(graph)
        p.set_zchunk(zchunk)
        p.set_template(tn, None, mu, sg)
        p.run(ang, 0)
        return p.finalize()


@pytest.mark.parametrize("X,Y,Z,box,batch,A,tiles", [
    (32, 16, 16, (8, 8, 8), 16, 35, (16, 16)), (64, 64, 64, (16, 16, 16), 16, 33, (16, 16)),
    (64, 64, 64, (24, 17, 9), 7, 16, (8, 32)), (64, 24, 40, (5, 24, 30), 16, 19, (32, 32)),
    (96, 48, 24, (20, 20, 20), 5, 11, (8, 8)), (160, 80, 16, (16, 16, 16), 3, 8, (16, 8)),
    (1024, 16, 32, (16, 16, 16), 16, 18, (16, 16)), (64, 48, 256, (24, 24, 24), 8, 12, (16, 16)),
])
def test_batches_equal_single_orientations(X, Y, Z, box, batch, A, tiles):
    import torch
    print(X, Y, Z, batch, tiles, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(X + Y + Z)
    V = torch.randn((Z, Y, X), generator=g, device="cuda") - 0.25
    rng = np.random.default_rng(X)
    T = np.asfortranarray(rng.standard_normal(box), np.float32)
    M = np.asfortranarray(rng.uniform(0.1, 1.0, box), np.float32)
    ang = rng.uniform(0, 360, (A, 3)).astype(np.float32)
    ang[A // 2] = ang[0]  # a tie at every voxel: the first stays
    ref_sc, ref_an = (a.cpu().numpy() for a in _run(V, T, M, ang, 1, tiles))
    assert not (ref_an == A // 2).any()
    for kw in ({}, {"graph": True}, {"zchunk": max(Z // 3, 1)}):
        sc, an = (a.cpu().numpy() for a in _run(V, T, M, ang, batch, tiles, **kw))
        assert np.array_equal(sc, ref_sc) and np.array_equal(an, ref_an), kw
