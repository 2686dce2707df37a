"""Reference weighting of template boxes at every edge length it is built for,
square planes and uneven ones, small and large batches, against the FP64
oracle. Tolerance: a score is a ratio of FP32 sums over at most 64^3 voxels
whose terms carry the rounding (2^-24 each, some 20 operations deep) of two
box and three volume transforms; the sums of such independent roundings stay
below 40 x 2^-24 of a score of order one, 1e-5 taken."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def oracle():
    from oracle import tom_oracle as o
    return o


@pytest.mark.gpu
@pytest.mark.parametrize("box", [(16, 16, 24), (24, 24, 40), (40, 40, 16), (32, 32, 48), (48, 48, 32), (64, 64, 64),
                                 (40, 32, 24), (24, 64, 48)])
@pytest.mark.parametrize("batch", [1, 5])
def test_weighted_search_matches_oracle(oracle, box, batch):
    from tom_amd import api
    print("box", box, batch, flush=True)
    rng = np.random.default_rng(sum(box))
    V = np.asfortranarray(rng.standard_normal((64, 64, 64)), np.float32)
    T = np.asfortranarray(rng.standard_normal(box), np.float32)
    M = np.asfortranarray(rng.uniform(0.2, 1.0, box), np.float32)
    W = oracle.wedge(box, 40).astype(np.float32)
    angles = np.concatenate([[[0, 0, 0]], rng.uniform(0, 360, (6, 3))])
    ccc, ang = api.tom_os3_findTemplate(V, T, M, angles, W=W, batch=batch)
    _, _, allm = oracle.find_template(V, T, M, angles, W=W, return_all=True)
    allm = np.asarray(allm)
    assert np.abs(np.asarray(ccc) - allm.max(0)).max() < 1e-5
    at = np.asarray(ang).astype(int) - 1
    picked = np.take_along_axis(allm, at[None], 0)[0]
    assert (allm.max(0) - picked).max() < 2e-5
