"""Rotations at sizes where the kernel's patches and planes do not fit, with
non-finite voxels, against the CPU oracle: the same bits."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def oracle():
    from oracle import tom_oracle as o
    return o


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 5), (15, 16, 3), (17, 33, 9), (64, 3, 70), (48, 31, 12),
                                   (16, 16, 64)])
def test_rotation_edges(oracle, shape):
    from tom_amd import api
    print("rotate", shape, flush=True)
    rng = np.random.default_rng(sum(shape))
    v = np.asfortranarray(rng.standard_normal(shape), np.float32)
    special = v.copy(order="F")
    if v.size > 1:
        flat = special.reshape(-1, order="F")
        flat[[0, v.size // 2, v.size - 1]] = np.nan, np.inf, -np.inf
    few = np.array([[0, 0, 0], [90, 0, 0], [30, 45, 60], [180, 0, 90]], np.float32)
    # rotations enough for eight planes a thread
    many = np.concatenate([few, rng.uniform(-360, 360, (196, 3)).astype(np.float32)])
    for vol, angles in ((v, few), (special, few), (special, many)):
        got = api.tom_rotate_batch(vol, angles)
        for a in range(0, len(angles), 1 if len(angles) < 9 else 13):
            want = oracle.rotate(vol, angles[a])
            assert np.array_equal(got[..., a], want, equal_nan=True), (a, angles[a])
            if a < 4:
                assert np.array_equal(api.tom_rotate(vol, angles[a]), want, equal_nan=True)
