"""Batched subtomogram scoring: a batch that takes several passes over the
device's spectra gives each particle what a call of its own gives, and
non-finite particles stay without a peak."""
import numpy as np
import pytest


def _inputs(n, count, orientations, seed, wedge_ref=None):
    rng = np.random.default_rng(seed)
    g = np.arange(n) - n / 2
    r = np.sqrt(g[:, None, None] ** 2 + g[None, :, None] ** 2 + g[None, None, :] ** 2)
    box = {"template": rng.standard_normal((n, n, n)).astype(np.float32),
           "mask": np.clip(n / 2 - 3 - r, 0, 1).astype(np.float32),
           "mask_cc": (r < 5).astype(np.float32)}
    if wedge_ref is not None:
        box["wedge_ref"] = wedge_ref
    parts = [rng.standard_normal((n, n, n)).astype(np.float32) for _ in range(count)]
    semi = [(-1.0, 30.0)[i % 2] for i in range(count)]
    angles = rng.uniform(0, 360, (count, orientations, 3)).astype(np.float32)
    return box, parts, semi, angles


@pytest.mark.gpu
@pytest.mark.parametrize("n,count,orientations,wedge_ref",
                         [(32, 70, 40, None), (32, 40, 40, 25.0), (48, 30, 21, None), (64, 17, 16, 30.0)])
def test_batch_equals_single_calls(n, count, orientations, wedge_ref):
    """Every item is worked on alone and its sums are taken in an order of its
    own, so the results are the same bits however a batch is cut."""
    from tom_amd import api
    box, parts, semi, angles = _inputs(n, count, orientations, n + count, wedge_ref)
    best, peak, ccc = api.subtomo_score_batch([box], parts, [0] * count, semi, angles)
    for i in (0, 1, count // 2, count - 2, count - 1):
        b, p, c = api.subtomo_score_batch([box], [parts[i]], [0], [semi[i]], angles[i:i + 1])
        assert best[i] == b[0] and list(peak[i]) == list(p[0]) and ccc[i] == c[0], i


@pytest.mark.gpu
def test_non_finite_particle_has_no_peak():
    from tom_amd import api
    box, parts, semi, angles = _inputs(32, 3, 5, 3)
    parts[1][0, 0, 0] = np.nan  # outside the mask: its spectrum is NaN all the same
    best, peak, ccc = api.subtomo_score_batch([box], parts, [0] * 3, semi, angles)
    assert best[1] == -1 and np.isnan(ccc[1]) and list(peak[1]) == [0, 0, 0]
    assert (best[[0, 2]] >= 0).all() and np.isfinite(ccc[[0, 2]]).all()
