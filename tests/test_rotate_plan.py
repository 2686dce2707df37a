"""Rotations by each way of dividing the volume: tiles of columns, columns
numbered through, one and several planes a thread, more plane groups than a
grid dimension holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,count", [
    ((12, 12, 12), 3), ((12, 12, 12), 1500), ((20, 20, 20), 300), ((17, 17, 17), 700), ((24, 40, 31), 120),
    ((60, 60, 5), 300), ((52, 50, 9), 300), ((47, 48, 33), 40), ((1, 1, 300), 4), ((2, 130, 3), 1100),
    ((3, 700, 600), 2), ((130, 70, 120), 1), ((16, 16, 2), 2100)])
def test_every_division_matches_the_oracle(shape, count):
    from oracle import tom_oracle as oracle
    from tom_amd import api
    print("rotate", shape, count, flush=True)
    rng = np.random.default_rng(count)
    v = np.asfortranarray(rng.standard_normal(shape), np.float32)
    m = np.asfortranarray(rng.standard_normal(shape), np.float32)
    ang = rng.uniform(-360, 360, (count, 3)).astype(np.float32)
    got = api.tom_rotate_batch(v, ang)
    gotm = api.tom_rotate_batch(v, ang, mask=m)
    for a in sorted({0, count // 2, count - 1}):
        want = oracle.rotate(v, ang[a])
        assert np.array_equal(got[..., a], want), a
        assert np.array_equal(gotm[..., a], want * m), a


def test_more_planes_than_a_grid_dimension_times_eight():
    """600,000 planes of 16 x 16: rotated about z each plane goes by itself, so
    any stretch of planes is what a short volume of them gives."""
    import torch

    from tom_amd import api
    g = torch.Generator(device="cuda")
    g.manual_seed(6)
    n = 600_000
    v = torch.randn((n, 16, 16), generator=g, device="cuda")
    e = np.array([37.0, 0.0, 0.0], np.float32)
    got = api.tom_rotate(v, e)
    for z in (0, 65535 * 8 - 20, n - 40):
        assert torch.equal(got[z:z + 40], api.tom_rotate(v[z:z + 40].contiguous(), e)), z
