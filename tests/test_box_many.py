"""More weighted boxes in one refinement than a grid dimension holds, uneven
and square planes: each candidate as in a refinement of a part of them, and in the
other order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [(24, 16, 16), (16, 16, 24)])
def test_refinement_of_many_boxes(box):
    import torch

    from tom_amd import api
    print("boxes", box, flush=True)
    P, A = 600, 112  # 67,200 boxes
    g = torch.Generator(device="cuda")
    g.manual_seed(8)
    V = torch.randn((48, 64, 64), generator=g, device="cuda")
    rng = np.random.default_rng(8)
    T = np.asfortranarray(rng.standard_normal(box), np.float32)
    M = np.ones(box, np.float32, order="F")
    W = np.asfortranarray(rng.uniform(0, 1, box), np.float32)
    ga = rng.uniform(0, 360, (A, P, 3)).astype(np.float32)
    cand = np.stack([rng.integers(0, 48, P) for _ in range(3)] + [np.arange(P)], 1).astype(np.int32)
    tn, mu, sg = api.prepare_template(T, M, W)
    with api.SearchPlan(V, box, M) as p:
        p.set_template(tn, W, mu, sg)
        got = p.refine(V, ga, cand)
        # the orientations past 65,535 boxes, the last three, are some candidates'
        # best, and the same ones where they come first
        last = got[1] >= 65536 // P
        assert last.sum() >= 5
        rev = p.refine(V, np.ascontiguousarray(ga[::-1]), cand)
        assert np.array_equal(rev[0], got[0]) and np.array_equal(rev[2], got[2])
        assert np.array_equal(A - 1 - rev[1], got[1])
        for i in (0, 590):
            part = cand[i:i + 10].copy()
            part[:, 3] -= i
            want = p.refine(V, ga[:, i:i + 10], part)
            for a, b in zip(got, want):
                assert np.array_equal(a[i:i + 10], b), i
