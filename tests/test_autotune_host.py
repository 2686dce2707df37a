"""The autotuner's host logic on the CPU, with a stand-in for the plan: results
of another set of kernels are not reused, and stages that cannot change what
runs are left out."""
import json

import numpy as np
import pytest


class Plan:
    fused = True
    made = []

    def __init__(self, volume, shape, mask, batch=4):
        self.n = np.shape(volume)
        self.cfg = dict(batch=batch)
        Plan.made.append(self.cfg)

    def __enter__(self):
        return self

    def __exit__(self, *a):
        pass

    def set_tiles(self, tz, ty):
        self.cfg.update(tz=tz, ty=ty)

    def set_zchunk(self, zc):
        self.cfg.update(zc=zc)

    def set_template(self, *a):
        pass

    def run(self, ang, first):
        pass

    def profile(self, on):
        sep = not Plan.fused or self.cfg["zc"] or (self.n[2] == 256 and self.cfg["tz"] != 16)
        return np.zeros(8), np.array([0, 0, 0, 1, 1 if sep else 0, 1, 0, 0])

    def finalize(self):
        return np.zeros((2, 2)), np.zeros((2, 2), np.int32)


@pytest.fixture
def tune(monkeypatch, tmp_path):
    import torch

    from tom_amd import api, autotune
    monkeypatch.setenv("TOM_AMD_CACHE", str(tmp_path))
    monkeypatch.setattr(api, "SearchPlan", Plan)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda *a: None)
    Plan.made = []

    def run(Z, fused):
        Plan.fused = fused
        Plan.made = []
        V = np.zeros((64, 64, Z), np.float32)
        t = np.zeros((16, 16, 16), np.float32)
        return autotune.tune_search(V, t, None, None, 0.0, 1.0, np.zeros((100, 3)), batches=(4, 16))
    return run, tmp_path, autotune


def test_tile_stages_that_change_nothing_are_left_out(tune):
    run, _, _ = tune
    run(128, True)
    assert {(c["tz"], c["ty"]) for c in Plan.made} == {(16, 16)}
    assert {c["zc"] for c in Plan.made} == {0, 64, 32}
    run(256, True)  # there the z tile selects the passes
    assert {c["tz"] for c in Plan.made} == {8, 16, 32}
    run(120, False)
    assert {c["tz"] for c in Plan.made} == {8, 16, 32} and {c["ty"] for c in Plan.made} == {8, 16, 32}


def test_results_of_other_kernels_are_not_reused(tune):
    run, path, autotune = tune
    key = autotune._key((64, 64, 128), (16, 16, 16))
    old = key.split("|", 1)[1]  # as it was without the set of kernels
    (path / "autotune.json").write_text(json.dumps({old: dict(batch=2, tile_z=8, tile_y=8, zchunk=64)}))
    assert not run(128, True)["cached"]
    assert run(128, True)["cached"]
