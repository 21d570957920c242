"""A plan over a projector takes the march of the projector as it is, whatever
was called before, and a schedule tuned for one march is not used for another
(no GPU needed: the plan itself is a stand-in)."""
import types

import pytest

from deepdrr_amd import batch, phantoms


def _plan(monkeypatch, march, add_noise):
    log = []
    monkeypatch.setattr(batch, "BatchPlan", lambda *a, tune_key=None, **k: log.append(("plan", tune_key)))
    vol = phantoms.uniform_volume((4, 5, 6))
    p = types.SimpleNamespace(initialized=True, max_ray_length=4000.0, source_to_detector_distance=1000.0,
                              volumes=[vol], priorities=[0], all_materials=["air"], march=march, add_noise=add_noise,
                              neglog=True, _ctx=None, _vols=[None], _torch_device=None)
    p._set_sums = lambda: log.append(("sums", p.add_noise))
    batch.plan_for_projector(p, [phantoms.ap_device(8, 8, 1.0).get_camera_projection()], tuning="auto")
    return log


@pytest.mark.parametrize("add_noise", [False, True])
def test_sums_are_set_before_the_plan(monkeypatch, add_noise):
    (a, noise), (b, _) = _plan(monkeypatch, "fast", add_noise)
    assert (a, b, noise) == ("sums", "plan", add_noise)


def test_keys_tell_the_marches_apart(monkeypatch):
    keys = [_plan(monkeypatch, *m)[-1][1] for m in (("fast", False), ("fast", True), ("exact", False), ("exact", True))]
    assert keys[0] != keys[1] and keys[0] != keys[2] and keys[1] != keys[2]
    assert keys[2] == keys[3]  # noise does not change the exact march
