"""Which march feeds the noise: with single sums (drr_ctx_set_single_sums) the
area densities differ from the closed ones and are nearer to the transcription;
a projector with noise renders, and plans, with single sums whatever was called
before, and one without noise never does."""
import ctypes as C

import numpy as np
import pytest
import torch

from deepdrr_amd import Projector, _abi, phantoms
from deepdrr_amd._abi_types import MARCH_FAST
from deepdrr_amd.batch import plan_for_projector
from deepdrr_amd.spectral_data import synthetic_120kv
from tests import scenes
from tests.scenes import GpuRunner
from tests.test_gpu_fast import _oracle

pytestmark = pytest.mark.gpu


def _body():
    """A smooth body of 240 mm: some 2400 samples a ray."""
    n = 40
    i, j, k = np.meshgrid(*(np.linspace(-1, 1, n),) * 3, indexing="ij")
    hu = np.where(i * i + j * j + k * k < 0.8, 60.0 + 40.0 * np.sin(9 * i) * np.cos(7 * j), -1000.0).astype(np.float32)
    vol = phantoms.Volume.from_hu(hu, origin=phantoms._centered_origin((n, n, n), (6, 6, 6)), spacing=(6, 6, 6),
                                  anatomical_coordinate_system="LPS",
                                  material_classes=phantoms.FIVE_MATERIAL_CLASSES)
    return vol, phantoms.ap_device(48, 36, 5.0, sdd=900.0)


def test_single_sums_are_nearer(gpu):
    vol, dev = _body()
    case = scenes.make_case("body", [vol], dev.get_camera_projection())
    case.scene.march = MARCH_FAST
    want = _oracle(case)[2].astype(np.float64)
    r = GpuRunner(case)
    try:
        ad = {}
        for single in (1, 0):
            _abi.call("drr_ctx_set_single_sums", r.ctx, single)
            ad[single] = r.project()[2]
    finally:
        r.close()
    assert not np.array_equal(ad[0], ad[1])
    # each sample's density is off by some 1e-7, and an addition rounds the other
    # way in one of thousands: a few ulp of the sum
    tot = want.sum(0)
    err = {s: float((np.abs(a - want).max(0) / np.where(tot > 0, tot, 1.0)).max()) for s, a in ad.items()}
    print(f"largest difference from the transcription: {err[1]:.2e} single, {err[0]:.2e} closed")
    assert err[1] <= 1e-6 and err[1] < err[0]


def _mode(p, proj, single):
    """The view with the context's flag set by hand."""
    _abi.call("drr_ctx_set_single_sums", p._ctx, single)
    view = p.view_for(proj)
    I, P = (torch.empty((view.height, view.width), device="cuda") for _ in range(2))
    _abi.call("drr_project", p._ctx, p._vol_array, C.byref(view), _abi.ptr(I), _abi.ptr(P), None, None, None)
    torch.cuda.synchronize()
    return I.cpu().numpy(), P.cpu().numpy()


def _plan(p, proj, tuning=None):
    plan = plan_for_projector(p, [proj], tuning=tuning)
    try:
        plan.launch()
        torch.cuda.synchronize()
        return plan.fetch("intensity")[0], plan.fetch("photon_prob")[0]
    finally:
        plan.close()


@pytest.mark.parametrize("tuning", [None, "auto"])
def test_plans_do_not_depend_on_earlier_calls(gpu, tuning):
    vol, dev = _body()
    proj = dev.get_camera_projection()
    with Projector(vol, device=dev, step=0.1, spectrum=synthetic_120kv(), neglog=False, add_noise=True,
                   photon_count=20000) as p:
        first = _plan(p, proj, tuning)  # before anything was projected
        area = [x.reshape(first[0].shape) for x in p.project_area_density(proj)[1:]]
        p.add_noise = False
        plain = _plan(p, proj, tuning)
        p.project(proj)
        p.add_noise = True
        again = _plan(p, proj, tuning)
        single, closed = _mode(p, proj, 1), _mode(p, proj, 0)
        assert not np.array_equal(single[1], closed[1])
        for k in range(2):
            assert np.array_equal(first[k], single[k]) and np.array_equal(again[k], single[k])
            assert np.array_equal(area[k], single[k]) and np.array_equal(plain[k], closed[k])
