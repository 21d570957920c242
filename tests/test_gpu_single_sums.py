"""The fast march with every sample added singly (drr_ctx_set_single_sums), which
views with noise take: the bars of the fast march against the transcription and
its other sums, batched images bit-identical to single views, and a projector
with noise marches so."""
import numpy as np
import pytest

from deepdrr_amd import _abi, phantoms
from deepdrr_amd._abi_types import MARCH_FAST
from tests import scenes
from tests.scenes import GpuRunner
from tests.test_gpu_fast import _check_close, _oracle
from tests.test_gpu_forward import _materials_scene, _random_scene

pytestmark = pytest.mark.gpu


def _single(r, on=True):
    _abi.call("drr_ctx_set_single_sums", r.ctx, 1 if on else 0)


@pytest.mark.parametrize("seed", range(12))
def test_random_scenes(gpu, seed):
    case = _random_scene(seed)
    case.scene.march = MARCH_FAST
    r = GpuRunner(case)
    try:
        _single(r)
        a = r.project()
        _check_close(case.name, a, _oracle(case))
        _single(r, False)
        _check_close(case.name, a, r.project()[:3])  # the two sums are as close
    finally:
        r.close()


@pytest.mark.parametrize("k", [1, 5, 16])
def test_batches(gpu, k):
    import torch

    from deepdrr_amd.batch import BatchPlan

    case, vol, projs = _materials_scene(40 + k, k)
    case.scene.march = MARCH_FAST
    r = GpuRunner(case)
    try:
        _single(r)
        _check_close(case.name, r.project(), _oracle(case))
        views = [case.view] + [scenes.P.build_view([vol], [0], pr, 4080.0) for pr in projs[1:]]
        singles = [r.project(v)[:2] for v in views]
        for tuning in ((8, 8, 4, 8), (16, 4, 2, 4)):
            plan = BatchPlan(r.ctx, [r.vols[0]], views, [0] * len(views), neglog=False, tuning=tuning)
            _single(r, False)  # a plan keeps the march it was made with
            plan.launch()
            torch.cuda.synchronize()
            I_b, P_b = plan.fetch("intensity"), plan.fetch("photon_prob")
            plan.close()
            _single(r)
            for i, (I, P) in enumerate(singles):
                assert np.array_equal(I.view(np.uint32), I_b[i].view(np.uint32)), f"view {i}, {tuning}"
                assert np.array_equal(P.view(np.uint32), P_b[i].view(np.uint32)), f"view {i}, {tuning}"
    finally:
        r.close()


def test_projector_with_noise(gpu):
    import ctypes as C

    import torch

    from deepdrr_amd import Projector
    from deepdrr_amd.spectral_data import synthetic_120kv

    n = 40
    i, j, k = np.meshgrid(*(np.linspace(-1, 1, n),) * 3, indexing="ij")
    hu = np.where(i * i + j * j + k * k < 0.8, 60.0 + 40.0 * np.sin(9 * i) * np.cos(7 * j), -1000.0).astype(np.float32)
    vol = phantoms.Volume.from_hu(hu, origin=phantoms._centered_origin((n, n, n), (6, 6, 6)), spacing=(6, 6, 6),
                                  anatomical_coordinate_system="LPS",
                                  material_classes=phantoms.FIVE_MATERIAL_CLASSES)
    dev = phantoms.ap_device(64, 48, 4.0, sdd=900.0)
    proj = dev.get_camera_projection()
    with Projector(vol, device=dev, step=0.1, spectrum=synthetic_120kv(), neglog=False, add_noise=True,
                   photon_count=20000) as p:
        p.noise_seed = 7
        noisy = p.project_batch(proj)
        _, I, P = p.project_area_density(proj)
        I, P = (np.asarray(x, np.float32) for x in (I, P))
        d = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (I, P)]
        want = torch.empty_like(d[0])
        _abi.call("drr_add_noise", p._ctx, _abi.ptr(d[0]), _abi.ptr(d[1]), _abi.ptr(want), 1, *I.shape[-2:],
                  C.c_float(20000), C.c_uint64(7), None)
        torch.cuda.synchronize()
        assert np.array_equal(noisy, want.cpu().numpy().reshape(noisy.shape))
        p.add_noise = False
        plain = p.project_batch(proj)
        _, I2, _ = p.project_area_density(proj)
        assert np.array_equal(plain, np.asarray(I2, np.float32).reshape(plain.shape))
        np.testing.assert_allclose(plain, I.reshape(plain.shape), rtol=1e-5)
