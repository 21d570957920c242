"""The fast march at finer steps than the usual 0.1 mm and in cells of many
samples: long sums, where the additions' roundings show, along a boundary of two
labels, in constant and in textured tissue, in voxels of 20 mm.  Against the exact
march (bit for bit the transcription, test_gpu_forward.py), to the fast march's
bar: images within 1e-5."""
import ctypes as C

import numpy as np
import pytest

from deepdrr_amd import _abi, phantoms
from deepdrr_amd._abi_types import MARCH_EXACT, MARCH_FAST, Scene
from deepdrr_amd.volume import Volume
from tests import scenes
from tests.scenes import GpuRunner

pytestmark = pytest.mark.gpu


def _volume(name):
    n, spacing = (12, 20.0) if name == "coarse" else (100, 2.5)
    rng = np.random.default_rng(7)
    upper = np.zeros((n, n, n), bool)
    upper[n // 2:] = True
    labels = {"soft tissue": np.ones_like(upper)}
    if name == "constant":
        dens = np.full(upper.shape, 0.93)
    elif name in ("textured", "coarse"):
        dens = 1.0 + (0.05 if name == "textured" else 0.1) * rng.standard_normal(upper.shape)
    else:  # the beam runs along the boundary
        dens = np.where(upper, 1.9, 1.0) if name == "boundary" else np.full(upper.shape, 1.03)
        labels = {"soft tissue": ~upper, "bone": upper}
    return Volume.from_parameters(dens.astype(np.float32), labels, origin=phantoms._centered_origin((n,) * 3, (spacing,) * 3),
                                  spacing=(spacing,) * 3, anatomical_coordinate_system="LPS")


@pytest.mark.parametrize("name", ["constant", "textured", "boundary", "boundary_same", "coarse"])
def test_fine_steps(gpu, name):
    pixel = 0.7 if name.startswith("boundary") else 4.0
    case = scenes.make_case(name, [_volume(name)], phantoms.ap_device(64, 48, pixel, sdd=1020.0).get_camera_projection())
    r = GpuRunner(case)
    try:
        for step in (0.1, 0.05, 0.02, 0.01, 0.004):
            images = {}
            for march in (MARCH_EXACT, MARCH_FAST):
                sc = Scene(step=step, n_materials=case.scene.n_materials, attenuate_outside=0, air_index=0, march=march)
                _abi.call("drr_ctx_set_scene", r.ctx, C.byref(sc))
                images[march] = r.project()[0].astype(np.float64)
            err = np.abs(images[MARCH_FAST] / images[MARCH_EXACT] - 1).max()
            print(f"{name}, step {step}: {err:.2e}", flush=True)
            assert err <= 1e-5, step
    finally:
        r.close()
