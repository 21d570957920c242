"""The Monte-Carlo kernel's schedule must not show in its results.

Which lanes run a block together depends on how many histories a launch has;
a history's own operations do not.  So a range of histories run in one launch
must give the flights and brick steps of the same range run in pieces, exactly,
and the same scores up to the order of the additions per pixel: m scores added
in two orders differ by at most 2 m 2^-24 times their sum, and m <= sum / 5 keV,
below which photons are absorbed.
"""
import ctypes as C

import numpy as np
import pytest

from deepdrr_amd import _abi, mc, phantoms
from deepdrr_amd import projector as P
from deepdrr_amd._abi_types import Scene
from deepdrr_amd.spectral_data import synthetic_120kv
from test_gpu_mc import _phantom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_hist, cuts", [
    (1, (0, 1)),
    (63, (0, 1, 63)),
    (64, (0, 33, 64)),
    (65, (0, 64, 65)),
    (257, (0, 100, 256, 257)),
    (5000, (0, 5, 2500, 4999, 5000)),
    (1 << 20, (0, 77, 300000, 1 << 20)),  # more than are resident at once
])
def test_histories_in_pieces(gpu, n_hist, cuts):
    vol = _phantom()
    mats = sorted(vol.materials[0].keys())
    dens, labs = P.volume_arrays(vol, mats)
    proj = phantoms.ap_device(32, 32, 4.0, sdd=600.0).get_camera_projection()
    p = mc.make_params(mats, synthetic_120kv(), proj, 600.0, vol.world_from_IJK.data,
                       max_density=float(dens.max()))
    ctx = C.c_void_p()
    _abi.call("drr_ctx_create", 0, C.byref(ctx))
    try:
        sc = Scene(step=0.1, n_materials=len(mats), attenuate_outside=0, air_index=0)
        _abi.call("drr_ctx_set_scene", ctx, C.byref(sc))
        h = C.c_void_p()
        nz, ny, nx = dens.shape
        _abi.call("drr_volume_create", ctx, dens.ctypes.data, labs.ctypes.data, nx, ny, nz, 0, C.byref(h))
        whole, parts = mc.MonteCarlo(ctx, h, p), mc.MonteCarlo(ctx, h, p)
        whole.run(n_hist, seed=99)
        for lo, hi in zip(cuts[:-1], cuts[1:]):
            parts.run(hi - lo, seed=99, first=lo)
        w, _, wsteps = whole.results()
        q, _, qsteps = parts.results()
        assert (wsteps, whole.brick_steps()) == (qsteps, parts.brick_steps())
        assert wsteps <= whole.brick_steps() or wsteps == 0
        w, q = w.astype(np.float64), q.astype(np.float64)
        assert np.all(np.abs(w - q) <= 2.0 * (w / 5.0) * 2.0**-24 * w + 1e-30)
        _abi.lib().drr_volume_destroy(h)
    finally:
        _abi.lib().drr_ctx_destroy(ctx)
