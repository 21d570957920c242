"""Views prepared together carry the numbers of views prepared one by one."""
import numpy as np
import pytest

from deepdrr_amd import geo, phantoms
from deepdrr_amd import projector as P
from deepdrr_amd._abi_types import view_to_dict


def _projections(n, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(n):
        K = geo.CameraIntrinsicTransform(np.array([[rng.uniform(500, 3000), 0, rng.uniform(50, 800)],
                                                   [0, rng.uniform(500, 3000), rng.uniform(50, 800)], [0, 0, 1]]))
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        E = np.eye(4)
        E[:3, :3] = q
        E[:3, 3] = rng.uniform(-1000, 1000, 3)
        # both a matrix to be inverted and one whose inverse is known
        T = geo.FrameTransform(E)
        out.append(geo.CameraProjection(K, T if k % 2 else T.inv))
    return out


@pytest.mark.parametrize("n, sdd", [(1, 1.0), (2, 1020.0), (9, 1.0)])
def test_cameras(n, sdd):
    projs = _projections(n, n)
    rows, centers = P.cameras(projs, sdd)
    for p, r, c in zip(projs, rows, centers):
        assert np.array_equal(r, P.world_from_index_rows(p, sdd))
        assert np.array_equal(c, np.array(p.center_in_world))


@pytest.mark.parametrize("which", [None, [1, 0, 1, 1, 0]])
def test_views(which):
    vols = [phantoms.uniform_volume((4, 5, 6)), phantoms.uniform_volume((3, 3, 7))]
    projs = _projections(5, 7)
    views = P.build_views(vols, [1, 0], projs, 4000.0, 900.0, which=which)
    for i, (v, p) in enumerate(zip(views, projs)):
        ks = [0, 1] if which is None else [which[i]]
        params = [P.volume_view_params(vols[k], p, [1, 0][k]) for k in ks]
        want = P.make_view(P.world_from_index_rows(p, 900.0), *p.intrinsic.sensor_size, 4000.0, params)
        a, b = view_to_dict(v), view_to_dict(want)
        assert bytes(v) == bytes(want), (a, b)
