"""A camera that says itself where it stands and looks (a subclass, or another
class with the same properties) is asked, among others whose matrices are inverted
together."""
import types

import numpy as np
import pytest

from deepdrr_amd import autograd, geo, phantoms
from deepdrr_amd import projector as P
from tests.test_cpu_views import _projections


class Shifted(geo.CameraProjection):
    """A camera with a shifted focal spot and a scaled ray map."""

    @property
    def center_in_world(self):
        return geo.point(np.array(super().center_in_world) + [1.0, -2.0, 0.5])

    @property
    def world_from_index(self):
        return geo.Transform(1.25 * super().world_from_index.data)


def _stand_in(p):
    """The properties a view reads, and nothing else."""
    return types.SimpleNamespace(intrinsic=types.SimpleNamespace(sensor_size=p.intrinsic.sensor_size),
                                 world_from_index=p.world_from_index, center_in_world=p.center_in_world)


class KnownInverse(geo.FrameTransform):
    """A pose that gives its own inverse."""

    @property
    def inv(self):
        m = np.eye(4)
        m[:3, 3] = [3.0, 2.0, 1.0]
        return geo.FrameTransform(m)


@pytest.mark.parametrize("sdd", [1.0, 900.0])
def test_overridden_cameras(sdd):
    a, b, c, d = _projections(4, 11)
    cams = [a, Shifted(b.intrinsic, b.extrinsic), _stand_in(c), geo.CameraProjection(d.intrinsic, KnownInverse(np.eye(4))), d]
    vols = [phantoms.uniform_volume((4, 5, 6))]
    for p, view in zip(cams, P.build_views(vols, [0], cams, 4000.0, sdd)):
        want = P.make_view(P.world_from_index_rows(p, sdd), *p.intrinsic.sensor_size, 4000.0,
                           [P.volume_view_params(vols[0], p, 0)])
        assert bytes(view) == bytes(want)
    g = autograd.PoseGeometry((4, 5, 6), np.eye(4))
    for p, (view, src) in zip(cams, g.views(cams, np.zeros(6))):
        assert np.array_equal(src, np.array(p.center_in_world).astype(np.float32))
        assert np.array_equal(np.array(view.world_from_index[:], np.float32), P.world_from_index_rows(p, 1.0).reshape(-1))
