"""What view preparation takes: any iterable of cameras, fewer volume indices than
cameras (the shorter list is rendered)."""
import numpy as np
import pytest

from deepdrr_amd import autograd, phantoms
from deepdrr_amd import projector as P
from tests.test_cpu_views import _projections


@pytest.mark.parametrize("which", [[1, 0], [1], np.array([0, 1])])
def test_fewer_indices_than_cameras(which):
    vols = [phantoms.uniform_volume((4, 5, 6)), phantoms.uniform_volume((3, 3, 7))]
    projs = _projections(4, 3)
    views = P.build_views(vols, [1, 0], projs, 4000.0, 900.0, which=which)
    want = P.build_views(vols, [1, 0], projs[:len(which)], 4000.0, 900.0, which=which)
    assert len(views) == len(which) and [bytes(v) for v in views] == [bytes(v) for v in want]


def _object_array(projs):
    a = np.empty(len(projs), object)
    a[:] = projs
    return a


@pytest.mark.parametrize("form", [tuple, iter, _object_array], ids=["tuple", "iterator", "array"])
def test_iterables_of_cameras(form):
    vols = [phantoms.uniform_volume((4, 5, 6))]
    projs = _projections(3, 5)
    want = P.build_views(vols, [0], projs, 4000.0, 900.0)
    assert [bytes(v) for v in P.build_views(vols, [0], form(projs), 4000.0, 900.0)] == [bytes(v) for v in want]
    g = autograd.PoseGeometry((4, 5, 6), np.eye(4))
    a, b = (g.views(f, np.zeros(6)) for f in (projs, form(projs)))
    assert len(b) == 3 and [bytes(v) for v, _ in a] == [bytes(v) for v, _ in b]
    assert all(np.array_equal(s, t) for (_, s), (_, t) in zip(a, b))


def test_no_cameras():
    assert P.build_views([phantoms.uniform_volume((4, 5, 6))], [0], iter([]), 4000.0) == []
    assert autograd.PoseGeometry((4, 5, 6), np.eye(4)).views(iter([]), np.zeros(6)) == []
