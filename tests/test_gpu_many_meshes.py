"""A scene of many meshes, empty ones and one with many triangles among them, is
the scene of one mesh that holds all their triangles: the same tree, source
ids, materials and texture coordinates."""
import numpy as np
import pytest

from convector_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cuts", [[0, 0, 1, 2, 2, 70001, 70050, 90000], list(range(0, 90001, 37))])
def test_many_meshes_equal_one(cv, cuts):
    n = 90000
    t, m = scenes.free_triangles(scenes.Stream(31), n)
    t, uv = np.asarray(t, np.float32), np.arange(6 * n, dtype=np.float32).reshape(n, 6) / n
    cuts = [0] + cuts + [n]
    one = cv.Scene.from_meshes([cv.Mesh.from_triangles(t, m, uv)])
    many = cv.Scene.from_meshes([cv.Mesh.from_triangles(t[a:b], m[a:b], uv[a:b])
                                 for a, b in zip(cuts, cuts[1:])])
    for a, b in zip(one.bvh(), many.bvh()):
        assert a.tobytes() == b.tobytes()
    rays = scenes.rays_inward(20000, 32, radius=2.0, target_scale=0.9)
    for a, b in zip(one.intersect_nearest(rays, full=True), many.intersect_nearest(rays, full=True)):
        assert a.tobytes() == b.tobytes()
    assert (one.intersect_nearest(rays)["tri_id"] != 0xFFFFFFFF).any()
