"""A query that asks for no output has nothing to do: it returns at once, without
allocating for the rays, copying them or leaving a copy of them under way."""
import ctypes
import time

import numpy as np
import pytest

from convector_amd import scenes

pytestmark = pytest.mark.gpu


def test_query_without_outputs_copies_nothing(cv):
    g = cv.Scene.from_scene_data(scenes.config0(subdivisions=2))
    n = 1 << 24
    rays = np.zeros((n, 6), np.float32)
    rays[:, 5] = 1.0  # 403 MB, of which a copy takes 10 ms and more
    times = []
    for _ in range(3):
        t = time.perf_counter()
        cv.check(cv.lib().cv_bvh_intersect_nearest(
            g._h, rays.ctypes.data_as(ctypes.c_void_p), n, None, None, 0))
        times.append(time.perf_counter() - t)
    print("%d rays, no output: %r s" % (n, times), flush=True)
    assert min(times) < 1e-3
    # and the arguments are checked as ever
    assert cv.lib().cv_bvh_intersect_nearest(g._h, None, 5, None, None, 0) == 1
    assert cv.lib().cv_bvh_intersect_nearest(g._h, rays.ctypes.data_as(ctypes.c_void_p), 1 << 31,
                                             None, None, 0) == 1
