"""Short queues dealt out to the traversal's waves beforehand (no cursor):
every ray is traversed once and gives the oracle's hit at the sizes where the
dealing changes shape -- fewer rays than the smallest share, one more than a
share or a stripe of 64 rays per wave, the last dealt size and the first that
goes through the cursors (2 rays per lane of the resident waves, 8 where 24
waves per CU are).  (The grids are all multiples of the 8 XCDs on a
device of 256 CUs; test_deal_map.py has the others.)"""
import numpy as np
import pytest

from convector_amd import scenes
from helpers import check_tolerance
from test_gpu_traversal import _check_exact

pytestmark = pytest.mark.gpu

LANES = 256 * 64  # one wave per CU


@pytest.mark.parametrize("block_waves", [1, 2, 4])
@pytest.mark.parametrize("waves_per_cu", [1, 3])
def test_dealt_queries_equal_oracle(cv, oracle, block_waves, waves_per_cu):
    sd = scenes.config0(subdivisions=2)
    g = cv.Scene.from_scene_data(sd)
    o = oracle.Scene.from_scene_data(sd)
    g.set_tuning(extend_waves_per_cu=waves_per_cu, block_waves=block_waves)
    lanes = LANES * waves_per_cu
    rays = scenes.rays_inward(4 * lanes + 1, 7, radius=0.9, target_scale=0.6)
    ref = o.intersect(rays)
    for n in (1, 3, 4, 5, 63, 65, 4096, 4097, lanes - 1, lanes, lanes + 1, lanes + 4097,
              2 * lanes, 2 * lanes + 1, 4 * lanes - 63, 4 * lanes, 4 * lanes + 1):
        print("%d rays, %d waves per CU, %d per block" % (n, waves_per_cu, block_waves), flush=True)
        hits = g.intersect_nearest(rays[:n])
        assert (hits["tri_id"] == ref["tri"][:n]).all(), n
        assert (hits["t"].view(np.uint32) == ref["tuv"][:n, 0].copy().view(np.uint32)).all(), n


@pytest.mark.parametrize("tuning,waves,rays", [
    ({}, 24, 8), ({"stack_entries": 16}, 20, 2), ({"stack_entries": 32, "block_waves": 4}, 8, 2),
    ({"bvh_width": 8}, None, 2)])
def test_dealt_queries_by_residency(cv, oracle, tuning, waves, rays):
    """The last dealt size and the first from the cursors for launch shapes that
    keep all 24 waves per CU resident and ones that do not."""
    sd = scenes.config0(subdivisions=2)
    g = cv.Scene.from_scene_data(sd)
    g.set_tuning(**tuning)
    last = (waves or 16) * LANES * rays
    r = scenes.rays_inward(last + 1, 8, radius=0.9, target_scale=0.6)
    ref = oracle.Scene.from_scene_data(sd).intersect(r)
    for n in (last - 1, last, last + 1):
        print("%d rays, %r" % (n, tuning), flush=True)
        hits = g.intersect_nearest(r[:n])
        if "bvh_width" in tuning:
            check_tolerance(sd, hits, {k: v[:n] for k, v in ref.items()}, r[:n])
        else:
            assert (hits["tri_id"] == ref["tri"][:n]).all()
            assert (hits["t"].view(np.uint32) == ref["tuv"][:n, 0].copy().view(np.uint32)).all()


@pytest.mark.parametrize("w,h", [(16, 4), (128, 124), (128, 128), (128, 132)])
def test_dealt_frames_equal_oracle(cv, oracle, w, h):
    """Bounces below, at and above one ray per lane of a one-wave-per-CU
    launch (16,384 paths)."""
    print("%dx%d" % (w, h), flush=True)
    sd = scenes.config0(subdivisions=2)
    g = cv.Scene.from_scene_data(sd)
    o = oracle.Scene.from_scene_data(sd)
    g.set_tuning(extend_waves_per_cu=1)
    r = cv.Renderer(g, w, h)
    hdr = r.new_buffer_f32()
    r.accumulate_frames_f32(hdr, 1, 1)
    ohdr, _ = o.accumulate_frames(w, h, 1, 1, oracle.RNG_PIXEL, 4)
    assert hdr.tobytes() == ohdr.tobytes()


@pytest.mark.parametrize("waves_per_cu", [1, 32])
@pytest.mark.parametrize("tuning", [{}, {"refill_threshold": 65, "queue_parts": 1},
                                    {"bvh_width": 4, "block_waves": 4}])
def test_records_equal_oracle(cv, oracle, tuning, waves_per_cu):
    """Full records, dealt out and through the cursors, under tunings of the
    hits-only query: every field the oracle's, the counters of the
    reference's tree whatever width the hits are traversed with."""
    sd = scenes.config0(subdivisions=2)
    g = cv.Scene.from_scene_data(sd)
    o = oracle.Scene.from_scene_data(sd)
    g.set_tuning(extend_waves_per_cu=waves_per_cu, **tuning)
    rays = scenes.rays_inward(4 * LANES + 65, 9, radius=0.9, target_scale=0.6)
    ref = o.intersect(rays, isect=True)
    for n in (1, 63, 65, LANES + 1, 4 * LANES, 4 * LANES + 65):
        print("%d rays, %d waves per CU, %r" % (n, waves_per_cu, tuning), flush=True)
        hits, rec = g.intersect_nearest(rays[:n], full=True)
        assert (hits["tri_id"] == rec["tri_id"]).all()
        _check_exact(hits, rec, {k: v[:n] for k, v in ref.items()})
        assert (rec["reserved"] == 0).all()


@pytest.mark.parametrize("stack", [8, 16, 24, 32])
@pytest.mark.parametrize("leaves", [None, 40])
def test_records_around_one_ray_per_lane(cv, oracle, stack, leaves):
    """Full records at the last dealt size and the first that goes through the
    cursors, for every stack size, on the built tree and on an imported one of
    two leaves of more triangles than a packed stack entry counts."""
    if leaves:
        t, m = scenes.free_triangles(scenes.Stream(5), 100)
        sd = scenes.SceneData(tris=np.asarray(t, np.float32), materials=m)
        nodes = np.zeros(2, cv.NODE_DTYPE)
        for k, (a, b) in enumerate([(0, leaves), (leaves, 100)]):
            v = sd.tris[a:b].reshape(-1, 3)
            nodes[k] = (v.min(0), v.max(0), a, b - a)
        g = cv.Scene.from_scene_data(sd, with_bvh=(nodes, np.arange(100, dtype=np.uint32)))
        assert g.bvh_info()["max_leaf"] == 60
    else:
        sd = scenes.config0(subdivisions=2)
        g = cv.Scene.from_scene_data(sd)
    g.set_tuning(extend_waves_per_cu=1, stack_entries=stack)
    rays = scenes.rays_inward(LANES + 65, 19, radius=0.9, target_scale=0.6)
    ref = oracle.Scene.from_scene_data(sd).intersect(rays, isect=True)
    for n in (LANES - 1, LANES, LANES + 1, LANES + 65):
        print("%d rays, stack %d, leaves %r" % (n, stack, leaves), flush=True)
        hits, rec = g.intersect_nearest(rays[:n], full=True)
        part = {k: v[:n] for k, v in ref.items()}
        if leaves:  # the counters are the imported tree's
            assert (hits["tri_id"] == part["tri"]).all()
            assert (hits["t"].view(np.uint32) == part["tuv"][:, 0].copy().view(np.uint32)).all()
            assert set(np.unique(rec["numi_aabb"])) == {2} and rec["numi_tri"].max() == 100
        else:
            _check_exact(hits, rec, part)
        assert (hits["tri_id"] == rec["tri_id"]).all()
