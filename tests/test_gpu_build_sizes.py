"""The GPU build at the triangle counts where it changes kernels: the small
subtrees (up to half the bins), a wave and a workgroup per node, the level
phase, and chunked nodes with one more reference than a chunk -- over free
triangles, over clusters whose centroid bins fall back to sorted ones on every
axis, and over coordinates with many ties.  The tree is the oracle's, byte for
byte."""
import numpy as np
import pytest

from convector_amd import scenes

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 8, 9, 16, 17, 31, 32, 33, 63, 64, 65, 255, 256, 257, 258, 1023, 1024, 1025, 1026,
         2049, 4095, 4096, 4097, 4609, 9000]


def _tris(kind, n, seed):
    t, m = scenes.free_triangles(scenes.Stream(seed), n)
    if kind == "clusters":
        # most triangles in small balls far apart: one bin above n / 8
        c = scenes.Stream(seed + 1).uniform(3 * 5, -50.0, 50.0).reshape(5, 3)
        k = (scenes.Stream(seed + 2).u64(n) % np.uint64(5)).astype(np.int64)
        t = t * 0.01 + np.tile(c[k], (1, 3))
    elif kind == "ties":
        # congruent triangles at the points of a coarse grid
        t = np.tile(np.round(t[:, 0:3] * 4.0) / 4.0, (1, 3)) + [0.0, 0.0, 0.0, 0.25, 0.0, 0.0, 0.0,
                                                                0.25, 0.125]
    return t.astype(np.float32), m


@pytest.mark.parametrize("bins", [64, 32, 16])
@pytest.mark.parametrize("kind", ["free", "clusters", "ties"])
def test_build_sizes_equal_oracle(cv, oracle, kind, bins):
    for n in SIZES:
        t, m = _tris(kind, n, 1000 + n)
        print("%s, %d triangles, %d bins" % (kind, n, bins), flush=True)
        st, on, oo, (ratio, per_leaf) = oracle.bvh_build(t, bins)
        mesh = cv.Mesh.from_triangles(t, m)
        if st != 0:
            with pytest.raises(cv.CvError):
                cv.Scene.from_meshes([mesh], bins=bins)
            continue
        g = cv.Scene.from_meshes([mesh], bins=bins)
        gn, go = g.bvh()
        info = g.bvh_info()
        assert len(gn) == len(on) and gn.tobytes() == on.tobytes(), (kind, n)
        assert (go == oo).all(), (kind, n)
        assert info["avg_tris_per_leaf"] == np.float32(per_leaf), (kind, n)
        assert info["avg_area_ratio"] == np.float32(ratio), (kind, n)
