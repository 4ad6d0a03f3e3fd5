"""The denoiser's 64-channel layers with their weights resident in LDS (images
or batches of more than 256 tiles of 8 x 32 at half resolution) against the
kernel that smaller calls take: a batch gives the bits of its images one by
one, at the tile counts around the rule and with partial last tile rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,h,w", [(8, 128, 256), (9, 128, 256), (9, 116, 256), (17, 64, 256),
                                    (33, 20, 448), (130, 8, 128)])
def test_batch_equals_single_images(cv, nb, h, w):
    """256, 288, 288 (a last row of 2 pixels), 272, 462 (10 rows a half image)
    and 260 tiles; a single image has at most 32."""
    print("%d x %d x %d" % (nb, h, w), flush=True)
    rng = np.random.default_rng(nb * 1000 + h)
    x = rng.normal(0.0, 1.0, (nb, h, w, 10)).astype(np.float32)
    d = cv.Denoiser(3)
    whole = d.forward(x)
    for k in (0, 1, nb // 2, nb - 1):
        one = d.forward(x[k:k + 1])
        assert one.tobytes() == whole[k:k + 1].tobytes(), k
    assert d.forward(x, materialize=True).tobytes() == whole.tobytes()


# (cin, cout) of the layers, the first one's ten channels padded to 16
NET = [(16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128), (192, 64), (64, 64),
       (96, 32), (32, 32), (32, 3)]


@pytest.mark.parametrize("h,few,many", [(16, 256, 512), (16, 64, 1024), (12, 256, 1024)])
def test_masked_input_gradients_equal(cv, h, few, many):
    """The input gradients of the 64-channel layers with the ReLU mask, in a
    training step of `few` images (of one tile at half resolution each: the
    other kernel) and of `many`, where only the first image is not black.
    With the biases zero a black image adds nothing to any weight gradient,
    the one tile of the first image is summed in the same order, and the
    loss's scale, 1 / the number of values, differs by a power of two: the
    gradients of the layers at half and quarter resolution are the same bits
    but for that power."""
    rng = np.random.default_rng(h + many)
    image = rng.normal(0.0, 1.0, (h, 64, 10)).astype(np.float32)
    target = np.abs(rng.normal(0.0, 1.0, (h, 64, 3))).astype(np.float32)
    grads = []
    for nb in (few, many):
        print("%d images of %d x 64" % (nb, h), flush=True)
        x, t = np.zeros((nb, h, 64, 10), np.float32), np.zeros((nb, h, 64, 3), np.float32)
        x[0], t[0] = image, target
        d = cv.Denoiser(7)
        d.train_step(x, t, 0.0)
        grads.append(d.grads() * np.float32(nb))
    off = 0
    for k, (cin, cout) in enumerate(NET):
        n = cout * 9 * cin
        a, b = (g[off:off + n] for g in grads)
        if 2 <= k <= 7:
            assert np.abs(a).max() > 0 and np.array_equal(a, b), k
        off += n + cout
