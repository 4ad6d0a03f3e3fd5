"""The denoiser beyond 2^32 input elements in one layer: the 96-channel layer at
full resolution gets there with 44.7 million pixels, where 32-bit offsets from
the tensor's start would wrap around to other pixels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_large_batch_equals_single_image(cv):
    """48 equal images of 1280 x 736 (45.2 million pixels): each has the bits of
    the image by itself."""
    h, w, nb = 736, 1280, 48
    x = np.random.default_rng(5).normal(0.0, 1.0, (1, h, w, 10)).astype(np.float32)
    one = cv.Denoiser(3).forward(x)[0]
    d = cv.Denoiser(3)
    print("batch of %d" % nb, flush=True)
    whole = d.forward(np.broadcast_to(x, (nb, h, w, 10)))
    differ = [k for k in range(nb) if not np.array_equal(whole[k].view(np.uint32),
                                                         one.view(np.uint32))]
    assert not differ


def test_large_image_equals_its_strip(cv):
    """One image of 6400 x 7168 (45.9 million pixels), whose 96-channel layer
    takes the general kernel: its last rows are those of a strip of it by
    itself, up to the order of the f32 sums.  That changes the rounding of some
    of that layer's bf16 outputs by one unit (2^-8 of the value), and with
    them the two layers behind it: 2^-7 in the 2-norm."""
    h, w, rows = 7168, 6400, 256
    block = np.random.default_rng(6).normal(0.0, 1.0, (rows, w, 10)).astype(np.float32)
    strip = cv.Denoiser(3).forward(block[None])[0]
    d = cv.Denoiser(3)
    print("%d x %d" % (w, h), flush=True)
    whole = d.forward(np.tile(block, (h // rows, 1, 1))[None])[0]
    # the strip's upper edge reaches 2 + 2 * 2 + 4 * 2 + 2 * 2 + 3 rows down,
    # rounded up to whole pixels of the lowest level
    a, b = whole[-(rows - 32):], strip[32:]
    assert np.linalg.norm(a - b) <= 2.0 ** -7 * np.linalg.norm(b)
