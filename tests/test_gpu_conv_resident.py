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
