"""average_pyramid_inpaint at sizes whose blocks cover 2, 4 and 16 rows a thread: the counts of valid
pixels end the recursion, so a hole of one pixel in the last row or column has to be seen, and a mask
without holes has to be seen as full.  Bit for bit against the NumPy form."""
import numpy as np
import pytest

from oracle import finish as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,cn", [(515, 1025, 1), (1021, 1030, 3), (2051, 2101, 1)])
@pytest.mark.parametrize("hole", ["none", "corner", "disc"])
def test_large_levels_count_every_pixel(h, w, cn, hole):
    import torch  # noqa: F401

    import serstacker_amd as S

    rng = np.random.default_rng(h + w)
    img = rng.random((h, w, cn) if cn > 1 else (h, w)).astype(np.float32)
    mask = np.full((h, w), 255, np.uint8)
    if hole == "corner":
        mask[h - 1, w - 1] = 0
    elif hole == "disc":
        y, x = np.mgrid[:h, :w]
        mask[(x - w // 3) ** 2 + (y - h + 20) ** 2 < 90 ** 2] = 0
    want, want_mask = F.average_pyramid_inpaint(img, mask)
    got, got_mask = S.average_pyramid_inpaint(img, mask)
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(got_mask, want_mask)
