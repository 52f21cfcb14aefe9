"""The batched frame quality where its tiles, borders and paths change: level sizes around the 64 x 16 tile,
levels of a few pixels (reflections that bounce), every gradient radius it takes and one that it leaves to the
single-frame kernels, two and more levels, 8 and 16 bits, rows that two pixels' loads fit and rows that they
do not.  Against the oracle, which holds the same whole numbers: double sums in another order, 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import torch  # noqa: F401

    import serstacker_amd as S

    S._lib.load()
    return S


CASES = [(16, 8, 8, 1, 1), (16, 8, 0, 1, 1), (5, 4, 0, 1, 1), (258, 130, 8, 1, 1), (256, 128, 0, 2, 1),
         (261, 66, 0, 3, 1), (250, 68, 11, 2, 2), (130, 190, 0, 1, 3), (24, 20, 8, 1, 4), (40, 36, 0, 4, 1),
         (64, 48, 9, 1, 0), (7, 300, 0, 1, 2)]


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
@pytest.mark.parametrize("w,h,colorid,kradius,dscale", CASES)
@pytest.mark.parametrize("pad,first", [(0, 0), (3, 1)])
def test_quality_of_a_batch(S, oracle32, dtype, w, h, colorid, kradius, dscale, pad, first):
    import torch
    from oracle import master

    r = np.random.default_rng(w * 5 + h + kradius)
    top = np.iinfo(dtype).max
    frames = [r.integers(0, top + 1, (h, w)).astype(dtype) for _ in range(3)]
    frames.append(np.full((h, w), top, dtype))
    big = torch.zeros((len(frames), h, w + pad), dtype=torch.int16 if dtype == np.uint16 else torch.uint8, device="cuda")
    views = []
    for i, f in enumerate(frames):
        t = torch.from_numpy(f.view(np.int16) if dtype == np.uint16 else f)
        big[i, :, first:first + w] = t.cuda()
        views.append(big[i, :, first:first + w])
    q = S.master_frame_quality(views, colorid, kradius, dscale)
    want = [master.frame_quality(oracle32, f, colorid, kradius, dscale) for f in frames]
    assert want[-1] == 0 and q[-1] == 0
    np.testing.assert_allclose(q, want, rtol=1e-12, atol=0)


def test_more_frames_than_a_launch(S, oracle32):
    import torch
    from oracle import master

    r = np.random.default_rng(3)
    frames = r.integers(0, 4096, (67, 40, 48)).astype(np.uint16)
    dev = torch.from_numpy(frames.view(np.int16)).cuda()
    q = S.master_frame_quality([dev[i] for i in range(67)], 8, 1, 2)
    np.testing.assert_allclose(q, [master.frame_quality(oracle32, f, 8, 1, 2) for f in frames], rtol=1e-12, atol=0)
