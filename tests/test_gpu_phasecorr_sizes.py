"""The phase correlation's half-plane transforms at the sizes where their plans change (4-point axes, one
pass of radix 4, radix 8 then 4, whole strips of 2 to 8 columns, 2 to 32 rows per block) and on the
sources their loads treat apart (odd sizes, odd pitches, unaligned rows), against the float64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ssg():
    import torch  # noqa: F401

    import serstacker_amd as S

    S._lib.load()
    return S


def frames_of(w, h, n, seed):
    """A smooth random scene cropped at whole-pixel offsets, with a little noise."""
    from scipy import ndimage

    r = np.random.default_rng(seed)
    m = 3
    scene = ndimage.gaussian_filter(r.normal(size=(h + 2 * m, w + 2 * m)), 1.0)
    scene /= scene.std()
    off = r.integers(-m, m + 1, (n, 2)) if min(w, h) > 16 else np.zeros((n, 2), int)
    return [(scene[m + dy:m + dy + h, m + dx:m + dx + w] + 0.01 * r.normal(size=(h, w))).astype(np.float32)
            for dx, dy in [(0, 0)] + [tuple(o) for o in off]]


# (width, height, binning, u16): padded axes of 4 .. 4096
SIZES = [(4, 4, 1, False), (4, 70, 1, False), (130, 5, 1, True), (9, 9, 2, False), (16, 33, 1, False),
         (31, 17, 1, True), (64, 64, 1, False), (127, 300, 2, True), (600, 257, 1, False), (1001, 77, 1, True),
         (75, 1025, 1, False), (2049, 40, 1, True), (40, 2049, 1, False), (4100, 66, 2, True), (8191, 9, 2, False)]


@pytest.mark.parametrize("w,h,binning,u16", SIZES)
def test_every_plan_matches_the_oracle(ssg, w, h, binning, u16):
    """0.002 px and 1e-5 of the peak, as for the sizes of the workloads: 32-bit transforms of up to 4096
    points (relative errors of a few 1e-7 of the spectrum) through a peak of sigma 1 px."""
    import torch
    from oracle import phasecorr as pc

    fr = frames_of(w, h, 4, seed=w * 7 + h)
    if u16:
        fr = [np.clip(np.rint(2000 + 400 * f), 0, 65535).astype(np.uint16) for f in fr]
    up = [torch.from_numpy(f.view(np.int16) if u16 else f).cuda() for f in fr]
    p = ssg.phase_correlation(w, h, binning)
    p.set_reference(up[0])
    out = p.estimate(up[1:])
    assert np.array_equal(out, p.estimate(up[1:]))
    spec = pc.spectrum(fr[0].astype(np.float64), binning)
    for f, o in zip(fr[1:], out):
        tx, ty, peak = pc.estimate(spec, f.astype(np.float64), binning)
        assert abs(o[2] - peak) < 1e-5, (o, peak)
        if min(w, h) // binning > 16:  # on a handful of pixels the surface has no single peak to agree on
            assert abs(o[0] - tx) < 2e-3 and abs(o[1] - ty) < 2e-3, (o, tx, ty)


@pytest.mark.parametrize("u16", [False, True])
@pytest.mark.parametrize("binning", [1, 2])
def test_unaligned_rows_give_the_aligned_rows_results(ssg, u16, binning):
    """Views whose rows start at an odd element or whose pitch is odd take the element loads: the same
    values, so the same results bit for bit; and a constant frame correlates to exactly zero."""
    import torch

    w, h = 118, 90
    fr = frames_of(w, h, 3, seed=5)
    if u16:
        fr = [np.rint(2000 + 400 * f).astype(np.uint16).view(np.int16) for f in fr]
    p = ssg.phase_correlation(w, h, binning)
    p.set_reference(torch.from_numpy(fr[0]).cuda())
    want = p.estimate([torch.from_numpy(f).cuda() for f in fr[1:]])
    for pitch, first in ((w + 10, 1), (w + 3, 0), (w + 3, 1)):
        views = []
        for f in fr[1:]:
            big = torch.zeros((h, pitch), dtype=torch.int16 if u16 else torch.float32, device="cuda")
            big[:, first:first + w] = torch.from_numpy(f).cuda()
            views.append(big[:, first:first + w])
        assert np.array_equal(p.estimate(views), want), (pitch, first)
    flat = torch.full((h, w), 7, dtype=torch.int16 if u16 else torch.float32, device="cuda")
    assert np.array_equal(p.estimate([flat]), np.zeros((1, 3)))


@pytest.mark.parametrize("w,h,n", [(33, 17, 131), (250, 250, 67), (129, 513, 20), (600, 70, 9)])
def test_any_number_of_frames_gives_the_single_frames_results(ssg, w, h, n):
    """More frames than a launch takes (64; the last of the even-sized chunks is shorter) and launches whose blocks hold
    4 to 32 rows by their number of frames: bit for bit the estimates of the frames one by one, also when a later call
    has fewer frames than the planes hold."""
    import torch

    fr = [torch.from_numpy(f).cuda() for f in frames_of(w, h, n, seed=n)]
    p = ssg.phase_correlation(w, h, 1)
    p.set_reference(fr[0])
    one = np.concatenate([p.estimate([f]) for f in fr[1:]])
    assert len({tuple(o) for o in one}) > n // 2
    for m in (n, n - 3, 5, n):
        assert np.array_equal(p.estimate(fr[1:1 + m]), one[:m]), m


def test_more_frames_than_a_grid_dimension(ssg):
    """70000 frames (a launch's second dimension ends at 65535): every result is its frame's own."""
    import torch

    w, h, n = 24, 20, 70000
    fr = [torch.from_numpy(f).cuda() for f in frames_of(w, h, 5, seed=3)]
    p = ssg.phase_correlation(w, h, 1)
    p.set_reference(fr[0])
    one = p.estimate(fr[1:])
    views = [ssg.image_view(f) for f in fr[1:]]
    at = np.arange(n) * 7 // 3 % len(views)
    assert np.array_equal(p.estimate(ssg._lib.images([views[k] for k in at])), one[at])
