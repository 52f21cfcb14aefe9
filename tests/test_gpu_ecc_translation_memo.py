"""Translation iterations that step back to a quantised position they were at: the moments kept from
the first visit must give the step a pass over the image gives, and the rule that says when a
translation quantises alike for every pixel must hold."""
import numpy as np
import pytest
from scipy import ndimage

from tests import synth_np


@pytest.mark.parametrize("n", [16, 61, 1920, 4096, 8192])
def test_key_rule_quantises_every_pixel_alike(n):
    """fl(fl(x + t) * 32) rounds to 32 x + rint(32 t) for every pixel x whenever 32 t is farther from a
    rounding tie than (n + |t| + 2) 2^-18 (the device's rule, restated in float32)."""
    rng = np.random.default_rng(n)
    x = np.arange(n, dtype=np.float32)
    t = rng.uniform(-40, 40, 400).astype(np.float32)
    ties = (rng.integers(-900, 900, 400) + 0.5) / 32  # and translations a few steps beside a tie
    t = np.concatenate([t, (ties + rng.normal(0, 1, 400) * n * 2.0 ** -24).astype(np.float32),
                        np.float32([0.0, 1.0, -1.0, 1 / 64, -1 / 64, 0.015625 + 1e-6])])
    seen = 0
    for v in t:
        u = np.float32(32) * v
        r = np.rint(u)
        if not abs(u - r) < np.float32(0.5) - (np.float32(n) + abs(v) + np.float32(2)) * np.float32(2.0 ** -18):
            continue
        seen += 1
        q = np.rint((x + v) * np.float32(32)).astype(np.int64)
        assert np.array_equal(q, 32 * x.astype(np.int64) + int(r)), v
    assert seen > 300


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(61, 65), (120, 64), (333, 241)])
def test_every_step_is_the_step_of_its_position(oracle64, w, h):
    """The positions after budgets of 1 .. 40 iterations (a threshold that is never met, so the aligner
    walks between neighbouring positions): each next one is one FP64 oracle step from the last.  32-bit
    sums of about 30 roundings (2e-6 of the sum of magnitudes, which is a few pixels of step at the most)
    leave 1e-4 px."""
    import serstacker_amd as S
    import torch

    ref, frames, _ = synth_np.frames(3, w, h, radius=0.4 * min(w, h), seed=w, shift=2.0, rot_deg=0.3, noise=0.004)
    dev = [torch.from_numpy(np.ascontiguousarray(f)).cuda() for f in frames]
    path = [np.zeros((3, 2), np.float32)]
    for k in range(1, 41):
        reg = S.c_frame_registration(S.c_image_registration_options(
            motion_type=0, scale=1.0, eps=1e-7, ecch_max_level=1, max_iterations=k, input_smooth_sigma=0.0,
            reference_smooth_sigma=0.0, min_rho=0.0))
        assert reg.setup_reference_frame(np.ascontiguousarray(ref, dtype=np.float32))
        st = reg.register_batch(dev)
        assert all(s.iterations == k + 1 for s in st)
        path.append(np.array([[s.params[0], s.params[1]] for s in st], np.float32))
    revisits = 0
    for f in range(3):
        seen = set()
        for k in range(40):
            p, u = path[k][f], path[k][f].astype(np.float64) * 32
            revisits += tuple(np.rint(u)) in seen
            seen.add(tuple(np.rint(u)))
            if np.abs(np.abs(u - np.rint(u)) - 0.5).min() < (max(w, h) + 4) * 2.0 ** -18:
                continue  # the oracle's exact sum may round to the other side
            t = oracle64.xform(0, [float(p[0]), float(p[1])])
            oracle64.ecc_fa_align(ref.astype(np.float32), frames[f], t, max_iterations=1, max_eps=1e-7)
            assert np.abs(np.array(t.p[:2]) - path[k + 1][f]).max() < 1e-4, (f, k)
    assert revisits > 20


def _path(S, dev, ref, budgets, masks=None, ref_mask=None, step=1.5):
    """The frames' positions after each budget of iterations on one level, from a fresh handle each."""
    path = [np.zeros((len(dev), 2), np.float32)]
    for k in budgets:
        reg = S.c_frame_registration(S.c_image_registration_options(
            motion_type=0, scale=1.0, eps=1e-9, ecch_max_level=1, max_iterations=k, input_smooth_sigma=0.0,
            reference_smooth_sigma=0.0, min_rho=0.0, update_step_scale=step))
        assert reg.setup_reference_frame(ref, ref_mask)
        st = reg.register_batch(dev, masks)
        assert all(s.iterations == k + 1 for s in st)
        path.append(np.array([[s.params[0], s.params[1]] for s in st], np.float32))
    return path


def _check_steps(oracle64, path, ref, frames, masks=None, ref_mask=None, step=1.5):
    """Each position is one FP64 oracle step from the last, to 1e-4 px (see above); returns, per frame, the numbers of
    distinct quantised positions and of returns to one."""
    w, h = ref.shape[1], ref.shape[0]
    counts = []
    for f in range(len(frames)):
        seen, back = set(), 0
        for k in range(len(path) - 1):
            p, u = path[k][f], path[k][f].astype(np.float64) * 32
            back += tuple(np.rint(u)) in seen
            seen.add(tuple(np.rint(u)))
            if np.abs(np.abs(u - np.rint(u)) - 0.5).min() < (max(w, h) + 4) * 2.0 ** -18:
                continue  # the oracle's exact sum may round to the other side
            t = oracle64.xform(0, [float(p[0]), float(p[1])])
            oracle64.ecc_fa_align(ref, frames[f], t, ref_mask, masks[f] if masks else None, max_iterations=1,
                                  max_eps=1e-9, update_step_scale=step)
            assert np.abs(np.array(t.p[:2]) - path[k + 1][f]).max() < 1e-4, (f, k)
        counts.append((len(seen), back))
    return counts


@pytest.mark.gpu
def test_more_positions_than_are_kept(oracle64):
    """Small steps over several pixels pass more than the 64 positions whose moments a frame keeps, then walk between a
    few: the oldest are replaced, and what is taken again belongs to its position."""
    import serstacker_amd as S
    import torch

    w, h, step = 120, 100, 0.03
    r = np.random.default_rng(4)
    big = synth_np.blob_scene(w, h, 3, smin=6.0, smax=12.0)
    ref = big([[1, 0, 0], [0, 1, 0]]).astype(np.float32)
    frames = [(big([[1, 0, dx], [0, 1, dy]]) + r.normal(0, 0.002, (h, w))).astype(np.float32)
              for dx, dy in ((3.2, -2.1), (-2.7, 3.3))]
    dev = [torch.from_numpy(f).cuda() for f in frames]
    path = _path(S, dev, ref, range(1, 301), step=step)
    for seen, back in _check_steps(oracle64, path, ref, frames, step=step):
        assert seen > 64 and back > 20, (seen, back)


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["frame", "reference", "both"])
def test_kept_moments_with_masks(oracle64, which):
    import serstacker_amd as S
    import torch

    w, h = 120, 100
    ref, frames, _ = synth_np.frames(3, w, h, radius=0.4 * h, seed=8, shift=2.0, rot_deg=0.3, noise=0.004)
    ref = np.ascontiguousarray(ref, dtype=np.float32)
    r = np.random.default_rng(6)
    masks = ref_mask = None
    if which != "reference":
        masks = [np.where(r.random((h, w)) < 0.003, 0, 255).astype(np.uint8) for _ in frames]
        for m in masks:
            m[:9, 20:60] = 0
    if which != "frame":
        ref_mask = np.full((h, w), 255, np.uint8)
        ref_mask[40:60, 30:70] = 0
    dev = [torch.from_numpy(np.ascontiguousarray(f)).cuda() for f in frames]
    dm = [torch.from_numpy(m).cuda() for m in masks] if masks else None
    path = _path(S, dev, ref, range(1, 41), dm, ref_mask)
    # a level's masks are eroded 5x5 (ecc2.cc:1187-1234)
    erode = lambda m: ndimage.grey_erosion(m, size=(5, 5), mode="nearest")  # noqa: E731
    counts = _check_steps(oracle64, path, ref, frames, [erode(m) for m in masks] if masks else None,
                          erode(ref_mask) if ref_mask is not None else None)
    assert sum(back for _, back in counts) > 20, counts


@pytest.mark.gpu
@pytest.mark.parametrize("motion", [0, 3])
def test_levels_and_batches_share_nothing(motion):
    """Batches one after another on one handle (three levels, the second batch larger, the third the first again) give
    what handles of their own give."""
    import serstacker_amd as S
    import torch

    w, h = 200, 160
    ref, frames, _ = synth_np.frames(12, w, h, radius=0.4 * h, seed=9, shift=3.0, rot_deg=0.3, noise=0.004)
    dev = [torch.from_numpy(np.ascontiguousarray(f)).cuda() for f in frames]

    def handle():
        reg = S.c_frame_registration(S.c_image_registration_options(
            motion_type=motion, scale=1.0, eps=1e-7, ecch_max_level=3, max_iterations=40))
        assert reg.setup_reference_frame(np.ascontiguousarray(ref, dtype=np.float32))
        return reg

    def result(reg, batch):
        return [(bytes(bytearray(s.params)), s.rho, s.iterations, s.iterations_translation) for s in
                reg.register_batch(batch)]

    one = handle()
    for batch in (dev[:4], dev[3:12], dev[:4]):
        assert result(one, batch) == result(handle(), batch)


@pytest.mark.gpu
def test_profile_counts_the_bytes_of_passes_only():
    """register_frame ends a level's passes with its last active frame, so for one frame the pass launches are the
    passes; iterations solved from kept moments read no image."""
    import ctypes as C

    import serstacker_amd as S
    from serstacker_amd import _lib
    import torch

    w, h = 120, 100
    ref, frames, _ = synth_np.frames(1, w, h, radius=0.4 * h, seed=8, shift=2.0, rot_deg=0.3, noise=0.004)
    reg = S.c_frame_registration(S.c_image_registration_options(
        motion_type=0, scale=1.0, eps=1e-7, ecch_max_level=1, max_iterations=40, min_rho=0.0))
    assert reg.setup_reference_frame(np.ascontiguousarray(ref, dtype=np.float32))
    lib, prof = _lib.load(), _lib.Profile()
    lib.ssg_registration_set_profiling(reg._h, 1)
    assert reg.register_frame(torch.from_numpy(np.ascontiguousarray(frames[0])).cuda())
    lib.ssg_registration_get_profile(reg._h, C.byref(prof), 1)
    passes = prof.launches[_lib.PROF_ECC_MAIN]
    assert reg.status().iterations == 41 and 0 < passes < 30, passes
    assert prof.bytes[_lib.PROF_ECC_MAIN] == passes * 8.0 * w * h
