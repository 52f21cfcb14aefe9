"""ECC passes over levels whose last row of 64-row tiles holds only some of its four 16-row strips: the
strips below the level and the halo rows past its last row are left out, which must not change a step."""
import numpy as np
import pytest

from tests import synth_np

START = {0: [0, 0], 1: [0, 0, 0], 2: [0, 0, 0, 1], 3: [1, 0, 0, 0, 1, 0]}


def one_step(oracle64, motion, w, h):
    """One iteration against the FP64 oracle's.  32-bit sums leave 2e-6 of the moments and the scaled
    Hessian of these images has a condition below 100: 2e-4 of a step of up to 4 px at a corner."""
    import serstacker_amd as S
    import torch

    ref, frames, _ = synth_np.frames(2, w, h, radius=0.4 * min(w, h), seed=h, shift=1.0, rot_deg=0.3, noise=0.004)
    reg = S.c_frame_registration(S.c_image_registration_options(
        motion_type=motion, scale=1.0, eps=1e-7, ecch_max_level=1, max_iterations=1, input_smooth_sigma=0.0,
        reference_smooth_sigma=0.0, min_rho=0.0, ecch_estimate_translation_first=False))
    assert reg.setup_reference_frame(np.ascontiguousarray(ref, dtype=np.float32))
    got = reg.register_batch([torch.from_numpy(np.ascontiguousarray(f)).cuda() for f in frames])
    corners = np.array([[x, y] for x in (0, w - 1) for y in (0, h - 1)], np.float64)

    def at(p):
        p = np.asarray(p, np.float64)
        x, y = corners.T
        if motion == 0:
            return np.stack([x + p[0], y + p[1]])
        if motion == 3:
            return np.stack([p[0] * x + p[1] * y + p[2], p[3] * x + p[4] * y + p[5]])
        s, c, sn = (p[3] if motion == 2 else 1.0), np.cos(p[2]), np.sin(p[2])
        return np.stack([s * (c * x - sn * y) + p[0], s * (sn * x + c * y) + p[1]])

    n = len(START[motion])
    for f in range(2):
        t = oracle64.xform(motion, [float(v) for v in START[motion]])
        oracle64.ecc_fa_align(ref.astype(np.float32), frames[f], t, max_iterations=1, max_eps=1e-7)
        assert np.abs(at(t.p[:n]) - at(got[f].params[:n])).max() < 8e-4, (f, list(t.p[:n]), list(got[f].params[:n]))


@pytest.mark.gpu
@pytest.mark.parametrize("h", [33, 64, 65, 80, 81, 96, 111, 113, 127, 129])
@pytest.mark.parametrize("motion", [0, 1, 2, 3])
def test_one_step_of_every_last_tile_height(oracle64, motion, h):
    one_step(oracle64, motion, 91, h)


@pytest.mark.gpu
@pytest.mark.parametrize("tx,ty", [(1, 1), (5, 1), (8, 4), (11, 3), (12, 3), (16, 8), (19, 7), (21, 7)])
@pytest.mark.parametrize("motion", [0, 3])
def test_one_step_of_every_count_of_tiles(oracle64, motion, tx, ty):
    """The four waves of the solve sum 1 .. 37 tiles each: one load batch, its remainder, and both."""
    one_step(oracle64, motion, 60 * tx, 64 * ty)
