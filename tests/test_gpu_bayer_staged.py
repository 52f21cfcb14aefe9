"""The batched Bayer accumulate's staged tiles where their rule ends: rows that are multiples of 16 bytes,
of 4 bytes and of neither, partial tiles, every pattern, rotations that fit the staged rows and that do not, shifts past the frame, few frames,
whole-pixel shifts (zero weights), and more frames than a wave classifies at a time.  Bit for bit against
the FP32 oracle's per-frame sequence."""
import numpy as np
import pytest

from tests.test_gpu_bayer import _statuses, check_same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ssg():
    import torch  # noqa: F401

    import serstacker_amd as S

    S._lib.load()
    return S


def run(S, oracle32, w, h, n, u16, colorid, motion, params, pitch, first):
    import torch

    r = np.random.default_rng(w + 31 * n + colorid)
    raws = [r.integers(0, 4096, (h, w)).astype(np.uint16) for _ in range(n)]
    fl = [a.astype(np.float32) / np.float32(4096) for a in raws]
    views = []
    for a, b in zip(raws, fl):
        v = a.view(np.int16) if u16 else b
        big = torch.zeros((h, pitch), dtype=torch.int16 if u16 else torch.float32, device="cuda")
        big[:, first:first + w] = torch.from_numpy(v).cuda()
        views.append(big[:, first:first + w])
    sts = _statuses(S, params, motion)
    acc = S.c_bayer_average(w, h, colorid, bpp=12)
    acc.add_registered_batch(views, sts, motion)
    st = oracle32.bayer_state(w, h)
    for k in range(n):
        rmap = oracle32.create_map(oracle32.xform(motion, [np.float32(v) for v in params[k]]), w, h)
        _, mask = oracle32.base_remap(np.zeros((h, w), np.float32), rmap, interp=1, border=4)
        oracle32.bayer_accumulate(fl[k], st, colorid, rmap=rmap, mask=mask)
    check_same(S, acc, oracle32, st)


@pytest.mark.parametrize("u16", [True, False])
@pytest.mark.parametrize("pad,first", [(0, 0), (2, 0), (3, 1)])
@pytest.mark.parametrize("w,h", [(192, 80), (201, 83)])
def test_translation_rows_and_tiles(ssg, oracle32, u16, pad, first, w, h):
    pitch = (w + 7) // 8 * 8 + pad
    r = np.random.default_rng(w + pad)
    params = [[2 * r.integers(-4, 5) + r.uniform(-1, 1), 2 * r.integers(-4, 5) + r.uniform(-1, 1)] for _ in range(5)]
    params += [[0.0, 0.0], [1.0, -2.0], [3.0, 0.5]]
    run(ssg, oracle32, w, h, len(params), u16, 8, 0, params, pitch, first)


@pytest.mark.parametrize("colorid", [8, 9, 10, 11])
def test_patterns_and_frame_groups(ssg, oracle32, colorid):
    r = np.random.default_rng(colorid)
    params = [[r.uniform(-5, 5), r.uniform(-5, 5)] for _ in range(70)]
    run(ssg, oracle32, 144, 64, 70, True, colorid, 0, params, 144, 0)


@pytest.mark.parametrize("motion", [1, 3])
@pytest.mark.parametrize("deg", [0.5, 1.9, 2.6, 9.0, 179.0])
def test_rotations_in_and_out_of_the_box(ssg, oracle32, motion, deg):
    w, h = 208, 160
    params = []
    for s in (1, -1):
        a = np.deg2rad(deg * s)
        cx, cy = w / 2 + 0.3, h / 2 - 0.2
        tx, ty = cx - (np.cos(a) * cx - np.sin(a) * cy), cy - (np.sin(a) * cx + np.cos(a) * cy)
        params.append([tx, ty, a] if motion == 1 else
                      [np.cos(a) * 1.002, -np.sin(a), tx, np.sin(a), np.cos(a) * 0.998, ty])
    run(ssg, oracle32, w, h, 2, True, 9, motion, params, w, 0)


@pytest.mark.parametrize("u16", [True, False])
@pytest.mark.parametrize("motion", [1, 3])
@pytest.mark.parametrize("deg", [0.5, 1.9, 2.9, 3.4, 9.0, 179.0])
def test_rotations_of_enough_frames_for_the_staged_kernel(ssg, oracle32, u16, motion, deg):
    w, h = 208, 160
    params = []
    for k, s in enumerate((1, -1, 0.9, -0.8)):
        a = np.deg2rad(deg * s)
        cx, cy = w / 2 + 0.3 * k, h / 2 - 0.2
        tx, ty = cx - (np.cos(a) * cx - np.sin(a) * cy), cy - (np.sin(a) * cx + np.cos(a) * cy)
        params.append([tx, ty, a] if motion == 1 else
                      [np.cos(a) * 1.002, -np.sin(a), tx, np.sin(a), np.cos(a) * 0.998, ty])
    run(ssg, oracle32, w, h, 4, u16, 9, motion, params, w, 0)


@pytest.mark.parametrize("u16", [True, False])
def test_one_frame_out_of_the_box(ssg, oracle32, u16):
    """A rotation that does not fit sends its whole batch to the general kernel."""
    r = np.random.default_rng(12)
    params = [[r.uniform(-5, 5), r.uniform(-5, 5), np.deg2rad(d)] for d in (0.3, -0.5, 4.0, 2.9, 0.0)]
    run(ssg, oracle32, 208, 96, 5, u16, 8, 1, params, 208, 0)


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_few_frames(ssg, oracle32, n):
    params = [[1.5 * k - 2.25, 3.0 - 1.25 * k] for k in range(n)]
    run(ssg, oracle32, 201, 83, n, True, 10, 0, params, 208, 0)


@pytest.mark.parametrize("u16", [True, False])
def test_translations_beyond_tiles_and_frames(ssg, oracle32, u16):
    """Tiles that a shift moves wholly past an edge, and frames of which nothing is left."""
    w, h = 208, 83
    params = [[70.5, 0.25], [-70.5, 3.0], [2.0, 20.75], [-1.5, -20.75], [130.0, -40.5], [w + 3.5, 0.0],
              [-w - 3.5, 1.0], [0.5, h + 2.0], [0.0, -h - 2.5], [3e4, -3e4], [0.25, -0.75]]
    run(ssg, oracle32, w, h, len(params), u16, 11, 0, params, w, 0)
