"""The rule that sends a Bayer batch to the staged kernel (bayer_box_fits, host code): wherever it accepts a map, every
tap of every tile's pixels lies in the box that the kernel stages, restated here in NumPy with the device's 32-bit
positions; what it must accept (translations, small rotations) and refuse (large ones, NaN, positions beyond 32-bit
accuracy) is accepted and refused."""
import ctypes as C
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "serstacker_amd", "libssg.so")
TW, TH, SH = 64, 16, 21
F = np.float32


@pytest.fixture(scope="module")
def fits():
    f = C.CDLL(LIB)["_ZN3ssg14bayer_box_fitsEiRKNS_7MapCoefEiibi"]
    f.restype = C.c_bool
    f.argtypes = [C.c_int, C.POINTER(C.c_float * 8), C.c_int, C.c_int, C.c_bool, C.c_int]
    return lambda motion, c, w, h, u16, unit: f(motion, (C.c_float * 8)(*c), w, h, u16, unit)


def fma(a, b, c):  # the 64-bit product of two floats is exact; its sum is rounded twice, by less than the rule allows for
    return F(np.asarray(a, np.float64) * np.asarray(b, np.float64) + np.asarray(c, np.float64))


def positions(motion, c, x, y):
    c = [F(v) for v in c]
    fx, fy = F(x), F(y)
    if motion == 0:
        return fx + c[0], fy + c[1]
    if motion == 3:
        return fma(c[1], fy, c[0] * fx) + c[2], fma(c[4], fy, c[3] * fx) + c[5]
    return fma(c[2], fma(c[1], fx, -(c[0] * fy)), c[3]), fma(c[2], fma(c[0], fx, c[1] * fy), c[4])


def boxes_hold(motion, c, w, h, u16, unit):
    """Over all tiles that are not outside the frame."""
    per = unit // (2 if u16 else 4)
    spr = (TW + 4 + per - 1) // per + 1
    for y0 in range(0, h, TH):
        for x0 in range(0, w, TW):
            x1, y1 = min(x0 + TW - 1, w - 1), min(y0 + TH - 1, h - 1)
            cx, cy = positions(motion, c, np.array([x0, x1, x0, x1]), np.array([y0, y0, y1, y1]))
            if np.isnan(cx).any() or np.isnan(cy).any() or not (
                    cx.max() > -1 and cy.max() > -1 and cx.min() < w and cy.min() < h):
                continue
            ix = int(np.floor(cx.min() - F(0.25)))
            bx, by = ix - ix % per, int(np.floor(cy.min() - F(0.25)))
            xs, ys = np.meshgrid(np.arange(x0, x1 + 1), np.arange(y0, y1 + 1))
            px, py = positions(motion, c, xs, ys)
            sx, sy = np.trunc(px), np.trunc(py)
            # the mask drops positions that quantise (1/32 px) to outside the frame
            taken = (px >= -1 / 64) & (sx < w - 1) & (py >= -1 / 64) & (sy < h - 1)
            if not taken.any():
                continue
            sx, sy = sx[taken], sy[taken]
            if sx.min() < bx or sx.max() + 1 >= bx + spr * per or sy.min() < by or sy.max() + 1 >= by + SH:
                return False
    return True


UNITS = [(True, 16), (False, 16), (True, 4), (False, 4)]


@pytest.mark.parametrize("u16,unit", UNITS)
def test_accepted_maps_stay_in_the_box(fits, u16, unit):
    r = np.random.default_rng(unit + u16)
    accepted = refused = 0
    for k in range(400):
        motion = int(r.integers(0, 4))
        w, h = int(r.integers(3, 700)), int(r.integers(3, 400))
        far = r.choice([1, 1, 1, 30000])
        tx, ty = r.uniform(-20, 20, 2) * far
        a = np.deg2rad(r.choice([0, 1, -1]) * r.uniform(0, 5) + r.choice([0, 0, 0, 180]))
        s = r.choice([1.0, r.uniform(0.9, 1.1)])
        if motion == 0:
            c = [tx, ty, 0, 0, 0, 0, 0, 0]
        elif motion == 3:
            c = [s * np.cos(a), -np.sin(a), tx, np.sin(a), np.cos(a) / s, ty, 0, 0]
        else:
            c = [np.sin(a), np.cos(a), s if motion == 2 else 1, tx, ty, 0, 0, 0]
        if fits(motion, c, w, h, u16, unit):
            accepted += 1
            assert boxes_hold(motion, c, w, h, u16, unit), (motion, c, w, h)
        else:
            refused += 1
    assert accepted > 100 and refused > 40


@pytest.mark.parametrize("u16,unit", UNITS)
def test_edges_of_the_rule(fits, u16, unit):
    w, h = 4096, 3000

    def turned(deg, motion=1, s=1.0):
        a = np.deg2rad(deg)
        return [np.sin(a), np.cos(a), s, 5.0, -3.0, 0, 0, 0]

    assert fits(0, [1000.5, -2000.25, 0, 0, 0, 0, 0, 0], w, h, u16, unit)
    assert fits(1, turned(2.9), w, h, u16, unit) and fits(1, turned(-2.9), w, h, u16, unit)
    assert boxes_hold(1, turned(2.9), 512, 256, u16, unit)
    assert fits(2, turned(0.5, 2, 1.02), w, h, u16, unit)
    assert not fits(1, turned(3.6), w, h, u16, unit) and not fits(2, turned(0, 2, 1.3), w, h, u16, unit)
    assert not fits(0, [float("nan"), 0, 0, 0, 0, 0, 0, 0], w, h, u16, unit)
    assert not fits(0, [3e5, 0, 0, 0, 0, 0, 0, 0], w, h, u16, unit)
    assert not fits(3, [1, 0, float("inf"), 0, 1, 0, 0, 0], w, h, u16, unit)
    assert not fits(1, [0, 1, 1, 0, 0, 100, 100, 0], w, h, u16, unit)
