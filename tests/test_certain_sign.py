"""The PIP test's certain-sign rule, checked on the CPU (tests/cpp/certain_sign_check.c).

The HIP test decides a (point, edge) from the scaled line form only when
|t| > 2^-48 s + 2^-1000; the checker draws adversarial (point, edge) pairs (points
on, beside and along segments, nearly vertical and horizontal edges, shared
coordinates, subnormal to 2^120 scales) and compares every certain decision with
the reference's rounded lhs < rhs and its 4-ULP collinearity test. The same file
built with a smaller tolerance, or with the lower limit on the edge's size
removed, finds counterexamples: the check has the power to fail.
"""

import os
import shutil
import subprocess

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "certain_sign_check.c")


def build(tmp_path, name, *defines):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    exe = str(tmp_path / name)
    subprocess.run([cc, "-O2", "-ffp-contract=off", *defines, SRC, "-o", exe, "-lm"],
                   check=True, capture_output=True)
    return exe


def run(exe, iters, seed):
    r = subprocess.run([exe, str(iters), str(seed)], capture_output=True, text=True)
    counts = dict(zip(r.stdout.split()[-8::2], map(int, r.stdout.split()[-7::2])))
    return r.returncode, counts, r.stdout


def test_certain_decisions_match_the_reference(tmp_path):
    exe = build(tmp_path, "csc")
    for seed in (1, 2, 3):
        rc, counts, out = run(exe, 3_000_000, seed)
        assert rc == 0 and counts["bad"] == 0, out
        assert counts["certain"] > 500_000 and counts["no_line"] > 0, out


@pytest.mark.parametrize("define", ["-DTOL_SCALE=0x1p-53", "-DN_MIN=0x1p-1074"])
def test_weaker_rules_fail(tmp_path, define):
    exe = build(tmp_path, "csc_weak", define)
    rc, counts, out = run(exe, 3_000_000, 1)
    assert rc == 1 and counts["bad"] > 0, out


def _high_as_float(v):
    return (np.asarray(v, np.float64).view(np.uint64) >> np.uint64(32)).astype(np.uint32).view(
        np.float32)


def test_sign_words_equal_comparisons():
    """The edge step's words against the comparisons they stand for, over signed zeros,
    subnormals, neighbours and 900 powers of two: the sign bit of (py + 0) - ay is ay > py, and a
    high word of |t| above tol's (as floats, NaN never above) implies |t| > tol."""
    rng = np.random.default_rng(3)
    base = np.concatenate([[0.0, -0.0, 5e-324, -5e-324, 2.0**-1022, 1e300, -1e300],
                           rng.normal(size=400) * 2.0 ** rng.integers(-500, 400, 400)])
    a = np.concatenate([base, np.nextafter(base, np.inf), np.nextafter(base, -np.inf)])
    for shift in (0, 1, 7, 401):
        p = np.roll(a, shift)
        assert np.array_equal(np.signbit((p + 0.0) - a), a > p)
    t = np.concatenate([a, [np.nan, np.inf, -np.inf]])
    for tol in (2.0**-1000, 2.0**-48, 1.0, 1e100, np.inf):
        with np.errstate(invalid="ignore"):
            above = np.abs(_high_as_float(t)) > _high_as_float([tol])[0]
        assert np.all(np.abs(t[above]) > tol)
        finite = np.nan_to_num(t, nan=0, posinf=0, neginf=0)
        assert above[np.abs(finite) > 1.001 * tol].all()


@pytest.mark.parametrize("exponent", [-50, 0, 50])
@pytest.mark.parametrize("offset", [0.0, 1e3])
def test_single_precision_ring_line_is_certain(exponent, offset):
    """The locator's float32 form of a short ring: wherever it vouches for its outcome
    (vertices off the point's y by more than 2^-21 s, every |lhs - rhs| above 2^-19 s^2),
    the reference's FP64 arithmetic gives the same side and no collinearity filter.
    Points at random, on vertices and edges, and a few ulps beside them."""
    rng = np.random.default_rng(exponent + 77)
    f32 = np.float32
    sure = total = 0
    for ne in (3, 4, 6, 7, 8, 13):
        for _ in range(15):
            ang = np.sort(rng.uniform(0, 2 * np.pi, ne))
            r = rng.uniform(0.3, 1.0, ne)
            scale = 2.0**exponent
            ax = (offset + r * np.cos(ang)) * scale
            ay = (offset + np.round(r * np.sin(ang), 2)) * scale
            bx, by = np.roll(ax, 1), np.roll(ay, 1)  # an edge's b: the vertex before
            k = rng.integers(0, ne, 600)
            f = np.where(rng.uniform(size=600) < 0.3, 0.0, rng.uniform(-0.2, 1.2, 600))
            px = np.concatenate([(offset + rng.uniform(-1.5, 1.5, 600)) * scale,
                                 ax[k] + f * (bx[k] - ax[k])])
            py = np.concatenate([(offset + rng.uniform(-1.5, 1.5, 600)) * scale,
                                 ay[k] + f * (by[k] - ay[k])])
            py[:200] = ay[rng.integers(0, ne, 200)]
            px[700:900] *= 1 + rng.integers(-4, 5, 200) * 2.0**-52
            # the form and its test
            cx, cy = f32(0.5 * (ax.min() + ax.max())), f32(0.5 * (ay.min() + ay.max()))
            vx, vy = f32(np.roll(ax, 1) - float(cx)), f32(np.roll(ay, 1) - float(cy))
            vx, vy = np.append(vx, vx[0]), np.append(vy, vy[0])
            m = f32(max(np.abs(vx).max(), np.abs(vy).max()) * f32(1 + 2.0**-20))
            dx, dy = f32(px - float(cx)), f32(py - float(cy))
            s = np.abs(dx) + np.abs(dy) + m
            ux, uy = vx[:, None] - dx, vy[:, None] - dy
            t = f32(ux[:-1].astype(float) * uy[1:] - (ux[1:] * uy[:-1]).astype(float))
            certain = (np.abs(uy).min(0) > f32(2.0**-21) * s) & \
                (np.abs(t).min(0) > f32(2.0**-19) * (s * s))
            flip = ((uy[1:] < 0) != (uy[:-1] < 0)) & ((t < 0) == (uy[1:] < 0))
            got = flip.sum(0) % 2 == 1
            # the reference's arithmetic
            lhs = (px - ax[:, None]) * (by - ay)[:, None]
            rhs = (bx - ax)[:, None] * (py - ay[:, None])
            y1, y0 = ay[:, None] > py, by[:, None] > py
            want = (((y1 != y0) & ((lhs < rhs) != y1)).sum(0) % 2) == 1
            near = (np.abs(rhs - lhs) - 2.0**-48 * np.abs(rhs) <= 2.0**-1020).any(0)
            assert not (certain & near).any()
            assert np.array_equal(got[certain], want[certain])
            sure += certain[200:600].sum()
            total += 400
    assert sure > 0.99 * total
