"""The prefilter's texel pairs (CPU, no GPU): a texel of a positive face and its
partner on the opposite one sample directions that are each other's image
under a half turn, and on every level extent the partner's bilinear lookup is
the same fractions at a shifted cell (turn about y: half the width, towards the
other sign of z) or a mirrored one with its texels in the opposite order (turn
about x).  A wrong branch, shift, mirror or tap order moves a lookup on a
noise map by whole texels."""
import numpy as np
import pytest

from tests.test_irradiance_fold import _angles, _frame


def _raw(face, x, y, S):
    sc, tc, m = 2 * x + 1 - S, 2 * y + 1 - S, S
    return np.array([(m, -tc, -sc), (-m, -tc, sc), (sc, m, tc), (sc, -m, -tc), (sc, -tc, m), (-sc, -tc, -m)][face], float)


def _bilinear(level, ix, iy, ax, ay, reverse=False):
    h, w = level.shape
    t = [level[(iy + j) % h, (ix + i) % w] for j in (0, 1) for i in (0, 1)]
    wt = [(1 - ax) * (1 - ay), ax * (1 - ay), (1 - ax) * ay, ax * ay]
    return sum(a * b for a, b in zip(t[::-1] if reverse else t, wt))


@pytest.mark.parametrize("size", [1, 2, 4, 8])
@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (1, 4), (4, 16), (16, 4), (64, 32)])
def test_pairs_share_directions_and_cells(size, w, h):
    rng = np.random.default_rng(size * 1000 + w + h)
    level = rng.uniform(0.0, 10.0, (h, w))
    local = rng.normal(size=(60, 3))
    local[:, 2] = np.abs(local[:, 2])
    local = np.concatenate([local / np.linalg.norm(local, axis=1, keepdims=True), [[0.0, 0.0, 1.0]]])
    seen = np.zeros((6, size, size), int)
    for face in (0, 2, 4):
        for y in range(size):
            for x in range(size):
                n = _raw(face, x, y, size)
                turn_y = abs(n[0]) > abs(n[1])
                f = np.array([-1, 1, -1] if turn_y else [1, -1, -1])
                mirror = face == 4 and not turn_y
                x2, y2 = (size - 1 - x, size - 1 - y) if mirror else (x, y)
                partner = _raw(face + 1, x2, y2, size)
                np.testing.assert_array_equal(partner + 0.0, n * f + 0.0)
                seen[face, y, x] += 1
                seen[face + 1, y2, x2] += 1
                a, b = (local @ np.array(_frame(v)) for v in (n, partner))
                np.testing.assert_allclose(b, a * f, atol=1e-12)
                near = np.abs(a[:, 2]) < 1e-9  # yaw on the seam: either side is the same texel
                yaw, pitch = _angles(a)
                X, Y = yaw * w / (2 * np.pi) + 0.5 * w - 0.5, -pitch * h / np.pi + 0.5 * h - 0.5
                ix, iy = np.floor(X).astype(int), np.floor(Y).astype(int)
                ax, ay = X - ix, Y - iy
                off_pole = np.hypot(a[:, 0], a[:, 2]) > 0.001
                turn = np.where(off_pole, np.where(np.signbit(a[:, 2]), 1, -1), 0)
                sx, sy = (ix + turn * (w // 2), iy) if turn_y else (w - 2 - ix, h - 2 - iy)
                ok = ~near
                assert sx[ok].min() >= -1 and sx[ok].max() <= w - 1 and sy[ok].min() >= -1 and sy[ok].max() <= h - 1
                got = _bilinear(level, sx, sy, ax, ay, reverse=not turn_y)
                yw, pt = _angles(b)
                X, Y = yw * w / (2 * np.pi) + 0.5 * w - 0.5, -pt * h / np.pi + 0.5 * h - 0.5
                jx, jy = np.floor(X).astype(int), np.floor(Y).astype(int)
                np.testing.assert_allclose(got, _bilinear(level, jx, jy, X - jx, Y - jy), atol=1e-8)
    assert (seen == 1).all()
