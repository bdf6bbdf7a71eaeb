"""The irradiance's folded source (CPU, no GPU): the eight images of a
direction under sign flips of x, y and z, read from one folded node's eight
slots, are the values that the unfolded lookup gives at each image; the frame
of a flipped texel samples the flipped set of directions; the orbit's texels
cover every face once.  A mistake in a mirror, a slot bit, the pole columns or
the fold's first node moves a lookup by whole texels of a noise map."""
import itertools

import numpy as np
import pytest

from tests.test_blend_grid import _bilinear, _cell

FLIPS = [(-1 if q & 1 else 1, -1 if q & 4 else 1, -1 if q & 2 else 1) for q in range(8)]


def _angles(d):
    xz = np.hypot(d[:, 0], d[:, 2])
    off_pole = xz > 0.001
    yaw = np.where(off_pole, np.arctan2(d[:, 2], d[:, 0]), 0.0)
    pitch = np.where(off_pole, np.arctan2(d[:, 1], xz), np.where(d[:, 1] > 0, 0.5, -0.5) * np.pi)
    return yaw, pitch


def _fold(value, w, h, blend):
    """The folded grid (rows, columns + 2, slot), as fold_grid_kernel forms it."""
    cols = (3 * w // 8 if blend else w // 4) + 2
    rows = (3 * h // 4 if blend else h // 2) + 2
    at = lambda k: 2.0 * ((k + 2) // 3) + 0.5 * ((k + 2) % 3) if blend else k + 1.0
    grid = np.zeros((rows, cols + 2, 8))
    c, r = np.arange(cols + 2), np.arange(rows)
    pole = c >= cols
    for slot in range(8):
        x = np.where(pole, 1.0 + (c - cols), at(c)) + 0.5 * w - 2.0
        y = at(r) + 0.5 * h - 2.0
        if slot & 1:
            x = np.where(pole, x, 1.5 * w - 1.0 - x)
        if slot & 2:
            x = np.where(pole, x, w - 1.0 - x)
        if not slot & 4:
            y = h - 1.0 - y
        X, Y = np.meshgrid(x, y)
        grid[..., slot] = value(X, Y)
    return grid, cols


def _fold_cell(x, blend):
    if blend:
        n, t = _cell(x)
        return n - 2, t
    return np.floor(x).astype(int) - 1, x - np.floor(x)


@pytest.mark.parametrize("w,h,delta", [(8, 4, 0.0), (8, 4, 0.4), (16, 16, 0.77), (32, 8, 0.0), (64, 32, 0.25), (16, 64, 0.5)])
def test_folded_lookup_is_the_unfolded_one_at_every_image(w, h, delta):
    rng = np.random.default_rng(w + h)
    fine = rng.uniform(0.0, 10.0, (h, w))
    coarse = 0.25 * (fine[0::2, 0::2] + fine[1::2, 0::2] + fine[0::2, 1::2] + fine[1::2, 1::2])
    blend = delta != 0.0

    def value(x, y):
        v = _bilinear(fine, x, y)
        return (1 - delta) * v + delta * _bilinear(coarse, 0.5 * x - 0.25, 0.5 * y - 0.25) if blend else v

    grid, cols = _fold(value, w, h, blend)
    d = rng.normal(size=(4000, 3))
    d[:200, [0, 2]] *= 1e-5  # inside the pole branch
    d[200:206] = [[1, 0, 0], [0, 0, 1], [0, 1, 0], [1, 1, 0], [0, 1, 1], [1, 0, 1]]
    d[206:300, 2] = 0.0
    d[300:400, 1] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    yaw, pitch = _angles(np.abs(d))
    off_pole = np.hypot(d[:, 0], d[:, 2]) > 0.001
    col, ax = _fold_cell(yaw * w / (2 * np.pi) + 1.5, blend)
    row, ay = _fold_cell(pitch * h / np.pi + 1.5, blend)
    col, ax = np.where(off_pole, col, cols), np.where(off_pole, ax, 0.5)
    assert col.min() >= 0 and row.min() >= 0 and row.max() + 1 < grid.shape[0]
    assert col[off_pole].max() + 1 < cols
    sign = np.signbit(d)
    own = sign[:, 0] * 1 + sign[:, 2] * 2 + sign[:, 1] * 4
    for q, f in enumerate(FLIPS):
        slot = own ^ q
        got = ((1 - ay) * ((1 - ax) * grid[row, col, slot] + ax * grid[row, col + 1, slot])
               + ay * ((1 - ax) * grid[row + 1, col, slot] + ax * grid[row + 1, col + 1, slot]))
        yw, pt = _angles(d * np.array(f))
        want = value(yw * w / (2 * np.pi) + 0.5 * w - 0.5, 0.5 * h - 0.5 - pt * h / np.pi)
        np.testing.assert_allclose(got, want, rtol=0, atol=1e-9)


def _frame(raw):
    n = raw / np.linalg.norm(raw)
    if abs(raw[0]) > abs(raw[1]):
        t = np.array([-n[2], 0.0, n[0]]) / np.hypot(n[0], n[2])
    else:
        t = np.array([0.0, n[2], -n[1]]) / np.hypot(n[1], n[2])
    return t, np.cross(n, t), n


@pytest.mark.parametrize("size,theta", [(1, 6), (2, 10), (3, 12), (4, 14)])
def test_orbits_cover_the_cube_and_share_their_samples(size, theta):
    half, even = (size + 1) // 2, 1 - size % 2
    seen = np.zeros((6, size, size), int)
    phi = [0.3, 0.9]
    ang = 2 * np.pi * np.arange(theta) / theta

    def samples(raw):
        t, b, n = _frame(raw)
        return np.array([n * np.cos(p) + (t * np.cos(a) + b * np.sin(a)) * np.sin(p) for p in phi for a in ang])

    order = lambda v: v[np.lexsort(np.round(v, 9).T + 0.0)]
    for axis, u, v in itertools.product(range(3), range(half), range(half)):
        cu, cv = 2 * u + even, 2 * v + even
        n = np.array([[size, cu, cv], [cu, size, cv], [cu, cv, size]][axis], float)
        base = samples(n)
        for q, f in enumerate(FLIPS):
            if any(f[k] < 0 and n[k] == 0 for k in range(3)):
                continue
            p = n * f
            np.testing.assert_allclose(order(samples(p)), order(base * f + 0.0), atol=1e-8)
            if axis == 0:
                face, sc, tc = (0, -p[2], -p[1]) if p[0] > 0 else (1, p[2], -p[1])
            elif axis == 1:
                face, sc, tc = (2, p[0], p[2]) if p[1] > 0 else (3, p[0], -p[2])
            else:
                face, sc, tc = (4, p[0], -p[1]) if p[2] > 0 else (5, -p[0], -p[1])
            x, y = (sc + size - 1) / 2, (tc + size - 1) / 2
            assert x == int(x) and y == int(y)
            seen[face, int(y), int(x)] += 1
    assert (seen == 1).all()
