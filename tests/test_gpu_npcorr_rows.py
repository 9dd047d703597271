"""Candidate rows of the n-point correlations: neighbours on the limits of the
rows and shells, and the smallest and largest scales of the coordinates,
against the brute-force oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

TASKS = [((1,), (2,))]


def check(ctx, xyz, ty, tasks, R, width, K):
    s2 = np.full(len(ty), np.inf, np.float32)
    cloud = ctx.upload(xyz, ty, s2)
    try:
        got = ctx.npcorr(cloud, tasks, R, width, K)
    finally:
        cloud.free()
    want = O.npcorr(xyz, ty, s2, tasks, R, width, K)
    assert want.sum() > 0
    assert np.array_equal(got, want)


@pytest.mark.parametrize("scale", [4e-19, 7e-19, 1e-18, 1.3e-18, 1e-17, 1.0, 1e18, 1.2e19])
def test_scales(ctx, scale):
    """R * R from the subnormal numbers' edge to the largest floats; from 7e-19 to
    1.3e-18 the width of a distance bucket is subnormal."""
    print(f"npcorr scale={scale}", flush=True)
    rng = np.random.default_rng(1)
    n = 2000
    xyz = (rng.uniform(0, 6, (n, 3)) * scale).astype(np.float32)
    ty = rng.choice([1, 2], n, p=[0.7, 0.3]).astype(np.uint8)
    R = float(np.float32(1.3 * scale))
    for K in (0, 7, 20):
        check(ctx, xyz, ty, [((1,), (1,)), ((2,), (1, 2))], R, R / 8, K)


@pytest.mark.parametrize("limit", ["ball", "bucket"])
@pytest.mark.parametrize("corner", [0.0, 20.0])
def test_neighbours_on_the_limits_of_rows(ctx, limit, corner):
    """900 centers far apart, each with one neighbour: on the near faces of a
    stencil row within an ulp, at R within a few ulp (ball), or on a cell
    face along x at the bound of a distance bucket (bucket)."""
    print(f"npcorr limits {limit} corner={corner}", flush=True)
    rng = np.random.default_rng(3)
    R = np.float32(1.25)
    w = float(np.float32(0.5) * R * np.float32(1.0 + 2.0**-10))  # the cells' width
    lo = corner
    xyz, ty = [(lo, lo, lo)], [3]  # (the grid's origin)
    for c in range(900):
        cell = 4 + 9 * np.array([c % 10, c // 10 % 10, c // 100])
        f = rng.uniform(0, 1, 3)
        if c % 3 == 0:
            f[rng.integers(3)] = rng.choice([0.0, 1.0 - 1e-7])
        p = np.float32(lo + (cell + f) * w)
        d = rng.integers(-2, 3, 3)  # the row, and the cell face along x
        face = lo + (cell + np.where(d > 0, d, d + 1)) * w
        q = np.where(d == 0, lo + (cell + rng.uniform(0, 1, 3)) * w, face)
        if limit == "ball":
            h2 = (q[1] - p[1]) ** 2 + (q[2] - p[2]) ** 2
            # (a row beyond R gives a neighbour that is none)
            q[0] = p[0] + rng.choice([-1, 1]) * np.sqrt(max(float(R) ** 2 - h2, 0.0))
        else:
            b = rng.integers(1, 257)
            r2 = b * float(R) ** 2 / 256
            left = max(r2 - (q[0] - p[0]) ** 2, 0.0)
            phi = rng.uniform(0, 2 * np.pi)
            q[1:] = p[1:] + np.sqrt(left) * np.array([np.cos(phi), np.sin(phi)])
        q = np.float32(q)
        for a in range(3):
            for _ in range(rng.integers(0, 3)):
                q[a] = np.nextafter(q[a], p[a] if rng.random() < 0.6 else np.float32(np.inf))
        xyz += [p, q]
        ty += [1, 2]
    check(ctx, np.array(xyz, np.float32), np.array(ty, np.uint8), TASKS, float(R), 0.05, 0)
