"""Ion-to-surface distances with more triangles than a launch has wavefronts for
(a wavefront walks several from 2^22 on) and than a grid of a wavefront per
triangle could hold (2^26)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2", [22, 26])
def test_many_triangles(ctx, log2):
    """All but 14 triangles lie beyond R of every ion, in cells without ions."""
    print(f"test_many_triangles 2^{log2} + 6", flush=True)
    rng = np.random.default_rng(log2)
    xyz = rng.uniform(0, 10, (3_000, 3)).astype(np.float32)
    xyz[-1] = 100.0  # (cells 44 wide: the far triangles' hold no ion)
    R = 2.0
    ntri = (1 << log2) + 6
    near = (rng.uniform(0, 10, (14, 1, 3)) + rng.uniform(-0.5, 0.5, (14, 3, 3))).astype(np.float32)
    far = rng.uniform([50, 0, 0], [84, 84, 84], (1 << 16, 1, 3)) + rng.uniform(0, 0.1, (1 << 16, 3, 3))
    tri = np.empty((ntri, 9), np.float32)
    tri[: 1 << log2].reshape(-1, 1 << 16, 9)[:] = far.reshape(1, 1 << 16, 9).astype(np.float32)
    # the first, the last, and one near the end of a launch's first pass
    at = [0, 1, (1 << 22) - 20, *range(ntri - 11, ntri)]
    tri[at] = near.reshape(14, 9)
    got = ctx.ion2surf(xyz, tri, R)
    want = np.asarray(O.ion2surf(xyz, near.reshape(14, 9), R), np.float32)
    assert (want < R * R).any()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("R", [0.3, 2.5, 2.54])
@pytest.mark.parametrize("ntri", [1, 63, 64, 65, 4_099])
def test_small_triangles(ctx, ntri, R):
    """Cells of about 5.04: a group of lanes per triangle where R is less than
    half of that, a wavefront from there on."""
    print(f"test_small_triangles ntri={ntri} R={R}", flush=True)
    rng = np.random.default_rng(ntri)
    xyz = rng.uniform(0, 20, (16_000, 3)).astype(np.float32)
    extent = rng.choice([0.01, 0.5, 6.0], (ntri, 1, 1))
    tri = rng.uniform(0, 20, (ntri, 1, 3)) + rng.uniform(-1, 1, (ntri, 3, 3)) * extent
    tri = np.clip(tri, 0, 20).astype(np.float32).reshape(ntri, 9)
    got = ctx.ion2surf(xyz, tri, R)
    want = np.asarray(O.ion2surf(xyz, tri, R), np.float32)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
