"""Triangle lists of the ion-to-surface distance: triangles that touch one cell,
a few, and many times the 64 cells a wavefront takes at once, against the
oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntri", [1, 3, 4, 5, 257])
@pytest.mark.parametrize("extent,R", [(0.01, 0.4), (1.5, 1.0), (40.0, 2.0)])
def test_triangle_cells(ctx, ntri, extent, R):
    print(f"test_triangle_cells ntri={ntri} extent={extent} R={R}", flush=True)
    rng = np.random.default_rng(ntri)
    xyz = rng.uniform(0, 20, size=(20_000, 3)).astype(np.float32)
    at = rng.uniform(-2, 22, size=(ntri, 1, 3))
    tri = (at + rng.uniform(-extent, extent, size=(ntri, 3, 3))).astype(np.float32)
    tri = tri.reshape(ntri, 9)
    got = ctx.ion2surf(xyz, tri, R)
    want = O.ion2surf(xyz, tri, R)
    assert np.array_equal(got.view(np.uint32), np.asarray(want, np.float32).view(np.uint32))
