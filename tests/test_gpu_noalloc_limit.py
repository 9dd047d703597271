"""The largest jobs that the no-allocation scratch holds, and small clouds with
many center types, whose lists take most beyond their ions' share."""
import numpy as np
import pytest

from paraprobe_amd import FAM_RDF, Job

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ntypes", [(5_576_575, 3), (931_181, 32), (3, 3), (33, 32)])
def test_scratch_holds(ctx, n, ntypes):
    print(f"noalloc: {n} ions, {ntypes} center types", flush=True)
    rng = np.random.default_rng(9)
    xyz = rng.uniform(0, 30, (n, 3)).astype(np.float32)
    xyz[0] = 0
    xyz[1] = 30  # (the box, so the cells)
    ty = (np.arange(n) % ntypes + 1).astype(np.uint8)
    s2 = np.zeros(n, np.float32)
    s2[: min(n, 500)] = 4.0
    job = Job([(tuple(range(1, ntypes + 1)), (1,))], 0.0, 0.1, 1.0, FAM_RDF)
    cloud = ctx.upload(xyz, ty, s2, cell_width=1.0)
    try:
        got = ctx.run_noalloc(cloud, job)
        want = ctx.run(cloud, job)
    finally:
        cloud.free()
    assert got.centers_considered == min(n, 500)
    assert np.array_equal(got.rdf, want.rdf)
