"""Preparation of runs of many jobs: a block's segment from the list, one
workgroup per block of mostly padded cells, clouds without ions between others."""
import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_MKNN, FAM_RDF, Job

pytestmark = pytest.mark.gpu

# ions and cell width of the clouds that the jobs go round; 7 clouds, 3 segments
# a job: 342 jobs have 1,026 blocks of cells, 341 have 1,023
CLOUDS = [(60, 0.5), (0, 0.5), (1, 0.5), (2_049, 0.5), (700, 0.25), (2_048, 1.0), (3, 0.5)]


@pytest.mark.parametrize("njobs", [1, 7, 341, 342, 1_500])
def test_many_jobs(ctx, njobs):
    print(f"test_many_jobs {njobs}", flush=True)
    rng = np.random.default_rng(2)
    job = Job([((1, 2), (1,)), ((3,), (1, 2, 3))], 0.0, 0.05, 1.0, FAM_RDF | FAM_MKNN,
              kvalues=[1, 6])
    clouds, want = [], []
    for n, w in CLOUDS:
        xyz = rng.uniform(0, max(n / 20, 1) ** (1 / 3), (n, 3)).astype(np.float32)
        ty = rng.integers(1, 4, n).astype(np.uint8)
        s2 = rng.uniform(0, 3, n).astype(np.float32)
        clouds.append(ctx.upload(xyz, ty, s2, cell_width=w))
        want.append(O.spatstat(xyz, ty, s2, job.tasks, job.rmin, job.rincr, job.rmax,
                               job.families, kvalues=job.kvalues) if n else None)
    try:
        got = ctx.run_batch([clouds[i % 7] for i in range(njobs)], [job] * njobs)
    finally:
        for c in clouds:
            c.free()
    for i, r in enumerate(got):
        if want[i % 7] is None:
            assert r.centers_considered == 0 and not r.rdf.any() and not r.mknn.any(), i
            continue
        hist, st = want[i % 7]
        assert r.centers_considered == st["considered"], i
        assert np.array_equal(r.rdf, hist["rdf"]) and np.array_equal(r.mknn, hist["mknn"]), i
