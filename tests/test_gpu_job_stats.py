"""A job's pair totals over many center types, alone and with other jobs in one
launch: each workgroup adds them behind its last tile of a job."""
import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_1NN, FAM_CNTNB, FAM_MKNN, FAM_RDF, Job

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("families", [FAM_1NN, FAM_RDF, FAM_CNTNB | FAM_1NN, FAM_RDF | FAM_MKNN])
def test_totals(ctx, families):
    print(f"test_job_stats families={families}", flush=True)
    rng = np.random.default_rng(families)
    clouds, jobs, want = [], [], []
    for ntypes, n in ((1, 900), (20, 9_000), (3, 64), (20, 5_001), (7, 1)):
        xyz = rng.uniform(0, 6, (n, 3)).astype(np.float32)
        p = np.full(ntypes, 0.1 / max(ntypes - 1, 1))
        p[0] = 1 - p[1:].sum()
        ty = rng.choice(np.arange(1, ntypes + 1), n, p=p).astype(np.uint8)
        s2 = rng.uniform(0, 3, n).astype(np.float32)
        al = tuple(range(1, ntypes + 1))
        # every type a center type, every type or all but one a neighbour type
        env = al if len(jobs) % 2 else al[: max(1, ntypes - 1)]
        job = Job([(al, env)], 0.0, 0.02, 1.1, families, kvalues=[1, 3])
        clouds.append((xyz, ty, s2))
        jobs.append(job)
        want.append(O.spatstat(xyz, ty, s2, job.tasks, job.rmin, job.rincr, job.rmax, families,
                               kvalues=job.kvalues, cntnb_cap=4096))
    dev = [ctx.upload(*c) for c in clouds]
    try:
        single = [ctx.run(c, j, cntnb_cap=4096) for c, j in zip(dev, jobs)]
        batch = ctx.run_batch(dev, jobs, cntnb_cap=4096)
    finally:
        for c in dev:
            c.free()
    for one, two, (hist, st) in zip(single, batch, want):
        for got in (one, two):
            assert got.pairs_inball == st["inball"]
            assert got.pairs_candidate == one.pairs_candidate
            assert got.pairs_candidate >= st["inball"]
            for name in hist:
                assert np.array_equal(getattr(got, name), hist[name]), name
