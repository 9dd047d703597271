"""Jobs whose histograms nearly fill the LDS: the rows of symmetric and
cross-type pair counting are left out where they do not fit, and never make a
job fail that runs without them."""
import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_1NN, FAM_MKNN, FAM_RDF, Job, PPError

pytestmark = pytest.mark.gpu


def cloud_of(n, frac, ids, edge):
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, edge, (n, 3)).astype(np.float32)
    ty = rng.choice(ids, n, p=frac).astype(np.uint8)
    return xyz, ty, np.full(n, 1e6, np.float32)


def run(ctx, cloud, job):
    try:
        return ctx.run(cloud, job)
    except PPError as e:
        assert "too large for LDS" in str(e)
        return None


# (families, k, type fractions, type ids, bins from, to, step): the hybrid mode
# with cross-type rows, the pair-count mode, large type ids, symmetric rows alone
CASES = [
    (FAM_RDF | FAM_MKNN, [1], [0.95, 0.04, 0.01], [1, 2, 3], 1800, 3000, 50),
    (FAM_RDF | FAM_1NN, [], [0.9, 0.1], [1, 225], 2600, 5000, 100),
    (FAM_RDF, [], [0.9, 0.1], [1, 254], 9800, 13800, 100),
    (FAM_RDF, [], [0.95, 0.04, 0.01], [1, 2, 3], 6400, 10400, 200),
    (FAM_RDF | FAM_MKNN, [2], [1.0], [1], 5000, 12000, 250),
]


@pytest.mark.parametrize("families,ks,frac,ids,first,last,step", CASES)
def test_no_job_is_refused_for_its_rows(ctx, families, ks, frac, ids, first, last, step):
    print(f"test_lds_limit types={ids} families={families}", flush=True)
    R = 2.0
    xyz, ty, s2 = cloud_of(2_000, frac, ids, 4.5)
    tasks = [((a,), (b,)) for a in ids for b in ids]
    cloud = ctx.upload(xyz, ty, s2)
    ran = refused = 0
    try:
        for bins in range(first, last + 1, step):
            job = Job(tasks, 0.0, float(np.float32(R / bins)), R, families, kvalues=ks)
            got = run(ctx, cloud, job)
            ctx.set_pair_symmetry(False)
            try:
                plain = run(ctx, cloud, job)
            finally:
                ctx.set_pair_symmetry(True)
            assert (got is None) == (plain is None), bins
            if got is None:
                refused += 1
                continue
            ran += 1
            for name, v in plain.arrays().items():
                assert np.array_equal(getattr(got, name), v), (bins, name)
            last_job, last_got = job, got
    finally:
        cloud.free()
    # the limit lies inside the range
    assert ran > 0 and refused > 0
    want, _ = O.spatstat(xyz, ty, s2, tasks, last_job.rmin, last_job.rincr, last_job.rmax,
                         families, kvalues=ks)
    for name in want:
        assert np.array_equal(getattr(last_got, name), want[name]), name
