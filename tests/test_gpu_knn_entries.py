"""k-th neighbour categories settled from the entries of several tasks, at the
sizes of their steps (64 entries, 256 categories, 4 categories a lane) and on
both sides of what the entries hold, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_1NN, FAM_CNTNB, FAM_MKNN, FAM_RDF, FAM_RIPK, Job, synth

pytestmark = pytest.mark.gpu

ALL_PAIRS = synth.ALL_PAIRS
ONE = [((1,), (2,))]
MIX = [((1,), (1,)), ((1, 2), (1, 3)), ((3,), (2,)), ((1,), (1, 2, 3)), ((2,), (3,))]
# (tasks, increment, ks): full-range and hybrid histograms follow from the k
# and the families; 300 and 700 are beyond the entries of these stencils
CASES = [
    (ONE, 0.02, [1]),
    (ONE, 0.0023, list(range(1, 32))),
    (MIX, 0.01, list(range(1, 33))),
    (MIX, 0.004, [1, 2, 17, 33]),
    (ALL_PAIRS, 0.005, list(range(1, 21))),
    (ALL_PAIRS, 0.0051, [64, 65, 100]),
    (MIX, 0.01, [1, 50, 300]),
    (ONE, 0.01, [2, 129, 700]),
    # 1,268 categories: more than an entry's byte numbers
    (ALL_PAIRS, 0.0015, [1, 20, 40]),
]


@pytest.mark.parametrize("families", [FAM_RDF | FAM_MKNN, FAM_MKNN | FAM_1NN,
                                      FAM_RDF | FAM_RIPK | FAM_MKNN | FAM_1NN | FAM_CNTNB])
@pytest.mark.parametrize("tasks,incr,ks", CASES)
def test_knn_categories(ctx, tasks, incr, ks, families):
    print(f"test_knn_entries tasks={len(tasks)} kmax={ks[-1]} families={families}", flush=True)
    tip = synth.tip(6_007, 3, "frustum", 9.0, 5.0, 8.0, [0.6, 0.3, 0.1])
    job = Job(tasks, 0.0, incr, 1.9, families, kvalues=ks)
    cloud = ctx.upload(tip.xyz, tip.types, tip.ion2surf_sqr)
    try:
        got = ctx.run(cloud, job, cntnb_cap=65536)
    finally:
        cloud.free()
    want, _ = O.spatstat(tip.xyz, tip.types, tip.ion2surf_sqr, tasks, job.rmin, job.rincr,
                         job.rmax, families, kvalues=ks, cntnb_cap=65536)
    for name in want:
        assert np.array_equal(getattr(got, name), want[name]), name


def test_nearest_neighbour_alone(ctx):
    """1NN without MKNN: one entry per task and center."""
    print("test_knn_entries 1NN", flush=True)
    tip = synth.tip(3_001, 4, "frustum", 9.0, 5.0, 6.0, [0.97, 0.02, 0.01])
    for tasks in (ONE, MIX):
        job = Job(tasks, 0.0, 0.01, 1.2, FAM_RDF | FAM_1NN)
        cloud = ctx.upload(tip.xyz, tip.types, tip.ion2surf_sqr)
        try:
            got = ctx.run(cloud, job)
        finally:
            cloud.free()
        want, _ = O.spatstat(tip.xyz, tip.types, tip.ion2surf_sqr, tasks, job.rmin, job.rincr,
                             job.rmax, job.families)
        for name in want:
            assert np.array_equal(getattr(got, name), want[name]), name
