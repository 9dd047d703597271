"""Pair counts of the dominant center type's tiles for the other center types
(pair-count mode), against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_MKNN, FAM_RDF, FAM_RIPK, Job, synth

pytestmark = pytest.mark.gpu

# (ions, type fractions, tasks): the other center types as minorities of one
# to several centers per cell, a center type that is no neighbour type, merged
# neighbour sets, one ion of the last type
CASES = [
    (30_000, [0.85, 0.12, 0.03], synth.ALL_PAIRS),
    (30_000, [0.55, 0.40, 0.05], [((1,), (1,)), ((2,), (1, 3)), ((3,), (2,))]),
    (20_001, [0.70, 0.20, 0.08, 0.02], [((1, 2), (1, 2, 3, 4)), ((4,), (1,))]),
    (4_099, [0.999, 0.001], [((1,), (1, 2)), ((2,), (1,))]),
]


@pytest.mark.parametrize("surface", ["frustum", "scattered"])
@pytest.mark.parametrize("n,frac,tasks", CASES)
def test_cross_type_pairs_count_once_for_both(ctx, n, frac, tasks, surface):
    """Every type of the cloud is a neighbour type, so the tiles of the type
    with the most centers count their pairs with the other types' centers for
    both sides; with scattered ion2surf every cell mixes centers and
    non-centers, values at fl32(R * R) and one ulp below it among them."""
    print(f"test_cross_type n={n} types={len(frac)} {surface}", flush=True)
    tip = synth.tip(n, 9, "frustum", 9.0, 5.0, 28.0 * n / 30_000 + 8.0, frac)
    s2 = tip.ion2surf_sqr.copy()
    R = np.float32(1.7)
    if surface == "scattered":
        rng = np.random.default_rng(n)
        s2 = rng.uniform(0, 6, size=n).astype(np.float32)
        edge = np.float32(R * R)
        s2[::7] = edge
        s2[3::7] = np.nextafter(edge, np.float32(0))
        s2[5] = np.inf
        s2[6] = np.nan
    job = Job(tasks, 0.0, 0.01, float(R), FAM_RDF | FAM_RIPK)
    cloud = ctx.upload(tip.xyz, tip.types, s2)
    try:
        got = ctx.run(cloud, job)
    finally:
        cloud.free()
    want, st = O.spatstat(tip.xyz, tip.types, s2, tasks, job.rmin, job.rincr, job.rmax,
                          job.families)
    assert np.array_equal(got.rdf, want["rdf"])
    assert np.array_equal(got.ripk, want["ripk"])
    assert got.pairs_inball == st["inball"]
    assert got.centers_considered == st["considered"]


@pytest.mark.parametrize("surface", ["frustum", "scattered"])
@pytest.mark.parametrize("n,frac,tasks", CASES)
def test_cross_type_pairs_hybrid(ctx, n, frac, tasks, surface):
    """The same with k-th neighbours: in the hybrid mode (which some of the cases
    take) the other types' tiles read the dominant type's ions over its kNN
    range only."""
    print(f"test_cross_type kNN n={n} types={len(frac)} {surface}", flush=True)
    tip = synth.tip(n, 9, "frustum", 9.0, 5.0, 28.0 * n / 30_000 + 8.0, frac)
    s2 = tip.ion2surf_sqr.copy()
    if surface == "scattered":
        s2 = np.random.default_rng(n + 1).uniform(0, 6, size=n).astype(np.float32)
    job = Job(tasks, 0.0, 0.01, 1.7, FAM_RDF | FAM_RIPK | FAM_MKNN, kvalues=[1, 2, 5])
    cloud = ctx.upload(tip.xyz, tip.types, s2)
    try:
        got = ctx.run(cloud, job)
    finally:
        cloud.free()
    print(got.kernel, flush=True)
    want, st = O.spatstat(tip.xyz, tip.types, s2, tasks, job.rmin, job.rincr, job.rmax,
                          job.families, kvalues=job.kvalues)
    for name in want:
        assert np.array_equal(getattr(got, name), want[name]), name
    assert got.pairs_inball == st["inball"]
