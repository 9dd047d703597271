"""The query kernel's variants, each with a job that is known to take it (read
from the launch trace), against the oracle and against the same job without
symmetric counting."""
import re

import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_1NN, FAM_MKNN, FAM_RDF, FAM_RIPK, Job, synth

pytestmark = pytest.mark.gpu

PAIRS = synth.ALL_PAIRS
MIX = [((1,), (1,)), ((1, 2), (1, 3)), ((3,), (2,)), ((2,), (3,))]


def traced(ctx, capfd, cloud, job):
    """The result and per launch (mode, jobs with entries, entry words, cross rows)."""
    capfd.readouterr()
    got = ctx.run(cloud, job)
    lines = re.findall(r"pp: query mode=(\d).*entw=(\d+) entries=(\d+) cross=(\d)",
                       capfd.readouterr().err)
    return got, [tuple(map(int, m)) for m in lines]


def check(ctx, capfd, monkeypatch, tip, s2, job):
    monkeypatch.setenv("PP_TRACE_LAUNCH", "1")
    cloud = ctx.upload(tip.xyz, tip.types, s2)
    try:
        got, lines = traced(ctx, capfd, cloud, job)
        ctx.set_pair_symmetry(False)
        try:
            plain, plain_lines = traced(ctx, capfd, cloud, job)
        finally:
            ctx.set_pair_symmetry(True)
    finally:
        cloud.free()
    want, st = O.spatstat(tip.xyz, tip.types, s2, job.tasks, job.rmin, job.rincr, job.rmax,
                          job.families, kvalues=job.kvalues)
    for r in (got, plain):
        for name in want:
            assert np.array_equal(getattr(r, name), want[name]), name
        assert r.pairs_inball in (st["inball"], -1)
    return got, lines, plain, plain_lines


@pytest.mark.parametrize("surface", ["frustum", "scattered"])
@pytest.mark.parametrize("families,mode", [(FAM_RDF | FAM_RIPK, 0), (FAM_RDF | FAM_MKNN, 2),
                                           (FAM_RDF | FAM_1NN, 2)])
@pytest.mark.parametrize("frac", [[0.85, 0.12, 0.03], [0.55, 0.40, 0.05]])
def test_cross_type_rows(ctx, capfd, monkeypatch, families, mode, frac, surface):
    """The dominant type's tiles count its pairs with the other types' centers for
    both, in the pair-count and in the hybrid mode."""
    tip = synth.tip(30_000, 9, "frustum", 9.0, 5.0, 36.0, frac)
    s2 = tip.ion2surf_sqr
    if surface == "scattered":
        s2 = np.random.default_rng(3).uniform(0, 12, size=len(s2)).astype(np.float32)
    job = Job(PAIRS, 0.0, 0.01, 2.6, families, kvalues=[1, 2] if families & FAM_MKNN else [])
    got, lines, plain, plain_lines = check(ctx, capfd, monkeypatch, tip, s2, job)
    assert lines[0][0] == mode and lines[0][3] == 1
    assert plain_lines[0][0] == mode and plain_lines[0][3] == 0
    assert got.pairs_candidate < plain.pairs_candidate


# (tasks, increment, ks, mode, by entries, in words of their own): in the stencil rows' words, in words
# of their own, k beyond both, categories beyond a byte, many types
KNN = [
    (PAIRS, 0.02, [1, 5], 1, 1, 0),
    (PAIRS, 0.005, list(range(1, 21)), 1, 1, 0),
    (MIX, 0.004, [1, 17, 60], 1, 1, 0),
    (PAIRS, 0.005, [64, 65, 100], 1, 1, 1),
    (PAIRS, 0.01, [3, 400], 1, 0, 0),
    (PAIRS, 0.0015, [1, 20], 1, 0, 0),
    (PAIRS, 1.9 / 1014.5, [1, 20, 60], 1, 1, 0),  # 1,016 categories, 254 groups of 4
    (PAIRS, 1.9 / 1015.5, [1, 20, 60], 1, 0, 0),
    (MIX, 0.02, [1, 150], 1, 0, 0),
]


@pytest.mark.parametrize("tasks,incr,ks,mode,entries,own", KNN)
def test_knn_way(ctx, capfd, monkeypatch, tasks, incr, ks, mode, entries, own):
    tip = synth.tip(6_007, 3, "frustum", 9.0, 5.0, 8.0, [0.6, 0.3, 0.1])
    ctx.set_knn_range(0)  # full-range histograms
    try:
        job = Job(tasks, 0.0, float(np.float32(incr)), 1.9, FAM_RDF | FAM_MKNN, kvalues=ks)
        _, lines, _, _ = check(ctx, capfd, monkeypatch, tip, tip.ion2surf_sqr, job)
    finally:
        ctx.set_knn_range()
    print(lines, flush=True)
    assert lines[0][0] == mode and lines[0][2] == entries and (lines[0][1] > 0) == bool(own)


def test_knn_way_hybrid(ctx, capfd, monkeypatch):
    """The hybrid mode's first pass and its full-range rerun, both by entries."""
    tip = synth.tip(30_000, 9, "frustum", 9.0, 5.0, 36.0, [0.85, 0.12, 0.03])
    job = Job(PAIRS, 0.0, 0.01, 2.6, FAM_RDF | FAM_MKNN, kvalues=[1, 2])
    got, lines, _, _ = check(ctx, capfd, monkeypatch, tip, tip.ion2surf_sqr, job)
    print(lines, got.centers_rerun, flush=True)
    assert lines[0][0] == 2 and lines[0][2] == 1


@pytest.mark.parametrize("bins,kmax,cells", [(800, 5, 3), (800, 10, 2), (1000, 5, 2), (1300, 5, 3)])
def test_cells_of_a_dense_cloud(ctx, capfd, monkeypatch, bins, kmax, cells):
    """Cells of Rmax/2 by Rmax/4, and cubes of Rmax/3 where only they leave room for
    symmetric or cross-type counting."""
    rng = np.random.default_rng(7)
    n, R = 6_000, 4.2
    xyz = rng.uniform(0, (n / 36) ** (1 / 3), (n, 3)).astype(np.float32)
    ty = rng.choice([1, 2, 3], n, p=[0.7, 0.2, 0.1]).astype(np.uint8)
    s2 = np.full(n, 100.0, np.float32)
    job = Job(PAIRS, 0.0, float(np.float32(R / bins)), R, FAM_RDF | FAM_MKNN, kvalues=[1, kmax])
    monkeypatch.setenv("PP_TRACE_LAUNCH", "1")
    cloud = ctx.upload(xyz, ty, s2)
    try:
        got, lines = traced(ctx, capfd, cloud, job)
    finally:
        cloud.free()
    print(got.kernel, lines, flush=True)
    assert got.kernel.endswith(f"hybrid> cells/Rmax={cells}")
    want, st = O.spatstat(xyz, ty, s2, job.tasks, job.rmin, job.rincr, job.rmax, job.families,
                          kvalues=job.kvalues)
    for name in want:
        assert np.array_equal(getattr(got, name), want[name]), name
    assert got.pairs_inball == st["inball"]
