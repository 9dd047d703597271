"""Center lists and tiles of a run (blocks of 2048 ions and of 2048 cells, words
of 64 ions) at the edges of their blocks, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_MKNN, FAM_RDF, Job

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 2047, 2048, 2049, 4096, 6145]
TASKS = [[((1,), (1, 2))], [((1,), (2,)), ((3,), (1, 3)), ((2,), (1,))]]


def case(n, ntasks, surface):
    rng = np.random.default_rng(100 * n + ntasks)
    # about 4 ions per unit volume, so cells and their blocks vary with n
    edge = max((n / 4.0) ** (1 / 3), 0.5)
    xyz = rng.uniform(0, edge, size=(n, 3)).astype(np.float32)
    types = rng.integers(1, 4, size=n).astype(np.uint8)
    s2 = rng.uniform(0, 4, size=n).astype(np.float32)
    if surface == "all":
        s2[:] = np.float32(1e6)  # every ion of the last block is a center
    elif surface == "last":
        s2[:] = 0
        s2[-1] = np.inf
    # k beyond what small clouds hold: the full-range rerun flags its centers
    job = Job(TASKS[ntasks], 0.0, 0.01, 1.2, FAM_RDF | FAM_MKNN, kvalues=[1, 30])
    return xyz, types, s2, job


@pytest.mark.parametrize("surface", ["scattered", "all", "last"])
@pytest.mark.parametrize("ntasks", [0, 1])
def test_center_lists_at_block_edges(ctx, ntasks, surface):
    """One by one and as one batch (segments of different jobs side by side)."""
    print(f"test_center_lists tasks={ntasks} {surface}", flush=True)
    cases = [case(n, ntasks, surface) for n in SIZES]
    clouds = [ctx.upload(x, t, s) for x, t, s, _ in cases]
    try:
        single = [ctx.run(cl, c[3]) for cl, c in zip(clouds, cases)]
        batch = ctx.run_batch(clouds, [c[3] for c in cases])
    finally:
        for cl in clouds:
            cl.free()
    for (xyz, types, s2, job), one, two in zip(cases, single, batch):
        want, st = O.spatstat(xyz, types, s2, job.tasks, job.rmin, job.rincr, job.rmax,
                              job.families, kvalues=job.kvalues)
        for got in (one, two):
            assert np.array_equal(got.rdf, want["rdf"])
            assert np.array_equal(got.mknn, want["mknn"])
            assert got.centers_considered == st["considered"]
