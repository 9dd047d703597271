"""k-th neighbours of tasks with many neighbour types: settled one center at a
time by windows where many k make the entries' repeated reads the slower way,
against the oracle, with the way taken read from the launch trace."""
import re

import numpy as np
import pytest

from oracle import oracle as O
from paraprobe_amd import FAM_1NN, FAM_MKNN, FAM_RDF, Job

pytestmark = pytest.mark.gpu

ALL = tuple(range(1, 21))
# (tasks, bins, kmax, by entries): both sides of the line, one step of 128
# categories and two or three, one step of 64 entries and several
CASES = [
    ([(ALL, ALL)], 50, 300, False),
    ([(ALL, ALL)], 50, 1, False),
    ([((1, 2), ALL[:4])], 254, 64, True),
    ([((1, 2), ALL[:4])], 254, 65, False),
    ([((1,), (2,))], 62, 32, True),
    ([((1,), (2,))], 62, 33, False),
    ([((1,), (2,)), ((1, 2), ALL[:12])], 256, 300, False),
    ([((1,), (2,)), ((3,), (1,)), ((1, 2), (1, 2))], 256, 70, True),
]


@pytest.mark.parametrize("families", [FAM_MKNN | FAM_1NN, FAM_RDF | FAM_MKNN])
@pytest.mark.parametrize("tasks,bins,kmax,entries", CASES)
def test_many_types(ctx, capfd, monkeypatch, tasks, bins, kmax, entries, families):
    print(f"test_knn_many_types tasks={len(tasks)} bins={bins} kmax={kmax}", flush=True)
    rng = np.random.default_rng(bins + kmax)
    n = 5_003
    xyz = rng.uniform(0, 7, (n, 3)).astype(np.float32)
    ty = rng.choice(ALL, n).astype(np.uint8)
    s2 = rng.uniform(0, 6, n).astype(np.float32)
    R = float(np.float32(1.6))
    ks = sorted({1, 2, kmax // 2 + 1, kmax})
    job = Job(tasks, 0.0, float(np.float32(R / (bins + 0.5))), R, families, kvalues=ks)
    cloud = ctx.upload(xyz, ty, s2)
    monkeypatch.setenv("PP_TRACE_LAUNCH", "1")
    ctx.set_knn_range(0)  # the full range: the categories the case names
    try:
        got = ctx.run(cloud, job)
    finally:
        ctx.set_knn_range()
        cloud.free()
    taken = re.findall(r"pp: query mode=1 .* entries=(\d)", capfd.readouterr().err)
    assert taken == [str(int(entries))]
    want, _ = O.spatstat(xyz, ty, s2, tasks, job.rmin, job.rincr, job.rmax, families, kvalues=ks)
    for name in want:
        assert np.array_equal(getattr(got, name), want[name]), name
