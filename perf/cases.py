"""The work this framework is run for, as cases that can be timed and compared.

A case names one pass through the public entry points of ``paraprobe_amd``:

* ``spatstat``: RDF / Ripley K / kNN / neighbour-count histograms of one job
  on a tip that stays on the GPU (``SpatStat.run``);
* ``batch``: many tips of uneven size, each with its own type pair, Rmax and
  k, in one call (``SpatStat.run_batch``);
* ``serve``: a burst of requests on resident tips (``Server``);
* ``npcorr``: the n-point correlation cubes (``SpatStat.npcorr``);
* ``ion2surf``: squared distances of all ions to a triangle hull;
* ``pos``: POS records to positions and ranged types, in device memory;
* ``tip``: from the bytes of a POS file, a range table and a hull to a tip on
  the GPU, one job on it, and the tip given back -- the whole way of a user
  with one new measurement.

Tips are frusta of the headline shape (radii and height 0.16 : 0.08 : 1), or
cylinders, at the densities of the repository's workloads, with type labels
1, 2, 3 at the repository's fractions and, for clustered tips, 2,500 spheres of
radius 1-2 nm per million ions in which type 2 is enriched to 40 %.  Ions are
made on the GPU from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from paraprobe_amd import (FAM_1NN, FAM_CNTNB, FAM_MKNN, FAM_RDF, FAM_RIPK, Job, SpatStat,
                           hist_geometry, synth, workloads)
from paraprobe_amd.capi import Server

FAMILIES = {"RDF": FAM_RDF, "1NN": FAM_1NN, "RIPK": FAM_RIPK, "MKNN": FAM_MKNN,
            "CNTNB": FAM_CNTNB}
TASKS = {
    "BB": [((2,), (2,))],
    "AB": [((1,), (2,))],
    "all": synth.ALL_PAIRS,  # the 9 ordered pairs of types 1, 2, 3
    "npc": [((1,), (1,)), ((2,), (2,)), ((1,), (2,)), ((2,), (1,))],
}
FRACTIONS = [0.95, 0.04, 0.01]
ENRICHED = 0.40
# Unknown's dummy range, then four elements as a small RRNG file holds them
RANGES = (np.array([0.0, 26.7, 55.7, 13.9, 44.8], np.float32),
          np.array([0.001, 26.9, 56.2, 14.1, 45.1], np.float32),
          np.array([0, 1, 2, 3, 4], np.uint8))
MASSES = (26.98, 55.94, 13.98)  # of types 1, 2, 3


def listed():
    return [
        # the smallest calls: a region of interest of 20,000 ions, every pair,
        # where launches and host work are most of the time
        dict(name="roi-20k-all-pairs", kind="spatstat", n=20_000, shape="frustum",
             clustered=False, density=27.3, tasks="all", families="RDF+1NN+MKNN", rmax=1.5,
             rincr=0.01, kmax=10),
        # a small uniform specimen and one minority pair: RDF, the sparse case
        dict(name="cylinder-1m-rdf-BB", kind="spatstat", n=1_000_000, shape="cylinder",
             clustered=False, density=22.1, tasks="BB", families="RDF", rmax=2.0, rincr=0.01,
             kmax=0),
        # families that need every neighbour of every center: Ripley K, 1NN
        # and the neighbour counts, full-range histograms per center
        dict(name="roi-333k-counts", kind="spatstat", n=333_333, shape="frustum",
             clustered=True, density=27.3, tasks="all", families="RIPK+1NN+CNTNB", rmax=2.0,
             rincr=0.02, kmax=0),
        # an ordinary tip, radial distributions of all pairs
        dict(name="tip-4m-rdf", kind="spatstat", n=4_000_037, shape="frustum", clustered=True,
             density=27.3, tasks="all", families="RDF", rmax=3.0, rincr=0.01, kmax=0),
        # the headline job: RDF and kNN up to k = 100 for all pairs
        dict(name="tip-20m-rdf-mknn100", kind="spatstat", n=20_000_000, shape="frustum",
             clustered=True, density=27.3, tasks="all", families="RDF+MKNN", rmax=5.0,
             rincr=0.01, kmax=100),
        # the largest reconstruction
        dict(name="tip-100m-rdf-mknn20", kind="spatstat", n=100_000_000, shape="frustum",
             clustered=True, density=22.0, tasks="all", families="RDF+MKNN", rmax=3.0,
             rincr=0.005, kmax=20),
        # a study over many tips: one pair, Rmax and k each
        dict(name="batch-24", kind="batch", count=24, spec=3, nmin=50_000, nmax=4_000_000),
        # requests that arrive together at a service with resident tips
        dict(name="serve-48", kind="serve", requests=48, stream=17, nmin=1_000_000, tips=3),
        # the 100th neighbour's difference vectors
        dict(name="npcorr-4m", kind="npcorr", n=4_000_000, rmax=2.5, rincr=0.05, order=99),
        # distance of every ion to the tip surface
        dict(name="ion2surf-5m-hull66k", kind="ion2surf", n=5_000_000, nseg=256, nz=128,
             radius=5.0),
        # decoding and ranging a large POS file in device memory
        dict(name="pos-20m", kind="pos", n=20_000_003),
        # one new measurement from file bytes to histograms
        dict(name="newtip-2m", kind="tip", n=2_000_000, nseg=128, nz=64, tasks="BB",
             families="RDF+MKNN", rmax=2.0, rincr=0.01, kmax=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spatstat", "spatstat", "spatstat", "spatstat", "batch", "serve",
                       "npcorr", "ion2surf", "pos", "tip"])
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(4, 30), spec=rng.randint(1, 10_000),
                    nmin=50_000, nmax=_log_int(rng, 200_000, 4_000_000))
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(4, 60), stream=rng.randint(1, 10_000),
                    nmin=_log_int(rng, 200_000, 1_000_000), tips=rng.randint(1, 3))
    if kind == "npcorr":
        return dict(kind=kind, n=_log_int(rng, 50_000, 8_000_000),
                    rmax=round(rng.uniform(1.5, 3.0), 2), rincr=0.05, order=rng.randint(0, 150))
    if kind == "ion2surf":
        return dict(kind=kind, n=_log_int(rng, 20_000, 20_000_000), nseg=rng.randint(24, 512),
                    nz=rng.randint(8, 256), radius=round(rng.uniform(1.0, 5.0), 2))
    if kind == "pos":
        return dict(kind=kind, n=_log_int(rng, 20_000, 50_000_000))
    if kind == "tip":
        return dict(kind=kind, n=_log_int(rng, 50_000, 4_000_000), nseg=rng.randint(24, 256),
                    nz=rng.randint(8, 128), tasks=rng.choice(["BB", "AB", "all"]),
                    families=rng.choice(["RDF", "RDF+MKNN", "RIPK+1NN"]),
                    rmax=round(rng.uniform(1.0, 3.0), 2), rincr=0.01, kmax=rng.randint(1, 50))
    c = dict(kind=kind, n=_log_int(rng, 20_000, 20_000_000), shape="frustum",
             clustered=rng.random() < 0.7, density=round(rng.uniform(22.0, 27.3), 1),
             tasks=rng.choice(["BB", "AB", "all", "all"]),
             families=rng.choice(["RDF", "RDF+MKNN", "RDF+MKNN", "MKNN", "RDF+1NN",
                                  "RIPK+1NN+CNTNB"]),
             rmax=round(rng.uniform(1.0, 5.0), 2), rincr=rng.choice([0.005, 0.01, 0.02]),
             kmax=rng.randint(1, 100))
    if "CNTNB" in c["families"]:
        # full-range histograms per center: regions of interest, coarser bins
        c["n"] = _log_int(rng, 20_000, 1_000_000)
        c["rmax"] = round(rng.uniform(1.0, 2.5), 2)
        c["rincr"] = 0.02
    return c


# ---------------------------------------------------------------------------
# synthetic tips on the GPU

def _shape(case_n, shape, density):
    """Radii at the bottom and the top, and height, in nm."""
    v = case_n / density
    if shape == "cylinder":  # height 64 for radius 15
        h = (v / (math.pi * (15.0 / 64.0) ** 2)) ** (1.0 / 3.0)
        return 15.0 / 64.0 * h, 15.0 / 64.0 * h, h
    h = (v / (math.pi / 3.0 * (0.16 ** 2 + 0.16 * 0.08 + 0.08 ** 2))) ** (1.0 / 3.0)
    return 0.16 * h, 0.08 * h, h


def _points(n, r0, r1, h, gen, shrink=1.0):
    """n points uniform in the solid (float32, [n, 3])."""
    dev = "cuda"
    u = torch.rand(n, generator=gen, device=dev)
    if r0 == r1:
        z = u * h
        r = torch.full_like(z, r0)
    else:
        r = (r0 ** 3 - u.double() * (r0 ** 3 - r1 ** 3)).pow_(1.0 / 3.0).float()
        z = (r0 - r) * (h / (r0 - r1))
    del u
    rho = torch.rand(n, generator=gen, device=dev).sqrt_().mul_(r).mul_(shrink)
    del r
    phi = torch.rand(n, generator=gen, device=dev).mul_(2.0 * math.pi)
    xyz = torch.empty((n, 3), device=dev)
    xyz[:, 0] = rho * torch.cos(phi)
    xyz[:, 1] = rho * torch.sin(phi)
    xyz[:, 2] = z.clamp_(0.0, h)
    return xyz


def _types(xyz, r0, r1, h, nclusters, gen):
    """Labels 1..3; inside the clusters type 2 at ENRICHED."""
    n = xyz.shape[0]
    u = torch.rand(n, generator=gen, device="cuda")
    a, b = FRACTIONS[0], FRACTIONS[0] + FRACTIONS[1]
    t = (1 + (u >= a).to(torch.uint8) + (u >= b).to(torch.uint8))
    if nclusters:
        vox = 0.5
        rm = max(r0, r1) + 3.0
        d = [int(2 * rm / vox) + 1, int(2 * rm / vox) + 1, int((h + 6.0) / vox) + 1]
        lo = torch.tensor([-rm, -rm, -3.0], device="cuda")
        inside = torch.zeros(d[0] * d[1] * d[2], dtype=torch.bool, device="cuda")
        c = _points(nclusters, r0, r1, h, gen)
        rad = 1.0 + torch.rand(nclusters, generator=gen, device="cuda")
        k = torch.arange(-4, 5, device="cuda")
        off = torch.stack(torch.meshgrid(k, k, k, indexing="ij"), -1).reshape(1, -1, 3)
        for s in range(0, nclusters, 20_000):
            cc, rr = c[s:s + 20_000], rad[s:s + 20_000]
            v = ((cc - lo) / vox).long()[:, None, :] + off
            mid = (v.float() + 0.5) * vox + lo
            m = (mid - cc[:, None, :]).square().sum(-1) <= rr[:, None] ** 2
            v = v[m]
            inside[(v[:, 2] * d[1] + v[:, 1]) * d[0] + v[:, 0]] = True
        for s in range(0, n, 1 << 25):
            v = ((xyz[s:s + (1 << 25)] - lo) / vox).long()
            m = inside[(v[:, 2] * d[1] + v[:, 1]) * d[0] + v[:, 0]]
            w = u[s:s + (1 << 25)]
            # types 1 and 3 share what type 2 leaves in their own ratio
            ea = (1.0 - ENRICHED) * a / (a + FRACTIONS[2])
            e = 1 + (w >= ea).to(torch.uint8) + (w >= ea + ENRICHED).to(torch.uint8)
            t[s:s + (1 << 25)] = torch.where(m, e, t[s:s + (1 << 25)])
    return t


def _surface(xyz, r0, r1, h):
    """Squared distance to the analytic surface of the solid."""
    rho = torch.hypot(xyz[:, 0], xyz[:, 1])
    z = xyz[:, 2]
    lat = (r0 + (r1 - r0) * (z / h) - rho) * (h / math.hypot(h, r0 - r1))
    return torch.minimum(torch.minimum(z, h - z), lat).clamp_(min=0.0).square_()


_ctx = None


def _context():
    """One context per program, as pp_spatstat_create's callers keep it."""
    global _ctx
    if _ctx is None:
        _ctx = SpatStat(0)
    return _ctx


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _cloud(n, shape, density, clustered, gen, widths=()):
    r0, r1, h = _shape(n, shape, density)
    xyz = _points(n, r0, r1, h, gen)
    ty = _types(xyz, r0, r1, h, round(2500e-6 * n) if clustered else 0, gen)
    s2 = _surface(xyz, r0, r1, h)
    torch.cuda.synchronize()
    c = _context().upload_device(xyz.data_ptr(), ty.data_ptr(), s2.data_ptr(), n,
                                 widths[0] if widths else 0.0)
    for w in widths[1:]:
        c.add_cell_list(w)
    return c


def _job(case):
    fam = 0
    for f in case["families"].split("+"):
        fam |= FAMILIES[f]
    k = list(range(1, case["kmax"] + 1)) if "MKNN" in case["families"] else []
    return Job(TASKS[case["tasks"]], 0.0, case["rincr"], case["rmax"], fam, kvalues=k)


def _hull(case, r0, r1, h):
    return synth.hull("frustum", r0, r1, h, case["nseg"], case["nz"])


def _records(xyz, ty, gen):
    """POS records: big-endian x, y, z, mass-to-charge; a few per cent of the
    mass-to-charge values lie in no range."""
    n = xyz.shape[0]
    rec = torch.empty((n, 4), device="cuda")
    rec[:, :3] = xyz
    m = torch.tensor([0.0, *MASSES], device="cuda")[ty.long()]
    rec[:, 3] = m + 0.04 * torch.randn(n, generator=gen, device="cuda")
    return rec.view(torch.uint8).reshape(n, 4, 4).flip(2).contiguous()


class _State:
    """What one case's program holds; clouds and servers are given back with it."""

    def __init__(self, case):
        self.case = case
        self.clouds = []
        self.server = None

    def __del__(self):
        if self.server is not None:
            self.server.close()
        for c in self.clouds:
            c.free()


def prepare(case, seed):
    gen = _generator(seed)
    s = _State(case)
    kind = case["kind"]
    if kind == "spatstat":
        s.clouds.append(_cloud(case["n"], case["shape"], case["density"], case["clustered"], gen))
        s.job = _job(case)
    elif kind == "batch":
        spec = workloads.batch_spec(case["count"], case["spec"], case["nmin"], case["nmax"])
        for it in spec:
            s.clouds.append(_cloud(it.n, "frustum", 27.3, it.clustered, gen))
        s.jobs = [it.job for it in spec]
    elif kind == "serve":
        for i in range(case["tips"]):  # the widths the service keeps resident
            s.clouds.append(_cloud(case["nmin"] << i, "frustum", 27.3, True, gen,
                                   (1.0, 1.3, 0.6)))
        s.requests = workloads.serve_stream(case["requests"], 50.0, case["tips"], case["stream"])
        s.server = Server(_context(), slots=2)
    elif kind == "npcorr":
        s.clouds.append(_cloud(case["n"], "frustum", 27.3, True, gen))
    else:
        r0, r1, h = _shape(case["n"], "frustum", 27.3)
        # inside the hull's polygon, whose edges lie within the circle
        inset = math.cos(math.pi / case["nseg"]) * (1.0 - 1e-5) if "nseg" in case else 1.0
        xyz = _points(case["n"], r0, r1, h, gen, inset)
        if kind == "ion2surf":
            s.xyz = xyz
            s.tri = torch.from_numpy(_hull(case, r0, r1, h)).cuda()
            s.out = torch.empty(case["n"], device="cuda")
        else:
            ty = _types(xyz, r0, r1, h, round(2500e-6 * case["n"]), gen)
            s.rec = _records(xyz, ty, gen)
            if kind == "pos":
                s.xyz = torch.empty_like(xyz)
                s.mq = torch.empty(case["n"], device="cuda")
                s.ty = torch.empty(case["n"], dtype=torch.uint8, device="cuda")
            else:
                s.rec = s.rec.cpu().numpy().tobytes()
                s.tri = _hull(case, r0, r1, h)
                s.job = _job(case)
        torch.cuda.synchronize()
    return s


def _outputs(r):
    return [*r.arrays().values(), r.centers_considered, r.pairs_inball]


def run(state):
    case, kind = state.case, state.case["kind"]
    ctx = _context()
    if kind == "spatstat":
        return _outputs(ctx.run(state.clouds[0], state.job))
    if kind == "batch":
        res = ctx.run_batch(state.clouds, state.jobs)
        return [[r.rdf, r.mknn] for r in res]
    if kind == "serve":
        at = {state.server.submit(state.clouds[q.cloud], q.job): i
              for i, q in enumerate(state.requests)}
        state.server.drain()
        out = [None] * len(at)
        for ticket, status, r in state.server.poll():
            if status != 0:
                raise RuntimeError(f"request failed with status {status}")
            out[at[ticket]] = r.mknn if r.rdf is None else r.rdf
        return out
    if kind == "npcorr":
        return ctx.npcorr(state.clouds[0], TASKS["npc"], case["rmax"], case["rincr"],
                          case["order"])
    if kind == "ion2surf":
        ctx.ion2surf_device(state.xyz.data_ptr(), case["n"], state.tri.data_ptr(),
                            state.tri.shape[0], case["radius"], state.out.data_ptr())
        return state.out
    if kind == "pos":
        ctx.pos_decode_device(state.rec.data_ptr(), 16 * case["n"], RANGES,
                              state.xyz.data_ptr(), state.mq.data_ptr(), state.ty.data_ptr())
        return [state.xyz, state.mq, state.ty]
    cloud = ctx.cloud_from_pos(state.rec, RANGES, state.tri, case["rmax"])
    try:
        return _outputs(ctx.run(cloud, state.job))
    finally:
        cloud.free()


# ---------------------------------------------------------------------------

def _spatstat_work(n, density, tasks, job, shape="frustum"):
    """17 bytes an ion, the histograms, and one distance (8 operations) for
    each pair within Rmax of a center of the tasks' types, a pair of two
    centers of one type once."""
    frac = {t: f for t, f in zip((1, 2, 3), FRACTIONS)}
    r0, r1, h = _shape(n, shape, density)
    R = job.rmax
    hi = max(h - 2 * R, 0.0)
    a, b = max(r0 - R, 0.0), max(r1 - R, 0.0)
    centers = density * math.pi / 3.0 * hi * (a * a + a * b + b * b)
    ball = density * 4.0 / 3.0 * math.pi * R ** 3
    pairs = 0.0
    for t in {t for trg, _ in tasks for t in trg}:
        env = {e for trg, en in tasks for e in en if t in trg}
        pairs += centers * frac.get(t, 0.0) * ball * sum(
            frac.get(e, 0.0) * (0.5 if e == t else 1.0) for e in env)
    nh = sum(len(tasks) * (len(job.kvalues) if f == FAM_MKNN else 1)
             for f in (FAM_RDF, FAM_1NN, FAM_RIPK, FAM_MKNN) if job.families & f)
    bins = hist_geometry(job.rmin, job.rincr, job.rmax) + 2
    return 17.0 * n + 8.0 * nh * bins, 8.0 * max(pairs, 1.0)


def work(case):
    kind = case["kind"]
    if kind == "spatstat":
        by, fl = _spatstat_work(case["n"], case["density"], TASKS[case["tasks"]], _job(case),
                                case["shape"])
    elif kind == "batch":
        by = fl = 0.0
        for it in workloads.batch_spec(case["count"], case["spec"], case["nmin"], case["nmax"]):
            b, f = _spatstat_work(it.n, 27.3, it.job.tasks, it.job)
            by, fl = by + b, fl + f
    elif kind == "serve":
        by = fl = 0.0
        for q in workloads.serve_stream(case["requests"], 50.0, case["tips"], case["stream"]):
            b, f = _spatstat_work(case["nmin"] << q.cloud, 27.3, q.job.tasks, q.job)
            by, fl = by + b, fl + f
    elif kind == "npcorr":
        # the ions, the cubes, and a distance for each neighbour up to the
        # order-th of each center and task
        edge = 1 + 2 * (math.ceil(case["rmax"] / case["rincr"]) + 1)
        by = 17.0 * case["n"] + 4.0 * 4 * edge ** 3
        fl = 8.0 * case["n"] * 2 * (case["order"] + 1)
    elif kind == "ion2surf":
        # the ions and triangles once, a distance (about 60 operations) to at
        # least one triangle for each ion
        by = 16.0 * case["n"] + 36.0 * (2 * case["nseg"] * (case["nz"] + 1))
        fl = 60.0 * case["n"]
    elif kind == "pos":
        by, fl = 33.0 * case["n"], 5.0 * case["n"]
    else:
        by, fl = _spatstat_work(case["n"], 27.3, TASKS[case["tasks"]], _job(case))
        by, fl = by + 33.0 * case["n"], fl + 60.0 * case["n"]
    return {"bytes": by, "flops": fl}


def exact(case, seed):
    """Histograms, counts and cubes are whole numbers.  The decoded floats and
    the distances of ions inside a convex hull (to its nearest facet plane, at
    most the radius) have values in 64 bits."""
    kind = case["kind"]
    if kind == "pos":
        s = prepare(case, seed)
        v = s.rec.flip(2).contiguous().view(torch.float32).reshape(-1, 4).double()
        return [v[:, :3].contiguous(), v[:, 3].contiguous(), None]
    if kind != "ion2surf":
        return None
    s = prepare(case, seed)
    tri = s.tri.double().reshape(-1, 3, 3)
    if case["n"] * tri.shape[0] > 5e11:
        return None
    nrm = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    off = (nrm * tri[:, 0]).sum(1)
    out = torch.empty(case["n"], dtype=torch.float64, device="cuda")
    step = max(1, int(2e9) // (8 * tri.shape[0]))
    nt = nrm.t().contiguous()
    for a in range(0, case["n"], step):
        out[a:a + step] = torch.addmm(-off[None, :], s.xyz[a:a + step].double(),
                                      nt).abs_().amin(1)
    return out.square_().clamp_(max=float(np.float32(case["radius"])) ** 2)
