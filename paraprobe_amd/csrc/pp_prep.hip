// pp_prep.hip -- the center lists and query tiles of a whole run of jobs in a
// fixed number of launches.
//
// A run (one job, a batch, a serving batch, or the full-range rerun of the
// short centers) is a sequence of segments, one per (job, center type): the
// considered centers of segment q are the ions of its job's cell-sorted list
// whose type has slot q.slot and whose ion2surf is at least fl32(R^2)
// (src/PARAPROBE_SolverHdl.cpp:3846-3860), or the ions a rerun selection
// flags.  All segments' ion ranges are laid end to end (the ion space, ion0
// onwards for segment q), each padded to whole blocks of kPrepTile, and so are
// their cell ranges (the cell space, cell0 onwards), so that no block spans
// segments.  Five launches: one pass over each job's ions sets a bit per
// (segment, ion) and counts it per 64 ions and per block for all of the job's
// segments at once; a one-block scan turns the block counts into offsets;
// then the compaction into the run's center list (segment after segment, each
// in cell order) and, in the same launch, the tiles per cell with their
// in-block prefix; a second scan; and the tiles -- up to T centers of one
// segment in one cell, first center as an index into the run's center list --
// with each job's largest stencil candidate count and its parts of the lists.
//
// What bounds it: reading 20 bytes an ion once (it was once per segment, with
// a 4-byte flag and a 4-byte scanned position for each written and read
// again), and for small runs the number of launches, 5 instead of 12.  A
// whole call, before and after: 20,000 ions with three center types 303 and
// 283 us, a batch of 24 jobs of 50,000 to 2,000,000 ions 7.73 and 7.20 ms, 100
// million ions with one center type 423 and 415 ms.  A run of many small jobs is
// bound by its blocks' first loads: the segment of a block is looked up in a list
// that the first launch writes (bisecting the segments in every block took
// 0.65 ms for 27,000 segments of 27 cells).
#include "pp_launch.h"

namespace pp {

namespace {

constexpr int kPrepBlock = 256;
constexpr int kPrepItems = kPrepTile / kPrepBlock;
constexpr int kPrepWords = kPrepTile / 64;  // 64-ion words of a block

// the last k in [0, n) with start(k) <= b (starts ascending, start(0) <= b),
// by the block's first thread
template <typename Start>
__device__ inline int find_last(uint64_t b, int n, Start start, int *s_q)
{
    if (threadIdx.x == 0) {
        int lo = 0, hi = n;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (start(mid) <= b)
                lo = mid;
            else
                hi = mid;
        }
        *s_q = lo;
    }
    __syncthreads();
    return *s_q;
}

// centers before element e of the ion space
__device__ inline uint32_t center_pos(const PrepLists &l, uint64_t e)
{
    uint32_t p = l.boff[e / kPrepTile];
    if (e % kPrepTile) {  // (at a block's start, or at the space's end, that is all)
        const uint64_t w = e >> 6;
        p += l.wpos[w] + (uint32_t)__builtin_popcountll(l.bits[w] & ((1ull << (e & 63)) - 1ull));
    }
    return p;
}

// One block per kPrepTile ions of a job, for all of the job's segments.
__global__ __launch_bounds__(kPrepBlock) void k_pflags(const PrepSeg *__restrict__ segs, int nseg,
                                                        uint32_t nion,
                                                        const int32_t *__restrict__ jseg, int njobs,
                                                        PrepLists l, PrepJobStat *__restrict__ js)
{
    __shared__ int s_q;
    __shared__ uint64_t s_bits[kMaxTrg][kPrepWords];
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < njobs; k += kPrepBlock)
            js[k].maxcand = 0u;
    // the segment of each block of the ion space and of the cell space
    for (int q = blockIdx.x; q < nseg; q += gridDim.x) {
        const PrepSeg &Q = segs[q];
        const uint64_t ib = Q.ion0 / kPrepTile, cb = nion + Q.cell0 / kPrepTile;
        const uint32_t in = (uint32_t)(((uint64_t)Q.n + kPrepTile - 1) / kPrepTile);
        const uint32_t cn = (uint32_t)(((uint64_t)Q.nc + kPrepTile - 1) / kPrepTile);
        for (uint32_t k = threadIdx.x; k < in; k += kPrepBlock)
            l.seg[ib + k] = (uint32_t)q;
        for (uint32_t k = threadIdx.x; k < cn; k += kPrepBlock)
            l.seg[cb + k] = (uint32_t)q;
    }
    // (a job without segments starts where the next one does and owns no block)
    const int j = find_last(blockIdx.x, njobs, [&](int k) {
        return jseg[k] < jseg[njobs] ? (uint64_t)segs[jseg[k]].jblk0 : ~0ull; }, &s_q);
    const int q0 = jseg[j], ns = jseg[j + 1] - q0;
    const PrepSeg S = segs[q0];  // by value: kept in registers, not re-read
    if (S.n == 0)
        return;  // no ions at all: the one block is here for the counters
    const uint32_t b0 = (blockIdx.x - S.jblk0) * (uint32_t)kPrepTile;
    const int lane = threadIdx.x & 63, wid = threadIdx.x / 64;
    int ts[kPrepItems];
#pragma unroll
    for (int k = 0; k < kPrepItems; ++k) {
        const uint64_t i = (uint64_t)b0 + (uint64_t)(k * kPrepBlock) + threadIdx.x;
        ts[k] = -1;
        if (i < S.n && (S.src ? S.src[i] != 0u : S.s2[i] >= S.R2))
            ts[k] = S.trgslot[__float_as_uint(S.pos[i].w) & 0xFFu];
    }
    // (the segments of a job are its center type slots in order)
    for (int q = 0; q < ns; ++q) {
#pragma unroll
        for (int k = 0; k < kPrepItems; ++k) {
            const uint64_t m = __ballot(ts[k] == q);
            if (lane == 0)
                s_bits[q][k * (kPrepBlock / 64) + wid] = m;
        }
    }
    __syncthreads();
    static_assert(kPrepWords == 32, "one word per lane of half a wavefront");
    for (int q = wid; q < ns; q += kPrepBlock / 64) {
        const uint64_t m = lane < kPrepWords ? s_bits[q][lane] : 0ull;
        const uint32_t n = (uint32_t)__builtin_popcountll(m);
        uint32_t incl = n;
        for (int d = 1; d < kPrepWords; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
            if (lane >= d)
                incl += o;
        }
        const uint64_t w = (segs[q0 + q].ion0 + b0) / 64 + (uint64_t)lane;
        if (lane < kPrepWords) {
            l.bits[w] = m;
            l.wpos[w] = incl - n;
        }
        if (lane == kPrepWords - 1)
            l.boff[(segs[q0 + q].ion0 + b0) / kPrepTile] = incl;
    }
}

// Exclusive scan of n block counts in place, the total at index n; one block
// (a block count stands for kPrepTile elements, so there are few).
__global__ __launch_bounds__(1024) void k_pscan(uint32_t *__restrict__ v, uint32_t n)
{
    __shared__ uint32_t s_w[16];
    const int lane = threadIdx.x & 63, wid = threadIdx.x / 64;
    uint32_t carry = 0;
    for (uint32_t b = 0; b < n; b += 4096) {
        const uint32_t i = b + threadIdx.x * 4u;
        uint32_t a[4], tot = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            a[k] = i + (uint32_t)k < n ? v[i + (uint32_t)k] : 0u;
            tot += a[k];
        }
        uint32_t incl = tot;
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
            if (lane >= d)
                incl += o;
        }
        if (lane == 63)
            s_w[wid] = incl;
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            const uint32_t x = s_w[w];
            before += w < wid ? x : 0u;
            all += x;
        }
        uint32_t run = carry + before + incl - tot;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (i + (uint32_t)k < n)
                v[i + (uint32_t)k] = run;
            run += a[k];
        }
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0)
        v[n] = carry;
}

// Blocks below nion: the centers of one block of the ion space (job-local
// sorted ion indices); the others: the tiles per cell of one block of the
// cell space, as their prefix in the block and the block's total.
__global__ __launch_bounds__(kPrepBlock) void k_pcompact(const PrepSeg *__restrict__ segs,
                                                          uint32_t nion, PrepLists l,
                                                          uint32_t *__restrict__ centers)
{
    __shared__ uint32_t s_w[kPrepBlock / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x / 64;
    if (blockIdx.x < nion) {
        const uint64_t e0 = (uint64_t)blockIdx.x * kPrepTile;
        const uint32_t i0 = (uint32_t)(e0 - segs[l.seg[blockIdx.x]].ion0), off = l.boff[blockIdx.x];
        for (int k = 0; k < kPrepItems; ++k) {
            const uint64_t w = e0 / 64 + (uint64_t)(k * (kPrepBlock / 64) + wid);
            const uint64_t m = l.bits[w];
            if ((m >> lane) & 1ull)
                centers[off + l.wpos[w] +
                        (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull))] =
                    i0 + (uint32_t)(k * kPrepBlock) + threadIdx.x;
        }
        return;
    }
    const uint32_t cb = blockIdx.x - nion;
    const uint64_t e0 = (uint64_t)cb * kPrepTile;
    const PrepSeg S = segs[l.seg[blockIdx.x]];
    const uint64_t c0 = e0 - S.cell0 + (uint64_t)threadIdx.x * kPrepItems;
    uint32_t cnt[kPrepItems], tot = 0;
    uint32_t lo = c0 < S.nc ? center_pos(l, S.ion0 + S.cellstart[c0]) : 0u;
#pragma unroll
    for (int k = 0; k < kPrepItems; ++k) {
        cnt[k] = 0;
        if (c0 + (uint64_t)k < S.nc) {
            const uint32_t hi = center_pos(l, S.ion0 + S.cellstart[c0 + (uint64_t)k + 1u]);
            cnt[k] = (hi - lo + (uint32_t)S.T - 1u) / (uint32_t)S.T;
            lo = hi;
        }
        tot += cnt[k];
    }
    uint32_t incl = tot;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
        if (lane >= d)
            incl += o;
    }
    if (lane == 63)
        s_w[wid] = incl;
    __syncthreads();
    uint32_t run = incl - tot, all = 0;
    for (int w = 0; w < kPrepBlock / 64; ++w) {
        run += w < wid ? s_w[w] : 0u;
        all += s_w[w];
    }
#pragma unroll
    for (int k = 0; k < kPrepItems; ++k) {
        if (c0 + (uint64_t)k < S.nc)
            l.tpre[S.tp0 + c0 + (uint64_t)k] = run;
        run += cnt[k];
    }
    if (threadIdx.x == 0)
        l.toff[cb] = all;
}

// stencil row rw around cell (cx, cy, cz): its candidate range, empty when
// the row lies outside the grid
__device__ inline uint32_t row_count(const Row &rw, int cx, int cy, int cz, const GridGeom &g,
                                     const uint32_t *__restrict__ cellstart)
{
    const int y = cy + rw.dy, z = cz + rw.dz;
    if (y < 0 || y >= g.ny || z < 0 || z >= g.nz)
        return 0u;
    const int x0 = cx - rw.dxm < 0 ? 0 : cx - rw.dxm;
    const int x1 = cx + rw.dxm >= g.nx ? g.nx - 1 : cx + rw.dxm;
    const uint64_t k0 = ((uint64_t)z * g.ny + y) * g.nx + x0;
    return cellstart[k0 + (uint32_t)(x1 - x0) + 1u] - cellstart[k0];
}

// The tiles of every cell with centers, and each job's largest stencil
// candidate count (a bound on any center's neighbour count); the first block
// also writes each job's parts of the run's lists.
__global__ __launch_bounds__(kPrepBlock) void k_ptilewrite(const PrepSeg *__restrict__ segs,
                                                            uint32_t nion, uint32_t ncell,
                                                            uint32_t per,
                                                            const int32_t *__restrict__ jseg,
                                                            int njobs, PrepLists l,
                                                            Tile *__restrict__ tiles,
                                                            PrepJobStat *__restrict__ js)
{
    if (blockIdx.x == 0)
        for (int j = threadIdx.x; j < njobs; j += kPrepBlock) {
            const int a = jseg[j], b = jseg[j + 1];
            uint32_t c0 = 0, c1 = 0, t0 = 0, t1 = 0;
            if (a < b) {
                // (a segment's blocks are its own, so the next one's offset
                // is where it ends)
                const PrepSeg &F = segs[a], &L = segs[b - 1];
                c0 = l.boff[F.ion0 / kPrepTile];
                c1 = l.boff[(L.ion0 + L.n + kPrepTile - 1) / kPrepTile];
                t0 = l.toff[F.cell0 / kPrepTile];
                t1 = l.toff[(L.cell0 + L.nc + kPrepTile - 1) / kPrepTile];
            }
            js[j].center0 = c0;
            js[j].centers = c1 - c0;
            js[j].tile0 = t0;
            js[j].tiles = t1 - t0;
        }
    // block blockIdx.x / per of the cell space, every per-th kPrepBlock of its cells
    const uint32_t cb = blockIdx.x / per;
    if (cb >= ncell)
        return;
    const PrepSeg S = segs[l.seg[nion + cb]];  // by value: kept in registers, not re-read
    for (uint32_t it = blockIdx.x % per; it < (uint32_t)kPrepItems; it += per) {
        const uint64_t cw = (uint64_t)cb * kPrepTile + it * (uint32_t)kPrepBlock - S.cell0;
        if (cw >= S.nc)
            return;
        const uint64_t c = cw + threadIdx.x;
        // every lane stays to the wave's reduction below
        uint32_t tot = 0;
        if (c < S.nc) {
            const uint32_t lo = center_pos(l, S.ion0 + S.cellstart[c]),
                           hi = center_pos(l, S.ion0 + S.cellstart[c + 1]);
            if (hi > lo) {
                const uint32_t T = (uint32_t)S.T, cnt = hi - lo;
                const uint32_t t0 = l.toff[cb] + l.tpre[S.tp0 + c];
                for (uint32_t m = 0; m * T < cnt; ++m) {
                    Tile t;
                    t.key = (uint32_t)c;
                    t.first = lo + m * T;
                    const uint32_t left = cnt - m * T;
                    t.count = (uint16_t)(left < T ? left : T);
                    t.job = (uint16_t)S.job;
                    t.pad = (uint32_t)S.slot;
                    tiles[t0 + m] = t;
                }
                const int cx = (int)(c % (uint64_t)S.g.nx);
                const int cy = (int)((c / (uint64_t)S.g.nx) % (uint64_t)S.g.ny);
                const int cz = (int)(c / ((uint64_t)S.g.nx * (uint64_t)S.g.ny));
#pragma unroll 4
                for (int r = 0; r < S.nrows; ++r)
                    tot += row_count(S.rows[r], cx, cy, cz, S.g, S.cellstart);
            }
        }
        // one atomic per wavefront (a block's cells belong to one job)
        for (int d = 32; d > 0; d >>= 1) {
            const uint32_t o = (uint32_t)__shfl_xor((int)tot, d, 64);
            tot = o > tot ? o : tot;
        }
        if ((threadIdx.x & 63) == 0 && tot > 0)
            atomicMax(&js[S.job].maxcand, tot);
    }
}

} // namespace

PrepWords prep_words(uint64_t E, uint64_t Ec, uint64_t nc)
{
    PrepWords w;
    w.bits = E / 32;
    w.wpos = E / 64;
    w.boff = E / kPrepTile + 1;
    w.tpre = nc;
    w.toff = Ec / kPrepTile + 1;
    w.seg = E / kPrepTile + Ec / kPrepTile;
    return w;
}

hipError_t launch_prep(const PrepLaunch &p, hipStream_t s)
{
    if (p.nseg <= 0 || p.njobs <= 0)
        return hipSuccess;
    const uint32_t nion = (uint32_t)(p.E / kPrepTile), ncell = (uint32_t)(p.Ec / kPrepTile);
    hipError_t e;
    hipLaunchKernelGGL(k_pflags, dim3(p.jblocks ? p.jblocks : 1), dim3(kPrepBlock), 0, s, p.segs, p.nseg,
                       nion, p.jseg, p.njobs, p.l, p.js);
    if ((e = hipGetLastError()) != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_pscan, dim3(1), dim3(1024), 0, s, p.l.boff, nion);
    if ((e = hipGetLastError()) != hipSuccess)
        return e;
    if (nion + ncell > 0) {
        hipLaunchKernelGGL(k_pcompact, dim3(nion + ncell), dim3(kPrepBlock), 0, s, p.segs, nion,
                           p.l, p.centers);
        if ((e = hipGetLastError()) != hipSuccess)
            return e;
    }
    hipLaunchKernelGGL(k_pscan, dim3(1), dim3(1024), 0, s, p.l.toff, ncell);
    if ((e = hipGetLastError()) != hipSuccess)
        return e;
    // workgroups for a block of the cell space: one per kPrepBlock of its cells,
    // or, where these are more padding than cells and the blocks fill the device
    // without, one
    const uint32_t per = ncell > 1024u && 2 * p.nc < p.Ec ? 1u : (uint32_t)kPrepItems;
    hipLaunchKernelGGL(k_ptilewrite, dim3(ncell ? ncell * per : 1), dim3(kPrepBlock), 0, s,
                       p.segs, nion, ncell, per, p.jseg, p.njobs, p.l, p.tiles, p.js);
    return hipGetLastError();
}

} // namespace pp
