// fipc_broad.hip -- spatial-hash broad phase and everything built on it:
// constraint search (NEWTON_IPC.py:159-357), CCD step filters (:377-468) and
// the collision check (:855-886).
//
// Grid: every inserted item is entered in each cell its box overlaps
// (cell size = 1 / inv_dx, as the reference's hash).  Entries are grouped by
// a hashed bucket; each entry keeps its exact 63-bit cell key and three bits
// telling whether the cell is the item's lowest cell along x, y, z.  A wave of
// a query takes up to 64 (query box, cell) pairs and runs over their cells'
// entries laid end to end, so neither huge boxes nor crowded cells serialise
// it; an entry is accepted only in the first cell common to both boxes, so
// every pair is tested exactly once.  Builds and queries size their
// buffers from capacities and never wait for the host; each operation
// synchronises once at its end and is redone when a capacity was exceeded.
#include <hip/hip_runtime.h>
#include <rocprim/device/device_merge_sort.hpp>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_select.hpp>
#include <algorithm>
#include <vector>
#include "fipc_ctx.h"
#include "fipc_rows.h"

using namespace fipc;

#define TPB 256
static inline int nblk(long n, int t = TPB) { return (int)((n + t - 1) / t); }


struct CellRange { int lo[3], hi[3]; };
__device__ __forceinline__ CellRange cells_of(v3 lo, v3 hi, double inv)
{
    CellRange r;
    r.lo[0] = (int)floor(lo.x * inv); r.lo[1] = (int)floor(lo.y * inv); r.lo[2] = (int)floor(lo.z * inv);
    r.hi[0] = (int)floor(hi.x * inv); r.hi[1] = (int)floor(hi.y * inv); r.hi[2] = (int)floor(hi.z * inv);
    return r;
}
__device__ __forceinline__ long long ncells(const CellRange& r)
{
    return (long long)(r.hi[0] - r.lo[0] + 1) * (r.hi[1] - r.lo[1] + 1) * (r.hi[2] - r.lo[2] + 1);
}
__device__ __forceinline__ unsigned long long cell_key(int i, int j, int k)
{
    const long long B = 1 << 20;
    return ((unsigned long long)(i + B) << 42) | ((unsigned long long)(j + B) << 21) | (unsigned long long)(k + B);
}
// bucket of a cell: splitmix64 finaliser of the exact cell key, so that the
// axis-aligned rows and planes of cells that lattice meshes produce spread
// evenly over a power-of-two table
__device__ __forceinline__ unsigned bucket_of(int i, int j, int k, unsigned M)
{
    unsigned long long z = cell_key(i, j, k) + 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (unsigned)z & (M - 1);
}

// ---- boxes ---------------------------------------------------------------
// kind of primitive: 0 boundary point, 1 boundary edge, 2 boundary triangle.
// sol != nullptr gives the swept box of x and x + sol.
struct BoxFn {
    const double* x;
    const double* sol;
    const int* idx;
    int kind;
    double infl;
    __device__ __forceinline__ void operator()(int i, v3& lo, v3& hi) const
    {
        int nvx = kind + 1;
        lo = mk(1e300, 1e300, 1e300);
        hi = mk(-1e300, -1e300, -1e300);
        for (int a = 0; a < nvx; a++) {
            int v = idx[nvx * i + a];
            v3 p = ldv(x, v);
            lo = vmin(lo, p);
            hi = vmax(hi, p);
            if (sol) {
                v3 q = p + ldv(sol, v);
                lo = vmin(lo, q);
                hi = vmax(hi, q);
            }
        }
        lo = lo - mk(infl, infl, infl);
        hi = hi + mk(infl, infl, infl);
    }
};

// Single-precision boxes around the double ones, for rejecting pairs before
// their vertices are loaded: rounded outward with a margin of a few units, and
// the query's widened by 1e-9 dHat (run_query), so a pair that the visitor's own
// box test in doubles accepts, up to that test's rounding, always passes.
struct FBox { float lo[3], hi[3]; int v[2]; };  // 32 bytes; v: an item's vertices (a point's twice)
__device__ __forceinline__ float f_down(double v) { const float f = (float)v; return f - fmaxf(fabsf(f) * 3e-7f, 1e-37f); }
__device__ __forceinline__ float f_up(double v) { const float f = (float)v; return f + fmaxf(fabsf(f) * 3e-7f, 1e-37f); }
__device__ __forceinline__ FBox fbox_of(v3 lo, v3 hi)
{
    return FBox{{f_down(lo.x), f_down(lo.y), f_down(lo.z)}, {f_up(hi.x), f_up(hi.y), f_up(hi.z)}, {-1, -1}};
}
// What the query kernel needs of a query, written by the pass that counts its
// cells: box, vertices (the last repeated), lowest cell and extents along y, z.
struct QInfo { float lo[3], hi[3]; int v[3], clo[3], ny, nz, pad[2]; };  // 64 bytes

#define GRID_MAXB 2048
static inline int stride_grid(long n) { return std::max(1, std::min(nblk(n), GRID_MAXB)); }

// ---- two-level offsets ----------------------------------------------------
// The entries of n boxes (one per overlapped cell) are numbered without a
// device-wide scan: k_count_cells stores each box's offset within its block
// of TPB boxes (loc) and the block's total (part); a consumer workgroup
// prefix-sums the ≤ OFF_PMAX block totals in LDS, and the offset of box i is
// P[i / TPB] + loc[i].  Saves a scan launch pair per grid build and query.
constexpr int OFF_PMAX = 8192;  // block totals per table: up to 2M boxes (32 KB of LDS)

// exclusive prefix of v over the workgroup (TPB threads), *total = the sum
__device__ __forceinline__ long long block_exscan(long long v, long long* total)
{
    __shared__ long long wsum[TPB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    long long x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        long long y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    long long before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < TPB / 64; k++) {
        if (k < w) before += wsum[k];
        all += wsum[k];
    }
    __syncthreads();
    *total = all;
    return before + x - v;
}
// cells of every box: loc[i] = offset of box i within its block, part[b] =
// the block's total; a box over more than 2^24 cells, or a block over 2^30,
// flags GF_HUGE (the operation fails with FIPC_ERR_CAPACITY)
// (a grid build also keeps the boxes in single precision, ibox; a query its
// QInfo, with the box widened by slack)
__global__ void __launch_bounds__(TPB) k_count_cells(int n, BoxFn box, double inv, int* loc, int* part, int* flag,
                                                     FBox* ibox, int* zero, long nzero, QInfo* qinfo, double slack)
{
    const int i = blockIdx.x * TPB + threadIdx.x;
    // a grid build clears its bucket counts here (the fill adds to them)
    for (long k = i; k < nzero; k += (long)gridDim.x * TPB) zero[k] = 0;
    long long c = 0;
    if (i < n) {
        v3 lo, hi;
        box(i, lo, hi);
        if (ibox) {
            FBox b = fbox_of(lo, hi);
            const int nvx = box.kind + 1;  // items are points and edges
            b.v[0] = box.idx[nvx * i];
            b.v[1] = box.idx[nvx * i + nvx - 1];
            ibox[i] = b;
        }
        const CellRange cr = cells_of(lo, hi, inv);
        c = ncells(cr);
        if (qinfo) {
            const FBox b = fbox_of(lo - mk(slack, slack, slack), hi + mk(slack, slack, slack));
            QInfo q;
            const int nvx = box.kind + 1;
            for (int d = 0; d < 3; d++) {
                q.lo[d] = b.lo[d];
                q.hi[d] = b.hi[d];
                q.v[d] = box.idx[nvx * i + min(d, nvx - 1)];
                q.clo[d] = cr.lo[d];
            }
            q.ny = cr.hi[1] - cr.lo[1] + 1;
            q.nz = cr.hi[2] - cr.lo[2] + 1;
            q.pad[0] = q.pad[1] = 0;
            qinfo[i] = q;
        }
        if (c > (1 << 24) || c < 0) { atomicOr(flag, GF_HUGE); c = 0; }
    }
    long long tot;
    const long long pre = block_exscan(c, &tot);
    if (tot >= (1LL << 30)) {
        if (threadIdx.x == 0) atomicOr(flag, GF_HUGE);
        tot = 0;
    }
    if (i < n) loc[i] = (int)pre;
    if (threadIdx.x == 0) part[blockIdx.x] = (int)tot;
}
// sP[0..np] = exclusive prefix of part[0..np) in LDS (every thread of the
// workgroup calls it); returns the total, or -1 past 2^31 - 1
__device__ int lds_prefix(const int* __restrict__ part, int np, int* sP)
{
    for (int k = threadIdx.x; k < np; k += TPB) sP[k] = part[k];
    __syncthreads();
    const int per = (np + TPB - 1) / TPB, k0 = min(np, (int)threadIdx.x * per), k1 = min(np, k0 + per);
    long long sum = 0;
    for (int k = k0; k < k1; k++) sum += sP[k];
    long long tot;
    long long pre = block_exscan(sum, &tot);
    if (tot > 0x7fffffffLL) tot = -1, pre = 0;
    for (int k = k0; k < k1; k++) {
        const int v = sP[k];
        sP[k] = (int)pre;
        pre += v;
    }
    __syncthreads();
    return (int)tot;
}
// the box whose entries hold entry e (0 <= e < total): the last box with
// offset <= e (boxes with no cells share the next box's offset); *first = its
// first entry
__device__ __forceinline__ int find_box(int e, const int* sP, int np, const int* __restrict__ loc, int n, int* first)
{
    int lo = 0, hi = np;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (sP[mid] <= e) lo = mid; else hi = mid;
    }
    const int r = e - sP[lo];
    int l = lo * TPB, h = min(n, l + TPB);
    while (h - l > 1) {
        const int mid = (l + h) >> 1;
        if (loc[mid] <= r) l = mid; else h = mid;
    }
    *first = sP[lo] + loc[l];
    return l;
}

// Grid-stride over the entries (their number is the sum of the block totals,
// so the host never waits for it).  A count above the capacity flags a retry
// and records the count needed; workgroup 0 stores the count to part[np]
// for the scatter.  The owning item of an entry is found by binary search
// in the offsets, so an item covering thousands of cells (a long plate edge)
// does not serialise a wave.  Dynamic LDS: (np + 1) ints.
__global__ void __launch_bounds__(TPB) k_grid_fill(int n, int np, int cap, BoxFn box, double inv, unsigned M,
                                                   const int* __restrict__ loc, int* part, unsigned* ekey,
                                                   int* eitem, unsigned long long* ecell, int* bcount, int* flag)
{
    extern __shared__ int sP[];
    const int ne = lds_prefix(part, np, sP);
    if (blockIdx.x == 0 && threadIdx.x == 0) part[np] = ne;
    if (ne > cap || ne < 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            atomicOr(flag, ne < 0 ? GF_HUGE : GF_RETRY);
            atomicMax(flag + 2, ne);
        }
        return;
    }
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < ne; e += gridDim.x * blockDim.x) {
        int first;
        const int i = find_box(e, sP, np, loc, n, &first);
        v3 blo, bhi;
        box(i, blo, bhi);
        CellRange r = cells_of(blo, bhi, inv);
        int ny = r.hi[1] - r.lo[1] + 1, nz = r.hi[2] - r.lo[2] + 1;
        int l = e - first;
        int a = r.lo[0] + l / (ny * nz), b = r.lo[1] + (l / nz) % ny, c = r.lo[2] + l % nz;
        unsigned flags = (a == r.lo[0] ? 1u : 0u) | (b == r.lo[1] ? 2u : 0u) | (c == r.lo[2] ? 4u : 0u);
        unsigned k = bucket_of(a, b, c, M);
        ekey[e] = k;
        eitem[e] = (int)((unsigned)i | (flags << 28));
        ecell[e] = cell_key(a, b, c);
        atomicAdd(&bcount[k], 1);
    }
}
// bstart holds the scanned bucket starts; each entry takes the next slot of
// its bucket, which leaves bstart[k] at the end of bucket k (the start of
// k + 1): bucket k is [k ? bstart[k - 1] : 0, bstart[k]) afterwards
__global__ void k_grid_scatter(const int* __restrict__ nep, int cap, const unsigned* ekey, const int* eitem,
                               const unsigned long long* ecell, int* bstart, int* items, unsigned long long* cells)
{
    int ne = *nep;
    if (ne > cap || ne < 0) return;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < ne; e += gridDim.x * blockDim.x) {
        unsigned k = ekey[e];
        int pos = atomicAdd(&bstart[k], 1);
        items[pos] = eitem[e];
        cells[pos] = ecell[e];
    }
}

// orders LDS accesses between the lanes of one wavefront
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// for visitors that test the boxes (the query's with its margin) themselves
__device__ __forceinline__ bool boxes_apart(const float* ilo, const float* ihi, const float* qlo, const float* qhi)
{
    bool near = true;
#pragma unroll
    for (int d = 0; d < 3; d++) near &= ilo[d] <= qhi[d] && qlo[d] <= ihi[d];
    return !near;
}
// LDS of a wave of the query kernel
struct QueryWave {
    unsigned long long key[64];  // cell key of each pair
    float lo[64][3], hi[64][3];  // its query's box
    int q[64];                   // its query, and that one's vertices (an edge's second twice)
    int qv[64][3];
    int e0[64];                  // first entry of its bucket
    int pre[65];                 // entries of the pairs before it
    unsigned low[64];            // 1 | 2 | 4: the cell is the query's lowest along x | y | z
    int loc[TPB];                // first pairs of the queries of one block (find_box's table)
    int2 hits[192];              // (query, item) pairs to visit
};
// Generic query: visit(q, item) is called once per (query, item) pair whose cell
// ranges overlap, in the first cell common to both, unless Visit::apart says of
// their boxes that it would reject them, the two share a vertex, or Visit::half
// is set and not q < item.  Does nothing when the grid build
// flagged a retry (the caller then redoes the whole operation).
//
// A wave takes up to 64 consecutive (query, cell) pairs (fewer when there are
// few, so that a small scene spreads over the chip), lays the entries of
// their buckets end to end, and runs over them 128 at a time: key, first common
// cell and boxes, all loads of a step independent.  The survivors queue in LDS
// and are visited 64 at a time.  With one thread per pair walking its bucket,
// every entry cost a chain of dependent loads (cell, item, vertex numbers,
// vertices) in a wave as long as its longest bucket.  Like that, and like this:
// edge-edge CCD candidates on 200 cubes of 8^3 (176,400 surface edges) 332 and
// 190 us, collision test 196 and 114; on the 1M-tet slab 84 and 70, 68 and 49;
// edge-edge search on two cubes of 10^3 45 and 19 us.  Registers set the waves
// in flight (Visit::waves per SIMD; one more spills and takes 1.3 to 2 times as
// long).
template <class Visit>
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(Visit::waves)))
k_grid_query(int nq, int np, const int* __restrict__ qloc, const int* __restrict__ qpart,
             const QInfo* __restrict__ qinfo, unsigned M, const int* __restrict__ bstart,
             const int* __restrict__ items, const unsigned long long* __restrict__ cells,
             const FBox* __restrict__ ibox, int* flag, Visit visit)
{
    extern __shared__ int sP[];
    __shared__ QueryWave qw[TPB / 64];
    // the whole workgroup leaves or stays (lds_prefix synchronises it)
    __shared__ int stop;
    if (threadIdx.x == 0) stop = flag[0] & (GF_RETRY | GF_HUGE);
    __syncthreads();
    if (stop) return;
    const int total = lds_prefix(qpart, np, sP);
    if (total < 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(flag, GF_HUGE);
        return;
    }
    const int lane = threadIdx.x & 63;
    QueryWave& W = qw[threadIdx.x >> 6];
    // pairs per wave: a power of two
    const int nw = (int)gridDim.x * (TPB / 64);
    int per = 1;
    while (per < 64 && (long)per * nw < total) per <<= 1;
    const int w0 = __builtin_amdgcn_readfirstlane((int)blockIdx.x + (int)gridDim.x * ((int)threadIdx.x >> 6));
    const int nbatch = (total - 1) / per + 1;  // total >= 1 where it is used
    for (int b = w0; total > 0 && b < nbatch; b += nw) {
        const int t = b * per + lane;
        const bool on = lane < per && t < total;
        // the query of each pair: its block of queries, then its place in the block
        int blk = 0, hi = np;
        while (hi - blk > 1) {
            const int mid = (blk + hi) >> 1;
            if (sP[mid] <= (on ? t : b * per)) blk = mid; else hi = mid;
        }
        const int blk0 = __builtin_amdgcn_readfirstlane(blk);
        wave_sync();  // the last batch's reads of W are done
        for (int k = lane; k < TPB; k += 64) W.loc[k] = blk0 * TPB + k < nq ? qloc[blk0 * TPB + k] : 0x7fffffff;
        wave_sync();
        int cnt = 0;
        if (on) {
            const int r = t - sP[blk];
            const int base = blk * TPB;
            auto first = [&](int i) { return blk == blk0 ? W.loc[i - base] : qloc[i]; };
            int l = base, h = min(nq, l + TPB);
            while (h - l > 1) {
                const int mid = (l + h) >> 1;
                if (first(mid) <= r) l = mid; else h = mid;
            }
            const int c0 = r - first(l);
            const QInfo Q = qinfo[l];
            const int a = Q.clo[0] + c0 / (Q.ny * Q.nz), bb = Q.clo[1] + (c0 / Q.nz) % Q.ny, c = Q.clo[2] + c0 % Q.nz;
            const unsigned bk = bucket_of(a, bb, c, M);
            const int e0 = bk ? bstart[bk - 1] : 0;
            cnt = bstart[bk] - e0;
            W.key[lane] = cell_key(a, bb, c);
#pragma unroll
            for (int d = 0; d < 3; d++) {
                W.lo[lane][d] = Q.lo[d];
                W.hi[lane][d] = Q.hi[d];
                W.qv[lane][d] = Q.v[d];
            }
            W.q[lane] = l;
            W.e0[lane] = e0;
            W.low[lane] = (a == Q.clo[0] ? 1u : 0u) | (bb == Q.clo[1] ? 2u : 0u) | (c == Q.clo[2] ? 4u : 0u);
        }
        int inc = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(inc, d, 64);
            if (lane >= d) inc += y;
        }
        W.pre[lane] = inc - cnt;
        const int ne = __shfl(inc, 63, 64);
        if (lane == 0) W.pre[64] = ne;
        wave_sync();
        int nh = 0;
        for (int i0 = 0; i0 < ne; i0 += 128) {
            int pr[2], item[2];
            unsigned long long ck[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int i = i0 + 64 * k + lane;
                int lo = 0, h = 64;  // the pair whose entries hold i: the last with pre <= i
                while (h - lo > 1) {
                    const int mid = (lo + h) >> 1;
                    if (W.pre[mid] <= i) lo = mid; else h = mid;
                }
                pr[k] = lo;
                const int e = W.e0[lo] + i - W.pre[lo];
                item[k] = i < ne ? items[e] : 0;
                ck[k] = i < ne ? cells[e] : ~0ull;
            }
            bool ok[2];
            FBox ib[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                // first common cell: along each axis the cell is the lowest
                // cell of the query or of the item
                ok[k] = i0 + 64 * k + lane < ne && ck[k] == W.key[pr[k]] && ((((unsigned)item[k] >> 28) | W.low[pr[k]]) & 7u) == 7u;
                item[k] &= 0x0fffffff;
                if (Visit::half) ok[k] = ok[k] && W.q[pr[k]] < item[k];
                if (ok[k]) ib[k] = ibox[item[k]];
            }
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (ok[k]) {
                    ok[k] = !Visit::apart(ib[k].lo, ib[k].hi, W.lo[pr[k]], W.hi[pr[k]]);
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        const int v = W.qv[pr[k]][d];
                        ok[k] &= v != ib[k].v[0] && v != ib[k].v[1];
                    }
                }
                const unsigned long long m = __ballot(ok[k]);
                if (ok[k]) W.hits[nh + __popcll(m & ((1ull << lane) - 1))] =
                    make_int2(W.q[pr[k]], item[k]);
                nh += __popcll(m);
            }
            wave_sync();
            while (nh >= 64) {  // the last 64
                nh -= 64;
                const int2 v = W.hits[nh + lane];
                visit(v.x, v.y);
            }
            wave_sync();
        }
        if (lane < nh) {
            const int2 v = W.hits[lane];
            visit(v.x, v.y);
        }
    }
}

// st: the stream (c->s if null); each stream has its own scan scratch
static int scan_inplace(fipc_ctx* c, int* d, int n, hipStream_t st = nullptr)
{
    const hipStream_t s = st ? st : c->s;
    DVec<unsigned char>& tmp = s == c->s ? c->cub_tmp : c->cub_tmp2;
    size_t bytes = 0;
    HIPCHK(rocprim::exclusive_scan(nullptr, bytes, d, d, 0, (size_t)n, rocprim::plus<int>(), s));
    if (bytes > tmp.cap) STCHK(ensure(tmp, bytes));
    bytes = tmp.cap;
    HIPCHK(rocprim::exclusive_scan(tmp.p, bytes, d, d, 0, (size_t)n, rocprim::plus<int>(), s));
    return FIPC_OK;
}

// Build the grid over n items without waiting for the host: buffers are
// sized by the capacity, overflow is flagged in flag[0] (see GF_RETRY).
static int grid_build(fipc_ctx* c, int slot, int n, const BoxFn& box, hipStream_t st = nullptr)
{
    const hipStream_t s = st ? st : c->s;
    Grid& g = c->grid[slot];
    // the same boxes at the same x: the grid is already there; or the grid
    // sweeps these boxes from the x of version g.x_version along the current
    // sol, and x lies on that segment
    if (g.reusable && !box.sol && g.kind == box.kind && g.n == n && g.infl == box.infl) {
        if (!g.swept && g.x_version == c->x_version) return FIPC_OK;
        if (g.swept && c->seg_x == c->x_version && c->seg_base == g.x_version && c->seg_sol == g.seg_sol &&
            c->seg_sol == c->sol_version)
            return FIPC_OK;
    }
    g.reusable = false;
    const int np = nblk(n);
    if (np > OFF_PMAX) return FIPC_ERR_CAPACITY;
    STCHK(fipc_tm_begin(c, TM_GRID, s));
    int cap = g.cap;
    // buckets: a power of two at least the entry capacity
    unsigned M = 1024;
    while (M < (unsigned)cap && M < (1u << 30)) M <<= 1;
    g.M = M;
    STCHK(ensure(g.cnt, (size_t)n + 2));
    STCHK(ensure(g.ibox, (size_t)std::max(n, 1) * (sizeof(FBox) / 4)));
    STCHK(ensure(g.part, (size_t)np + 2));
    STCHK(ensure(g.ekey, cap)); STCHK(ensure(g.eitem, cap)); STCHK(ensure(g.items, cap));
    STCHK(ensure(g.ecell, cap)); STCHK(ensure(g.cells, cap));
    STCHK(ensure(g.bstart, (size_t)M + 1));
    if (np)
        k_count_cells<<<np, TPB, 0, s>>>(n, box, c->inv_dx, g.cnt.p, g.part.p, c->flag.p, (FBox*)g.ibox.p, g.bstart.p,
                                        (long)M + 1, nullptr, 0.0);
    else
        HIPCHK(hipMemsetAsync(g.bstart.p, 0, ((size_t)M + 1) * 4, s));
    HIPCHK(hipGetLastError());
    const int* nep = g.part.p + np;  // the entry count, stored by k_grid_fill
    int nb = stride_grid(cap);
    k_grid_fill<<<nb, TPB, (np + 1) * sizeof(int), s>>>(n, np, cap, box, c->inv_dx, M, g.cnt.p, g.part.p, g.ekey.p,
                                                         g.eitem.p, g.ecell.p, g.bstart.p, c->flag.p);
    HIPCHK(hipGetLastError());
    STCHK(scan_inplace(c, g.bstart.p, M + 1, s));
    k_grid_scatter<<<nb, TPB, 0, s>>>(nep, cap, g.ekey.p, g.eitem.p, g.ecell.p, g.bstart.p, g.items.p, g.cells.p);
    HIPCHK(hipGetLastError());
    // reusable once built; an overflow found after the operation's
    // synchronisation clears this again (bp_check).  A swept grid is reusable
    // only when it sweeps along sol itself
    g.swept = box.sol != nullptr;
    g.reusable = !g.swept || box.sol == c->sol.p;
    g.seg_sol = c->sol_version;
    g.x_version = c->x_version;
    g.kind = box.kind;
    g.n = n;
    g.infl = box.infl;
    STCHK(fipc_tm_end(c, TM_GRID, s));
    return FIPC_OK;
}

// query the last grid with nq boxes; no host synchronisation
template <class Visit>
static int run_query(fipc_ctx* c, int slot, int nq, const BoxFn& qbox, Visit visit, int timer,
                     hipStream_t st = nullptr)
{
    if (nq == 0) return FIPC_OK;
    const hipStream_t s = st ? st : c->s;
    Grid& g = c->grid[slot];
    const int np = nblk(nq);
    if (np > OFF_PMAX) return FIPC_ERR_CAPACITY;
    STCHK(ensure(g.qoff, (size_t)nq + 2));
    STCHK(ensure(g.qinfo, (size_t)nq * (sizeof(QInfo) / 4)));
    STCHK(ensure(g.qpart, (size_t)np + 2));
    STCHK(fipc_tm_begin(c, timer, s));
    k_count_cells<<<np, TPB, 0, s>>>(nq, qbox, c->inv_dx, g.qoff.p, g.qpart.p, c->flag.p, nullptr, nullptr, 0,
                                     (QInfo*)g.qinfo.p, 1e-9 * c->dHat);
    HIPCHK(hipGetLastError());
    k_grid_query<<<GRID_MAXB, TPB, (np + 1) * sizeof(int), s>>>(nq, np, g.qoff.p, g.qpart.p, (const QInfo*)g.qinfo.p,
                                                                 g.M, g.bstart.p, g.items.p, g.cells.p,
                                                                 (const FBox*)g.ibox.p, c->flag.p, visit);
    HIPCHK(hipGetLastError());
    STCHK(fipc_tm_end(c, timer, s));
    return FIPC_OK;
}

// start of a broad-phase operation, one launch: clears the status word and
// needed count (flag[0..2]) and ncnt counters, and sets namin minima to 1.0
__global__ void k_bp_begin(int* flag, int* cnt, int ncnt, unsigned long long* amin, int namin)
{
    const int i = threadIdx.x;
    if (i < 3) flag[i] = 0;
    if (i < ncnt) cnt[i] = 0;
    if (i < namin) amin[i] = 0x3ff0000000000000ull;  // the bits of 1.0
}
static int bp_begin(fipc_ctx* c, int* cnt = nullptr, int ncnt = 0, unsigned long long* amin = nullptr,
                    int namin = 0)
{
    k_bp_begin<<<1, 64, 0, c->s>>>(c->flag.p, cnt, ncnt, amin, namin);
    HIPCHK(hipGetLastError());
    return FIPC_OK;
}
// after the operation's synchronisation: error, retry (capacity grown) or done
static int bp_check(fipc_ctx* c, const int* hflag, bool* retry)
{
    *retry = false;
    if (hflag[0] & (GF_HUGE | GF_RETRY)) c->grid[0].reusable = c->grid[1].reusable = false;
    if (hflag[0] & GF_HUGE) return FIPC_ERR_CAPACITY;
    if (hflag[0] & GF_RETRY) {
        long need = (long)hflag[2];
        long cap = need + need / 4 + 4096;
        if (cap > (1L << 30)) return FIPC_ERR_CAPACITY;
        for (Grid& g : c->grid) g.cap = (int)std::max<long>(g.cap, cap);
        *retry = true;
    }
    return FIPC_OK;
}

// ---- constraint search ----------------------------------------------------
// one atomic per wavefront: adds the number of active lanes to *cnt
__device__ __forceinline__ void wave_count(int* cnt)
{
    unsigned long long m = __ballot(1);
    if (__lane_id() == __ffsll((unsigned long long)m) - 1) atomicAdd(cnt, (int)__popcll(m));
}
struct RowSink {
    int* cnt;                       // 7 raw counters
    int* cand;                      // broad-phase candidates (PT, EE), or null when not counted
    long long cap[NTYPES];
    unsigned long long* kpp;        // PP keys (a << 21 | b)
    unsigned long long* kpe;        // PE keys (p << 42 | e0 << 21 | e1)
    int* rows[NTYPES];
    // appends a row of type t (-1: none); every active lane calls it.  The lanes
    // of a type take consecutive places with one atomic per wave: at one per row
    // (about 13 ns each on one address) the edge-edge search of 200 cubes of 8^3,
    // 53,000 rows, took 726 us, like this 151
    __device__ __forceinline__ void row(int t, int a, int b, int c, int d) const
    {
        const int lane = __lane_id();
        unsigned long long todo = __ballot(t >= 0);
        int s = 0;
        while (todo) {
            const int lead = __ffsll(todo) - 1;
            const int tt = __shfl(t, lead, 64);
            const unsigned long long m = __ballot(t == tt);
            int base = 0;
            if (lane == lead) base = atomicAdd(&cnt[tt], __popcll(m));
            base = __shfl(base, lead, 64);
            if (t == tt) s = base + __popcll(m & ((1ull << lane) - 1));
            todo &= ~m;
        }
        if (t < 0 || s >= cap[t]) return;
        if (t == 0) kpp[s] = ((unsigned long long)a << 21) | (unsigned long long)b;
        else if (t == 1)
            kpe[s] = ((unsigned long long)a << 42) | ((unsigned long long)b << 21) | (unsigned long long)c;
        else *(int4*)(rows[t] + 4 * (size_t)s) = make_int4(a, b, c, d);
    }
};

// attempt_PT (NEWTON_IPC.py:181-212); query = triangle, item = boundary point
struct VisitPT {
    static constexpr bool half = false;
    static constexpr int waves = 4;  // per SIMD
    static __device__ __forceinline__ bool apart(const float* ilo, const float* ihi, const float* qlo, const float* qhi)
    {
        return boxes_apart(ilo, ihi, qlo, qhi);
    }
    const double* x;
    const int *bp, *bt;
    double dHat, dHat2;
    RowSink out;
    __device__ __forceinline__ void operator()(int tri, int pi) const
    {
        int p = bp[pi], t0 = bt[3 * tri], t1 = bt[3 * tri + 1], t2 = bt[3 * tri + 2];
        v3 P = ldv(x, p), T0 = ldv(x, t0), T1 = ldv(x, t1), T2 = ldv(x, t2);
        // point_triangle_ccd_broadphase (ipc.py:332-336)
        v3 mx = vmax(vmax(T0, T1), T2), mn = vmin(vmin(T0, T1), T2);
        int t = -1, a = p, b = 0, c = 0, d = 0;
        if (P.x < mx.x + dHat && P.y < mx.y + dHat && P.z < mx.z + dHat && mn.x - dHat < P.x && mn.y - dHat < P.y &&
            mn.z - dHat < P.z) {
            if (out.cand) wave_count(out.cand);
            const int k = PT_type(P, T0, T1, T2);
            if (PT_dist2(P, T0, T1, T2, k) < dHat2) {
                t = k < 3 ? 0 : (k < 6 ? 1 : 2);
                b = k == 1 || k == 4 ? t1 : (k == 2 || k == 5 ? t2 : t0);
                c = k == 3 || k == 6 ? t1 : (k == 4 ? t2 : t0);
                d = t2;
            }
        }
        out.row(t, a, b, c, d);
    }
};
// attempt_EE (NEWTON_IPC.py:235-312); query = edge i, item = edge j, keep i < j
struct VisitEE {
    static constexpr bool half = true;
    static constexpr int waves = 4;  // per SIMD
    static __device__ __forceinline__ bool apart(const float* ilo, const float* ihi, const float* qlo, const float* qhi)
    {
        return boxes_apart(ilo, ihi, qlo, qhi);
    }
    const double *x, *x0;
    const int* be;
    double dHat, dHat2;
    RowSink out;
    __device__ __forceinline__ void operator()(int i, int j) const
    {
        int a0 = be[2 * i], a1 = be[2 * i + 1], b0 = be[2 * j], b1 = be[2 * j + 1];
        v3 A0 = ldv(x, a0), A1 = ldv(x, a1), B0 = ldv(x, b0), B1 = ldv(x, b1);
        // edge_edge_ccd_broadphase (ipc.py:348-354)
        v3 mxa = vmax(A0, A1), mna = vmin(A0, A1), mxb = vmax(B0, B1), mnb = vmin(B0, B1);
        int t = -1, ra = a0, rb = a1, rc = b0, rd = b1;
        if (mna.x < mxb.x + dHat && mna.y < mxb.y + dHat && mna.z < mxb.z + dHat && mnb.x - dHat < mxa.x &&
            mnb.y - dHat < mxa.y && mnb.z - dHat < mxa.z) {
            if (out.cand) wave_count(out.cand + 1);
            const int k = EE_type(A0, A1, B0, B1);
            if (EE_dist2(A0, A1, B0, B1, k) < dHat2) {
                double cn2 = EECN2(A0, A1, B0, B1);
                double eps = M_threshold(ldv(x0, a0), ldv(x0, a1), ldv(x0, b0), ldv(x0, b1));
                const bool moll = cn2 < eps;
                // the mollified row: the edge with the nearest end first (that
                // end first), then the other (its nearest end first); the plain
                // row leaves out the far ends
                if (k == 6 || k == 7) {
                    ra = k == 6 ? b0 : b1; rb = k == 6 ? b1 : b0; rc = a0; rd = a1;
                } else if (k < 6) {
                    if (k >= 3) { ra = a1; rb = a0; }
                    if (k == 1 || k == 4) { rc = b1; rd = b0; }
                }
                const bool pp = k == 0 || k == 1 || k == 3 || k == 4;
                if (k == 8) t = moll ? 4 : 3;
                else if (moll) t = pp ? 5 : 6;
                else { t = pp ? 0 : 1; rb = rc; rc = rd; }
            }
        }
        out.row(t, ra, rb, rc, rd);
    }
};

// decode the unique sorted keys (count read on the device) into rows
__global__ void k_decode_pp(const int* __restrict__ np, const unsigned long long* k, int* rows)
{
    int n = *np;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        unsigned long long v = k[i];
        rows[2 * i] = (int)(v >> 21);
        rows[2 * i + 1] = (int)(v & ((1ull << 21) - 1));
    }
}
__global__ void k_decode_pe(const int* __restrict__ np, const unsigned long long* k, int* rows)
{
    int n = *np;
    unsigned long long m = (1ull << 21) - 1;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        unsigned long long v = k[i];
        rows[3 * i] = (int)(v >> 42);
        rows[3 * i + 1] = (int)((v >> 21) & m);
        rows[3 * i + 2] = (int)(v & m);
    }
}

// np.unique order: radix sort of the packed keys, unique into uniq; the
// unique count is left on the device (*d_n)
static int dedup(fipc_ctx* c, const unsigned long long* keys, int n, int end_bit, unsigned long long* sorted,
                 unsigned long long* uniq, int* d_n)
{
    size_t b1 = 0, b2 = 0;
    HIPCHK(rocprim::radix_sort_keys(nullptr, b1, keys, sorted, n, 0, end_bit, c->s));
    HIPCHK(rocprim::unique(nullptr, b2, sorted, uniq, d_n, (size_t)n, rocprim::equal_to<unsigned long long>(), c->s));
    size_t need = std::max(b1, b2);
    if (need > c->cub_tmp.cap) STCHK(ensure(c->cub_tmp, need));
    b1 = c->cub_tmp.cap;
    HIPCHK(rocprim::radix_sort_keys(c->cub_tmp.p, b1, keys, sorted, n, 0, end_bit, c->s));
    b2 = c->cub_tmp.cap;
    HIPCHK(rocprim::unique(c->cub_tmp.p, b2, sorted, uniq, d_n, (size_t)n, rocprim::equal_to<unsigned long long>(),
                           c->s));
    return FIPC_OK;
}

// lexicographic order of four-index rows (np.unique order)
struct Row4Less {
    __device__ __forceinline__ bool operator()(const int4& a, const int4& b) const
    {
        if (a.x != b.x) return a.x < b.x;
        if (a.y != b.y) return a.y < b.y;
        if (a.z != b.z) return a.z < b.z;
        return a.w < b.w;
    }
};
// sorts the n rows of a four-index type in place (through the scratch
// rows_tmp): the row order, and so every later sum over rows, no longer
// depends on the order the search appended them in
static int sort_rows4(fipc_ctx* c, DVec<int>& rows, int n)
{
    if (n < 2) return FIPC_OK;
    STCHK(ensure(c->rows_tmp, (size_t)n * 4));
    const int4* in = reinterpret_cast<const int4*>(rows.p);
    int4* out = reinterpret_cast<int4*>(c->rows_tmp.p);
    size_t b = 0;
    HIPCHK(rocprim::merge_sort(nullptr, b, in, out, (size_t)n, Row4Less(), c->s));
    if (b > c->cub_tmp.cap) STCHK(ensure(c->cub_tmp, b));
    b = c->cub_tmp.cap;
    HIPCHK(rocprim::merge_sort(c->cub_tmp.p, b, in, out, (size_t)n, Row4Less(), c->s));
    std::swap(rows, c->rows_tmp);
    return FIPC_OK;
}

// Few rows: per type, up to ROWS_SMALL rows are sorted (PP and PE also
// deduplicated and decoded) by their ranks, each row compared with all others
// from LDS, 256 rows to a block and four lanes to a row.  It runs right behind the
// queries, on the counts on the device, so that one readback returns the final
// counts; a type with more rows is left to the host, which then runs the
// library's sorts.  A merge sort of 500 rows is a 13 us launch, a radix sort, unique
// and decode of 20 keys five launches with a readback of their own: line search
// (two searches) on two cubes (520 rows) 0.51 ms with those, like this 0.44; on
// the 1M-tet slab (4,000 PT, 180 EE, 21 PE) 1.16 and 1.02.
constexpr int ROWS_SMALL = 1024;  // no more than any type's first capacity
struct SmallRows {
    const int* cnt;                         // raw counts
    const unsigned long long *kpp, *kpe;
    const int4* in[NTYPES];                 // 4-index types: rows as appended
    int4* out[NTYPES];                      // and sorted
    int *pp, *pe;                           // decoded unique rows
    int* nuniq;                             // unique PP and PE
};
constexpr int ROWS_PB = ROWS_SMALL / 4;  // rows per block
// ranks of the block's rows r0 + (thread % ROWS_PB) among n (hi, lo) keys in LDS,
// padded with all ones to a multiple of 16; lane part p takes every fourth block
// of four keys
__device__ __forceinline__ void rank_rows(const unsigned long long* hi, const unsigned* lo, int n, int row, int* rank)
{
    const unsigned long long h = hi[min(row, n - 1)];
    const unsigned l = lo[min(row, n - 1)];
    int r = 0;
#pragma unroll 2
    for (int j = 4 * ((int)threadIdx.x / ROWS_PB); j < n; j += 16)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const unsigned long long q = hi[j + k];
            r += q < h || (q == h && lo[j + k] < l) ? 1 : 0;
        }
    if (r) atomicAdd(&rank[(int)threadIdx.x % ROWS_PB], r);
}
__global__ void __launch_bounds__(ROWS_SMALL) k_rows_small(SmallRows a)
{
    __shared__ __attribute__((aligned(16))) unsigned long long hi[ROWS_SMALL + 16];
    __shared__ __attribute__((aligned(16))) unsigned lo[ROWS_SMALL + 16];
    __shared__ unsigned long long sorted[ROWS_SMALL];
    __shared__ int rank[ROWS_PB], wsum[ROWS_SMALL / 64];
    const int t = blockIdx.x, n = a.cnt[t], i = threadIdx.x, r0 = (int)blockIdx.y * ROWS_PB;
    if (n > ROWS_SMALL) return;
    // PP and PE: one block ranks all, for the numbering of the unique keys
    if (t < 2 ? blockIdx.y > 0 : r0 >= n) return;
    // 63 key bits in hi; lo breaks ties by place (rows of four: their last index,
    // then the place)
    int4 v = make_int4(0, 0, 0, 0);
    hi[i] = ~0ull;
    lo[i] = ~0u;
    if (i < 16) { hi[ROWS_SMALL + i] = ~0ull; lo[ROWS_SMALL + i] = ~0u; }
    if (i < n) {
        if (t >= 2) {
            v = a.in[t][i];
            hi[i] = ((unsigned long long)v.x << 42) | ((unsigned long long)v.y << 21) | (unsigned long long)v.z;
            lo[i] = ((unsigned)v.w << 10) | (unsigned)i;
        } else {
            hi[i] = (t == 0 ? a.kpp : a.kpe)[i];
            lo[i] = (unsigned)i;
        }
    }
    __syncthreads();
    if (t >= 2) {
        if (i < ROWS_PB) rank[i] = 0;
        __syncthreads();
        rank_rows(hi, lo, n, r0 + i % ROWS_PB, rank);
        __syncthreads();
        if (i >= r0 && i < min(n, r0 + ROWS_PB)) a.out[t][rank[i - r0]] = v;
        return;
    }
    for (int b = 0; b < n; b += ROWS_PB) {
        __syncthreads();
        if (i < ROWS_PB) rank[i] = 0;
        __syncthreads();
        rank_rows(hi, lo, n, b + i % ROWS_PB, rank);
        __syncthreads();
        if (i >= b && i < min(n, b + ROWS_PB)) sorted[rank[i - b]] = hi[i];
    }
    __syncthreads();
    // the first of equal keys, numbered in order
    const bool head = i < n && (i == 0 || sorted[i] != sorted[i - 1]);
    const unsigned long long m = __ballot(head);
    const int lane = i & 63, w = i >> 6;
    if (lane == 0) wsum[w] = __popcll(m);
    __syncthreads();
    int before = __popcll(m & ((1ull << lane) - 1)), all = 0;
    for (int v = 0; v < ROWS_SMALL / 64; v++) {
        if (v < w) before += wsum[v];
        all += wsum[v];
    }
    if (i == 0) a.nuniq[t] = all;
    if (!head) return;
    const unsigned long long key = sorted[i], low = (1ull << 21) - 1;
    if (t == 0) {
        a.pp[2 * before] = (int)(key >> 21);
        a.pp[2 * before + 1] = (int)(key & low);
    } else {
        a.pe[3 * before] = (int)(key >> 42);
        a.pe[3 * before + 1] = (int)((key >> 21) & low);
        a.pe[3 * before + 2] = (int)(key & low);
    }
}

static int bits_for(int n)
{
    int b = 1;
    while ((1 << b) < n) b++;
    return b;
}

// one pass of both searches and the sorts of small row sets; raw counts (12),
// unique PP and PE counts (2) and the status word come back with the single
// synchronisation
static int find_once(fipc_ctx* c, int* counts, int* hflag)
{
    STCHK(bp_begin(c, c->counters.p, 14));
    RowSink sink;
    sink.cnt = c->counters.p;
    // one same-address atomic per wavefront and candidate test would
    // serialise the queries: the candidates are counted only on request
    sink.cand = c->search_stats ? c->counters.p + 10 : nullptr;
    for (int t = 0; t < NTYPES; t++) { sink.cap[t] = c->cap[t]; sink.rows[t] = c->rows[t].p; }
    sink.kpp = c->keys_pp.p;
    sink.kpe = c->keys_pe.p;
    // PT: points inserted with +-dHat, triangles query their box
    BoxFn pts{c->x.p, nullptr, c->bp.p, 0, c->dHat};
    STCHK(grid_build(c, 0, c->nbp, pts));
    BoxFn tris{c->x.p, nullptr, c->bt.p, 2, 0.0};
    VisitPT vpt{c->x.p, c->bp.p, c->bt.p, c->dHat, c->dHat2, sink};
    STCHK(run_query(c, 0, c->nbt, tris, vpt, TM_FIND));
    // EE: edges inserted with their box, queried with box +- dHat
    BoxFn edges{c->x.p, nullptr, c->be.p, 1, 0.0};
    STCHK(grid_build(c, 1, c->nbe, edges));
    BoxFn qedges{c->x.p, nullptr, c->be.p, 1, c->dHat};
    VisitEE vee{c->x.p, c->x0.p, c->be.p, c->dHat, c->dHat2, sink};
    STCHK(run_query(c, 1, c->nbe, qedges, vee, TM_FIND));
    SmallRows sr;
    sr.cnt = c->counters.p;
    sr.kpp = c->keys_pp.p;
    sr.kpe = c->keys_pe.p;
    for (int t = 2; t < NTYPES; t++) {
        sr.in[t] = reinterpret_cast<const int4*>(c->rows[t].p);
        sr.out[t] = reinterpret_cast<int4*>(c->rows_small[t].p);
    }
    sr.pp = c->rows[0].p;
    sr.pe = c->rows[1].p;
    sr.nuniq = c->counters.p + 12;
    k_rows_small<<<dim3(NTYPES, ROWS_SMALL / ROWS_PB), ROWS_SMALL, 0, c->s>>>(sr);
    HIPCHK(hipGetLastError());
    STCHK(d2h_async(c, counts, c->counters.p, 14 * 4));
    STCHK(d2h_async(c, hflag, c->flag.p, 12));
    STCHK(d2h_wait(c));
    return FIPC_OK;
}

extern "C" int fipc_find_constraints(fipc_ctx* c, int* counts_out)
{
    if (!c || !c->nv) return FIPC_ERR_STATE;
    int raw[14];
    for (int attempt = 0;; attempt++) {
        if (attempt == 6) return FIPC_ERR_CAPACITY;
        STCHK(ensure(c->keys_pp, c->cap[0]));
        STCHK(ensure(c->keys_pe, c->cap[1]));
        for (int t = 2; t < NTYPES; t++) {
            STCHK(ensure(c->rows[t], c->cap[t] * 4));
            STCHK(ensure(c->rows_small[t], 4 * ROWS_SMALL));
        }
        STCHK(ensure(c->rows[0], 2 * ROWS_SMALL));
        STCHK(ensure(c->rows[1], 3 * ROWS_SMALL));
        int hflag[3];
        STCHK(find_once(c, raw, hflag));
        bool grow = false;
        STCHK(bp_check(c, hflag, &grow));
        if (grow) continue;
        for (int t = 0; t < NTYPES; t++)
            if (raw[t] > c->cap[t]) { c->cap[t] = (int64_t)raw[t] * 2; grow = true; }
        if (!grow) break;
    }
    for (int t = 0; t < NTYPES; t++) c->raw_count[t] = raw[t];
    c->cand_last[0] = c->search_stats ? raw[10] : -1;
    c->cand_last[1] = c->search_stats ? raw[11] : -1;
    int bits = bits_for(c->nv);
    // sorted and unique keys of PP then PE share keys_tmp
    size_t npp_raw = raw[0], npe_raw = raw[1];
    STCHK(ensure(c->keys_tmp, 2 * (npp_raw + npe_raw) + 4));
    unsigned long long* kt = c->keys_tmp.p;
    STCHK(ensure(c->rows[0], std::max<size_t>(npp_raw, 1) * 2));
    STCHK(ensure(c->rows[1], std::max<size_t>(npe_raw, 1) * 3));
    const bool big_pp = raw[0] > ROWS_SMALL, big_pe = raw[1] > ROWS_SMALL;
    int nu[2] = {raw[12], raw[13]};
    if (big_pp) {
        STCHK(dedup(c, c->keys_pp.p, raw[0], std::min(64, 21 + bits), kt, kt + npp_raw, c->nuniq.p));
        k_decode_pp<<<stride_grid(npp_raw), TPB, 0, c->s>>>(c->nuniq.p, kt + npp_raw, c->rows[0].p);
    }
    if (big_pe) {
        unsigned long long* k2 = kt + 2 * npp_raw;
        STCHK(dedup(c, c->keys_pe.p, raw[1], std::min(64, 42 + bits), k2, k2 + npe_raw, c->nuniq.p + 1));
        k_decode_pe<<<stride_grid(npe_raw), TPB, 0, c->s>>>(c->nuniq.p + 1, k2 + npe_raw, c->rows[1].p);
    }
    HIPCHK(hipGetLastError());
    for (int t = 2; t < NTYPES; t++) {
        if (raw[t] > ROWS_SMALL) {
            STCHK(sort_rows4(c, c->rows[t], raw[t]));
        } else {
            // the sorted rows are the type's rows now; a search appends into a
            // buffer of the type's capacity again (ensured at its start)
            std::swap(c->rows[t], c->rows_small[t]);
        }
    }
    if (big_pp || big_pe) {
        int big[2];
        STCHK(d2h_async(c, big, c->nuniq.p, 8));
        STCHK(d2h_wait(c));
        if (big_pp) nu[0] = big[0];
        if (big_pe) nu[1] = big[1];
    }
    c->count[0] = nu[0];
    c->count[1] = nu[1];
    for (int t = 2; t < NTYPES; t++) c->count[t] = raw[t];
    c->sys_version++;   // the contact rows of the SpMV changed
    c->cons_version++;  // and those of the barrier energy
    for (int t = 0; t < NTYPES; t++) {
        int N = 3 * (t == 0 ? 2 : (t == 1 ? 3 : 4));
        STCHK(ensure(c->cH[t], (size_t)std::max(c->count[t], 1) * N * N));
        if (counts_out) counts_out[t] = c->count[t];
    }
    return FIPC_OK;
}

extern "C" int fipc_get_constraints(fipc_ctx* c, int type, int* rows_out)
{
    if (!c || type < 0 || type >= NTYPES || !rows_out) return FIPC_ERR_ARG;
    int w = type == 0 ? 2 : (type == 1 ? 3 : 4);
    if (c->count[type])
        HIPCHK(hipMemcpyAsync(rows_out, c->rows[type].p, (size_t)c->count[type] * w * 4, hipMemcpyDeviceToHost, c->s));
    HIPCHK(hipStreamSynchronize(c->s));
    return FIPC_OK;
}

// ---- CCD filters ----------------------------------------------------------
// Candidate pairs: the grid walk applies the moving-box test of the reference
// and the CCD lower bound (a pair whose bound lb = (1 - eta) d / maxDisp is
// at least 1 keeps toc = 1, wrapper.cpp:254-328), and appends the rest; the
// narrow phase (CTCD) then runs one thread per candidate, so its long,
// data-dependent root finding neither stalls the grid walk nor unbalances
// its waves.
// One atomic per wavefront: the active lanes that append take consecutive slots.
__device__ __forceinline__ int wave_append(int* cnt)
{
    unsigned long long mask = __ballot(1);
    int leader = __ffsll((unsigned long long)mask) - 1;
    int lane = __lane_id();
    int base = 0;
    if (lane == leader) base = atomicAdd(cnt, __popcll(mask));
    base = __shfl(base, leader, 64);
    unsigned long long below = lane == 0 ? 0ull : (mask & (~0ull >> (64 - lane)));
    return base + __popcll(below);
}
struct PairSink {
    int* cnt;
    int cap;
    int2* pairs;
    __device__ __forceinline__ void push(int a, int b) const
    {
        int s = wave_append(cnt);
        if (s < cap) pairs[s] = make_int2(a, b);
    }
};
// compute_filter_3D_PT (NEWTON_IPC.py:377-406); query = triangle, item = point
struct CandCCDPT {
    static constexpr bool half = false;
    static constexpr int waves = 3;  // per SIMD
    static __device__ __forceinline__ bool apart(const float* ilo, const float* ihi, const float* qlo, const float* qhi)
    {
        return boxes_apart(ilo, ihi, qlo, qhi);
    }
    const double *x, *p;
    const int *bp, *bt;
    double dHat, eta;
    PairSink out;
    __device__ __forceinline__ void operator()(int tri, int pi) const
    {
        const int q = bp[pi], t0 = bt[3 * tri], t1 = bt[3 * tri + 1], t2 = bt[3 * tri + 2];
        v3 P = ldv(x, q), dP = ldv(p, q);
        v3 T0 = ldv(x, t0), T1 = ldv(x, t1), T2 = ldv(x, t2);
        v3 d0 = ldv(p, t0), d1 = ldv(p, t1), d2 = ldv(p, t2);
        // moving_point_triangle_ccd_broadphase (ipc.py:339-345)
        v3 mxp = vmax(P, P + dP), mnp = vmin(P, P + dP);
        v3 mxt = vmax(vmax(T0, T0 + d0), vmax(vmax(T1, T1 + d1), vmax(T2, T2 + d2)));
        v3 mnt = vmin(vmin(T0, T0 + d0), vmin(vmin(T1, T1 + d1), vmin(T2, T2 + d2)));
        if (!(mnp.x < mxt.x + dHat && mnp.y < mxt.y + dHat && mnp.z < mxt.z + dHat)) return;
        if (!(mnt.x - dHat < mxp.x && mnt.y - dHat < mxp.y && mnt.z - dHat < mxp.z)) return;
        // the lower bound of pt_ccd, same expressions
        double maxDisp = sqrt(n2(dP)) + sqrt(fmax(fmax(n2(d0), n2(d1)), n2(d2)));
        if (maxDisp == 0) return;
        double d2c = PT_dist2(P, T0, T1, T2, PT_type(P, T0, T1, T2));
        if (!((1 - eta) * sqrt(d2c) / maxDisp < 1)) return;
        out.push(tri, pi);
    }
};
// compute_filter_3D_EE (NEWTON_IPC.py:409-440); query edge i, item edge j
struct CandCCDEE {
    static constexpr bool half = true;
    static constexpr int waves = 3;  // per SIMD
    static __device__ __forceinline__ bool apart(const float* ilo, const float* ihi, const float* qlo, const float* qhi)
    {
        return boxes_apart(ilo, ihi, qlo, qhi);
    }
    const double *x, *p;
    const int* be;
    double dHat, eta;
    PairSink out;
    __device__ __forceinline__ void operator()(int i, int j) const
    {
        const int a0 = be[2 * i], a1 = be[2 * i + 1], b0 = be[2 * j], b1 = be[2 * j + 1];
        v3 A0 = ldv(x, a0), A1 = ldv(x, a1), dA0 = ldv(p, a0), dA1 = ldv(p, a1);
        v3 B0 = ldv(x, b0), B1 = ldv(x, b1), dB0 = ldv(p, b0), dB1 = ldv(p, b1);
        // moving_edge_edge_ccd_broadphase (ipc.py:357-363)
        v3 mxa = vmax(vmax(A0, A0 + dA0), vmax(A1, A1 + dA1)), mna = vmin(vmin(A0, A0 + dA0), vmin(A1, A1 + dA1));
        v3 mxb = vmax(vmax(B0, B0 + dB0), vmax(B1, B1 + dB1)), mnb = vmin(vmin(B0, B0 + dB0), vmin(B1, B1 + dB1));
        if (!(mna.x < mxb.x + dHat && mna.y < mxb.y + dHat && mna.z < mxb.z + dHat)) return;
        if (!(mnb.x - dHat < mxa.x && mnb.y - dHat < mxa.y && mnb.z - dHat < mxa.z)) return;
        // the lower bound of ee_ccd, same expressions
        double maxDisp = sqrt(fmax(n2(dA0), n2(dA1))) + sqrt(fmax(n2(dB0), n2(dB1)));
        if (maxDisp == 0) return;
        double d2c = EE_dist2(A0, A1, B0, B1, EE_type(A0, A1, B0, B1));
        if (!((1 - eta) * sqrt(d2c) / maxDisp < 1)) return;
        out.push(i, j);
    }
};
__device__ __forceinline__ void amin_d(unsigned long long* a, double v)
{
    atomicMin(a, (unsigned long long)__double_as_longlong(v));
}
// narrow phase over the candidates (count read on the device, capped at cap:
// an overflowing count makes the host redo the filter with more room).  A
// pair's time of impact is the lesser of its two roundings (strict and
// fused); the two run in different wavefronts (wavefront w takes the pairs
// of group w / 2 of 64 in rounding w % 2), so each wavefront runs one root
// isolation per pair: the minimum over (pair, rounding) is the minimum over
// pairs of the lesser, bit for bit, with twice the wavefronts in flight.
__device__ __forceinline__ bool ccd_slot(long t, int n, int* i, bool* fused)
{
    *i = (int)((t >> 7) * 64 + (t & 63));
    *fused = (t >> 6) & 1;
    return *i < n;
}
__global__ void __launch_bounds__(TPB) k_ccd_pt(const int* __restrict__ cnt, int cap, const int2* __restrict__ pairs,
                                                const double* __restrict__ x, const double* __restrict__ p,
                                                const int* __restrict__ bp, const int* __restrict__ bt, double eta,
                                                unsigned long long* amin)
{
    const int n = min(*cnt, cap);
    const long nt = 2L * ((n + 63) / 64) * 64;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += (long)gridDim.x * blockDim.x) {
        int i;
        bool fused;
        if (!ccd_slot(t, n, &i, &fused)) continue;
        int2 pr = pairs[i];
        int q = bp[pr.y], t0 = bt[3 * pr.x], t1 = bt[3 * pr.x + 1], t2 = bt[3 * pr.x + 2];
        v3 P = ldv(x, q), T0 = ldv(x, t0), T1 = ldv(x, t1), T2 = ldv(x, t2);
        v3 dP = ldv(p, q), d0 = ldv(p, t0), d1 = ldv(p, t1), d2 = ldv(p, t2);
        double d2c = PT_dist2(P, T0, T1, T2, PT_type(P, T0, T1, T2));
        double toc = fused ? ccd_fused::pt_ccd(P, T0, T1, T2, dP, d0, d1, d2, eta, d2c)
                           : ccd_strict::pt_ccd(P, T0, T1, T2, dP, d0, d1, d2, eta, d2c);
        if (toc < 1.0) amin_d(amin, toc);
    }
}
__global__ void __launch_bounds__(TPB) k_ccd_ee(const int* __restrict__ cnt, int cap, const int2* __restrict__ pairs,
                                                const double* __restrict__ x, const double* __restrict__ p,
                                                const int* __restrict__ be, double eta, unsigned long long* amin)
{
    const int n = min(*cnt, cap);
    const long nt = 2L * ((n + 63) / 64) * 64;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += (long)gridDim.x * blockDim.x) {
        int i;
        bool fused;
        if (!ccd_slot(t, n, &i, &fused)) continue;
        int2 pr = pairs[i];
        int a0 = be[2 * pr.x], a1 = be[2 * pr.x + 1], b0 = be[2 * pr.y], b1 = be[2 * pr.y + 1];
        v3 A0 = ldv(x, a0), A1 = ldv(x, a1), B0 = ldv(x, b0), B1 = ldv(x, b1);
        v3 dA0 = ldv(p, a0), dA1 = ldv(p, a1), dB0 = ldv(p, b0), dB1 = ldv(p, b1);
        double d2c = EE_dist2(A0, A1, B0, B1, EE_type(A0, A1, B0, B1));
        double toc = fused ? ccd_fused::ee_ccd(A0, A1, B0, B1, dA0, dA1, dB0, dB1, eta, d2c)
                           : ccd_strict::ee_ccd(A0, A1, B0, B1, dA0, dA1, dB0, dB1, eta, d2c);
        if (toc < 1.0) amin_d(amin, toc);
    }
}

extern int fipc_inversion_alpha(fipc_ctx* c, unsigned long long* dst);

// compute_intersection_free_step_size (NEWTON_IPC.py:456-468)
extern "C" int fipc_ccd_alpha(fipc_ctx* c, double eta, int inversion, double* alpha, double* parts)
{
    if (!c || !c->nv || !alpha) return FIPC_ERR_STATE;
    double a[3];
    for (int attempt = 0;; attempt++) {
        if (attempt == 6) return FIPC_ERR_CAPACITY;
        int cap = c->ccd_cap;
        STCHK(ensure(c->ccd_pairs[0], cap)); STCHK(ensure(c->ccd_pairs[1], cap));
        int* pc = c->counters.p + 8;
        STCHK(bp_begin(c, pc, 2, c->amin.p, 3));
        // the edge-edge half (the longer one) runs on the second stream while
        // the point-triangle half and the inversion bound run on the first:
        // separate grids, pair lists, counters and minima; the first waits
        // for the second before the readback
        HIPCHK(hipEventRecord(c->ev_rhs, c->s));
        HIPCHK(hipStreamWaitEvent(c->s2, c->ev_rhs, 0));
        BoxFn edges{c->x.p, c->sol.p, c->be.p, 1, 0.0};
        STCHK(grid_build(c, 1, c->nbe, edges, c->s2));
        BoxFn qedges{c->x.p, c->sol.p, c->be.p, 1, c->dHat};
        CandCCDEE vee{c->x.p, c->sol.p, c->be.p, c->dHat, eta, PairSink{pc + 1, cap, c->ccd_pairs[1].p}};
        STCHK(run_query(c, 1, c->nbe, qedges, vee, TM_CCD, c->s2));
        STCHK(fipc_tm_begin(c, TM_NARROW, c->s2));
        k_ccd_ee<<<stride_grid(2L * cap), TPB, 0, c->s2>>>(pc + 1, cap, c->ccd_pairs[1].p, c->x.p, c->sol.p, c->be.p, eta,
                                                      c->amin.p + 1);
        HIPCHK(hipGetLastError());
        STCHK(fipc_tm_end(c, TM_NARROW, c->s2));
        HIPCHK(hipEventRecord(c->ev_contact, c->s2));
        BoxFn pts{c->x.p, c->sol.p, c->bp.p, 0, c->dHat};
        STCHK(grid_build(c, 0, c->nbp, pts));
        BoxFn tris{c->x.p, c->sol.p, c->bt.p, 2, 0.0};
        CandCCDPT vpt{c->x.p, c->sol.p, c->bp.p, c->bt.p, c->dHat, eta, PairSink{pc, cap, c->ccd_pairs[0].p}};
        STCHK(run_query(c, 0, c->nbt, tris, vpt, TM_CCD));
        STCHK(fipc_tm_begin(c, TM_NARROW));
        k_ccd_pt<<<stride_grid(2L * cap), TPB, 0, c->s>>>(pc, cap, c->ccd_pairs[0].p, c->x.p, c->sol.p, c->bp.p, c->bt.p, eta,
                                                     c->amin.p);
        HIPCHK(hipGetLastError());
        STCHK(fipc_tm_end(c, TM_NARROW));
        if (inversion) STCHK(fipc_inversion_alpha(c, c->amin.p + 2));
        HIPCHK(hipStreamWaitEvent(c->s, c->ev_contact, 0));
        unsigned long long out[3];
        int hflag[3], hc[2];
        STCHK(d2h_async(c, out, c->amin.p, 24));
        STCHK(d2h_async(c, hflag, c->flag.p, 12));
        STCHK(d2h_async(c, hc, pc, 8));
        STCHK(d2h_wait(c));
        bool retry = false;
        STCHK(bp_check(c, hflag, &retry));
        int need = std::max(hc[0], hc[1]);
        if (need > cap) {
            c->ccd_cap = need + need / 2 + 1024;
            retry = true;
        }
        if (retry) continue;
        memcpy(a, out, 24);
        c->ccd_last[0] = hc[0];
        c->ccd_last[1] = hc[1];
        break;
    }
    if (parts) { parts[0] = a[0]; parts[1] = a[1]; parts[2] = a[2]; }
    *alpha = std::min(std::min(a[0], a[1]), a[2]);
    return FIPC_OK;
}

extern "C" int fipc_search_stats(fipc_ctx* c, int on)
{
    if (!c) return FIPC_ERR_ARG;
    c->search_stats = on != 0;
    return FIPC_OK;
}

extern "C" int fipc_search_counts(fipc_ctx* c, int* cand)
{
    if (!c || !cand) return FIPC_ERR_ARG;
    cand[0] = c->cand_last[0];
    cand[1] = c->cand_last[1];
    return FIPC_OK;
}

extern "C" int fipc_ccd_counts(fipc_ctx* c, int* pairs)
{
    if (!c || !pairs) return FIPC_ERR_ARG;
    pairs[0] = c->ccd_last[0];
    pairs[1] = c->ccd_last[1];
    return FIPC_OK;
}

// ---- collision check --------------------------------------------------------
struct VisitCollide {
    static constexpr bool half = false;
    static constexpr int waves = 4;  // per SIMD
    // the test has no box test of its own, and passes pairs of long edges whose
    // boxes are apart: left out are only those that it rejects (line search on
    // 200 cubes 1.83 ms; with a fixed distance of a tenth of a cell, which left
    // out pairs that the test passes, 1.91)
    static __device__ __forceinline__ bool apart(const float* ilo, const float* ihi, const float* qlo, const float* qhi)
    {
        return seg_tri_apart(ilo, ihi, qlo, qhi);
    }
    const double* x;
    const int *be, *bt;
    int* hit;
    __device__ __forceinline__ void operator()(int tri, int ei) const
    {
        const int a0 = be[2 * ei], a1 = be[2 * ei + 1], t0 = bt[3 * tri], t1 = bt[3 * tri + 1], t2 = bt[3 * tri + 2];
        if (seg_tri(ldv(x, a0), ldv(x, a1), ldv(x, t0), ldv(x, t1), ldv(x, t2))) atomicOr(hit, 1);
    }
};

// check_collision (NEWTON_IPC.py:855-886)
extern "C" int fipc_check_collision(fipc_ctx* c, int* hit)
{
    if (!c || !c->nv || !hit) return FIPC_ERR_STATE;
    for (int attempt = 0;; attempt++) {
        if (attempt == 6) return FIPC_ERR_CAPACITY;
        STCHK(bp_begin(c));
        // the edge grid of the constraint search (boxes without margin), so
        // either reuses the other's at the same x; the margin d-hat moves to
        // the triangle queries, which pairs the same boxes
        BoxFn edges{c->x.p, nullptr, c->be.p, 1, 0.0};
        STCHK(grid_build(c, 1, c->nbe, edges));
        BoxFn tris{c->x.p, nullptr, c->bt.p, 2, c->dHat};
        VisitCollide v{c->x.p, c->be.p, c->bt.p, c->flag.p + 1};
        STCHK(run_query(c, 1, c->nbt, tris, v, TM_FIND));
        int hflag[3];
        STCHK(d2h_async(c, hflag, c->flag.p, 12));
        STCHK(d2h_wait(c));
        bool retry = false;
        STCHK(bp_check(c, hflag, &retry));
        if (retry) continue;
        *hit = hflag[1];
        return FIPC_OK;
    }
}

// ---- batched CCD -----------------------------------------------------------
// 64 pairs per block, the strict rounding on its first wave and the fused one on
// its second; the lesser time is the pair's.  (One thread ran both before, at
// default launch bounds, whose 128 registers spilled 190: 30,011 edge pairs took
// 1045 us, 469 waves on 1,024 SIMDs; like this, with the bisections in registers,
// 232.)
template <int TYPE>
__global__ void __launch_bounds__(128) k_batch_ccd(int n, const double* __restrict__ pts,
                                                   const double* __restrict__ disp, double eta,
                                                   const double* __restrict__ d2, double* __restrict__ toc)
{
    __shared__ double other[64];
    const int lane = threadIdx.x & 63, i = blockIdx.x * 64 + lane;
    const bool fused = threadIdx.x >= 64;
    double t = 1.0;
    if (i < n) {
        const double* P = pts + 12 * (size_t)i;
        const double* D = disp + 12 * (size_t)i;
        v3 a = ld3(P), b = ld3(P + 3), cc = ld3(P + 6), d = ld3(P + 9);
        v3 da = ld3(D), db = ld3(D + 3), dc = ld3(D + 6), dd = ld3(D + 9);
        if (TYPE == 0)
            t = fused ? ccd_fused::pt_ccd(a, b, cc, d, da, db, dc, dd, eta, d2[i])
                      : ccd_strict::pt_ccd(a, b, cc, d, da, db, dc, dd, eta, d2[i]);
        else
            t = fused ? ccd_fused::ee_ccd(a, b, cc, d, da, db, dc, dd, eta, d2[i])
                      : ccd_strict::ee_ccd(a, b, cc, d, da, db, dc, dd, eta, d2[i]);
    }
    if (fused) other[lane] = t;
    __syncthreads();
    if (!fused && i < n) toc[i] = fmin(t, other[lane]);
}
// device arrays of n pairs, on the default stream
int fipc_launch_batch_ccd(int type, int n, const double* pts, const double* disp, double eta, const double* d2,
                          double* toc)
{
    if (type == 0) k_batch_ccd<0><<<nblk(n, 64), 128>>>(n, pts, disp, eta, d2, toc);
    else k_batch_ccd<1><<<nblk(n, 64), 128>>>(n, pts, disp, eta, d2, toc);
    HIPCHK(hipGetLastError());
    return FIPC_OK;
}
extern "C" int fipc_batch_ccd(int type, int n, const double* pts, const double* disp, double eta, const double* dist2, double* toc)
{
    if (n < 0 || (type != 0 && type != 1)) return FIPC_ERR_ARG;
    if (n == 0) return FIPC_OK;
    double* dp;  // one allocation for the inputs and the times
    HIPCHK(hipMalloc(&dp, (size_t)n * 26 * 8));
    double *dd = dp + 12 * (size_t)n, *d2 = dd + 12 * (size_t)n, *dt = d2 + n;
    hipError_t e = hipMemcpy(dp, pts, (size_t)n * 96, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dd, disp, (size_t)n * 96, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d2, dist2, (size_t)n * 8, hipMemcpyHostToDevice);
    const int st = e == hipSuccess ? fipc_launch_batch_ccd(type, n, dp, dd, eta, d2, dt) : FIPC_OK;
    if (e == hipSuccess && st == FIPC_OK) e = hipMemcpy(toc, dt, (size_t)n * 8, hipMemcpyDeviceToHost);
    (void)hipFree(dp);
    HIPCHK(e);
    STCHK(st);
    return FIPC_OK;
}

