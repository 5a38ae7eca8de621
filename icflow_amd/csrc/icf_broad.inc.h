// icf_broad.inc.h -- broad phase and (node, tet) de-duplication on the device (included by
// icf_lib.hip).
//
// Broad phase: every pair (a < b) of surface tets whose 12-direction k-DOPs on the current
// positions overlap -- the set the reference's BVH reports (v3Library/Collisions/BVH/
// BVHN.cs:166-196 with kDOP24.cs:84-140), which is the set icfh_kdop_pairs finds on the host.
// The k-DOP extents are sums and differences of coordinates and the overlap test is a
// comparison, so both produce the same pairs; the order is (a, b) ascending.  The search is
// a uniform grid of cells at least as large as the largest AABB extent: tets are binned by
// the cell of their AABB's minimum corner, so overlapping tets lie in neighbouring cells.
//
// NL2set: the (node, tet) tuples of GPU_Functionality.NarrowPhaseCollisionDetection
// (GPU_Functionality.cs:565-600), de-duplicated keeping each tuple's first occurrence, in
// the order of first occurrence (a HashSet without removals enumerates in insertion order):
// a device hash table keeps each key's smallest insertion position, and the positions that
// are their key's first are compacted in order.
#pragma once

namespace icf {

constexpr int BP_DIRS = 12;

// Words of a call's report: a node id is out of range, positions are not finite, the grid has more
// cells than the buffers; and values: the grid's cells with and without margin, the pairs, the
// candidates of the fullest region.
constexpr int BP_BAD = 0, BP_NONFINITE = 1, BP_BIG = 2, BP_G = 19, BP_NCELL = 20, BP_NV = 21, BP_CAND = 22;

// Clears what the launches of one search count into.
__global__ __launch_bounds__(256) void k_bp_clear(int *__restrict__ count, int ncount, int *__restrict__ acount,
                                                  int nacount, unsigned long long *__restrict__ total, int ntotal,
                                                  Tiles ct, unsigned nct, Tiles at, unsigned nat)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ncount) count[i] = 0;
    if (i < nacount) acount[i] = 0;
    if (i < ntotal) total[i] = 0ULL;
    if (blockIdx.x == 0) {
        Tiles::clear(ct.groups, nct);
        Tiles::clear(at.groups, nat);
    }
}

// The 12 planes' value at a point, d a constant.
__device__ inline double bp_plane(int d, double x, double y, double z)
{
#pragma clang fp contract(off)
    switch (d) {
    case 0: return x;
    case 1: return y;
    case 2: return z;
    case 3: return x + y;
    case 4: return x + z;
    case 5: return y + z;
    case 6: return x - y;
    case 7: return x - z;
    case 8: return y - z;
    case 9: return x + y - z;
    case 10: return x + z - y;
    default: return y + z - x;
    }
}

// Current positions of tet t's 4 nodes; false if a node id is out of range.
__device__ inline bool bp_tet_nodes(const double *__restrict__ dn, int ns, const int *__restrict__ ie, int es, int t,
                                    double p[4][3])
{
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int n = ie[t + (size_t)es * v];
        if (n < 0 || n >= ns) return false;
#pragma unroll
        for (int k = 0; k < 3; k++) p[v][k] = dn[n + (size_t)ns * (ND_XC + k)];
    }
    return true;
}

// The tet's extent (l, h) in direction d, a constant.  All launches below compute it with this code, so
// their values agree bit for bit.
__device__ inline void bp_extent(int d, const double p[4][3], double &l, double &h)
{
    l = 1e300;
    h = -1e300;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const double x = bp_plane(d, p[v][0], p[v][1], p[v][2]);
        l = fmin(l, x);
        h = fmax(h, x);
    }
}

// Bounds of the k-DOPs: {largest AABB extent, min of the AABB minimum corners (x, y, z), max of the
// same}, one set per workgroup; BP_BLOCKS of them at most, each taking every so many tets.
constexpr int BP_NBOUNDS = 7, BP_BLOCKS = 256;
__device__ inline bool bp_is_max(int k) { return k == 0 || k >= 4; }
__device__ inline void bp_bounds256(double b[BP_NBOUNDS], double part[4][BP_NBOUNDS])
{
#pragma unroll
    for (int k = 0; k < BP_NBOUNDS; k++) {
        for (int o = 32; o > 0; o >>= 1) {
            const double w = __shfl_xor(b[k], o);
            b[k] = bp_is_max(k) ? fmax(b[k], w) : fmin(b[k], w);
        }
        if (__lane_id() == 0) part[threadIdx.x >> 6][k] = b[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BP_NBOUNDS; k++)
        for (int w = 0; w < 4; w++) b[k] = bp_is_max(k) ? fmax(b[k], part[w][k]) : fmin(b[k], part[w][k]);
}

// Per surface tet: the minimum corner of its AABB (the k-DOP's first three lo planes, which
// bin it into the grid), and the workgroup's bounds.  (With one atomic per bound and 256 tets the
// 9,700 atomics of 353,000 tets, one after the other on one cache line, made it 40 us, now 18.)  k_bp_sorted
// computes the whole k-DOP.
__global__ __launch_bounds__(256) void k_bp_kdop(const double *__restrict__ dn, int ns, const int *__restrict__ ie,
                                                 int es, int nT, double *__restrict__ lo, double *__restrict__ bounds,
                                                 Report rep)
{
#pragma clang fp contract(off)
    __shared__ double part[4][BP_NBOUNDS];
    double b[BP_NBOUNDS] = {0, 1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
    bool bad = false;
    for (int t = blockIdx.x * 256 + threadIdx.x; t < nT; t += gridDim.x * 256) {
        double p[4][3], l[3], h[3];
        if (!bp_tet_nodes(dn, ns, ie, es, t, p)) {
            bad = true;
            continue;
        }
#pragma unroll
        for (int d = 0; d < 3; d++) bp_extent(d, p, l[d], h[d]);
#pragma unroll
        for (int d = 0; d < 3; d++) lo[(size_t)d * nT + t] = l[d];
        b[0] = fmax(b[0], fmax(h[0] - l[0], fmax(h[1] - l[1], h[2] - l[2])));
#pragma unroll
        for (int k = 0; k < 3; k++) {
            b[1 + k] = fmin(b[1 + k], l[k]);
            b[4 + k] = fmax(b[4 + k], l[k]);
        }
    }
    if (bad) rep.set(BP_BAD);
    bp_bounds256(b, part);
    if (threadIdx.x < BP_NBOUNDS) {
        double v = b[0];
#pragma unroll
        for (int k = 1; k < BP_NBOUNDS; k++) v = (int)threadIdx.x == k ? b[k] : v;
        bounds[(size_t)blockIdx.x * BP_NBOUNDS + threadIdx.x] = v;
    }
}

// The search grid: cells of size cs (at least the largest AABB extent), n[k] cells per axis
// over the AABB minimum corners, stored with a margin -- one cell below and two above in x,
// one below and one above in y and z -- so that the neighbour rows a cell reads never wrap.
// Cell (x, y, z) of the margin grid has the linear key x + gx (y + gy z).  Tets are binned
// by the cell of their AABB's minimum corner; with cs >= every extent, overlapping tets lie
// in the same or neighbouring cells.  It lies in device memory: the launches are sized by what the
// last search found (with room for more), and do nothing where it does not fit (ok == 0).
struct BpGrid {
    double cs, org[3], invq;
    int n[3], gx, gy, gz, G, ncell, ok;
};

// A k-DOP plane in whole steps of cs / BP_STEPS from the grid's origin, modulo 2^16.  The steps do not
// decrease with the plane, so lo <= hi of two tets means that the steps' difference hi - lo is not
// negative, and in 16 bits that is its sign: tets of neighbouring cells are at most 3 cs apart along
// an axis, 9 cs along a sum of three, 18,432 steps.  (Where rounding of the planes could add
// to that, positions beyond 2^40 cs, all steps are 0, and every pair is left to the exact test.)
//   Tets far smaller than the largest one, whose extent makes the cells, look alike in these steps: a
// single tet drawn out to a hundred times the others' size, as before a Newton loop diverges, leaves
// all pairs of a cell as candidates.  A search that finds more than BP_DENSE candidates per tet is
// therefore repeated with the FP32 comparison behind that of the steps (168,000 tets
// in eight cells, 1.8e9 pairs: 0.6 s a call, 7 s with FP32 alone; refused without).  Surfaces in contact have
// some 5 candidates per tet (1.66M for 353,000).
constexpr long long BP_DENSE = 64;
constexpr double BP_STEPS = 2048;
__device__ inline unsigned bp_step(double plane, double org, double invq)
{
#pragma clang fp contract(off)
    if (invq == 0) return 0u;
    const double t = floor((plane - org) * invq);
    return (unsigned)(int)(t - 65536.0 * floor(t * (1.0 / 65536.0)));
}

// The grid of these bounds: cells at least the largest extent, coarsened (any size >= the extents
// finds the same pairs) until the margin grid has at most 2^24 cells.  False if they are not finite.
__device__ inline bool bp_make_grid(const double b[BP_NBOUNDS], BpGrid &g)
{
#pragma clang fp contract(off)
    double span[3];
    for (int k = 0; k < 3; k++) {
        g.org[k] = b[1 + k];
        span[k] = b[4 + k] - b[1 + k];
        if (!isfinite(g.org[k]) || !isfinite(span[k])) return false;
    }
    g.cs = b[0] > 0 ? b[0] * 1.000001 : 1.0;
    for (;;) {
        double cells = 1;
        for (int k = 0; k < 3; k++) {
            const double c = floor(span[k] / g.cs) + 1;
            g.n[k] = c < (double)(1 << 24) ? (int)c : (1 << 24);
            cells *= (double)g.n[k] + (k == 0 ? 3 : 2);
        }
        if (cells <= (double)(1 << 24)) break;
        g.cs *= 1.25;
    }
    double far = 0;
    for (int k = 0; k < 3; k++) far = fmax(far, fmax(fabs(b[1 + k]), fabs(b[4 + k])));
    g.invq = isfinite(g.cs) && far <= g.cs * 1099511627776.0 ? BP_STEPS / g.cs : 0.0;
    g.gx = g.n[0] + 3;
    g.gy = g.n[1] + 2;
    g.gz = g.n[2] + 2;
    g.G = g.gx * g.gy * g.gz;
    g.ncell = g.n[0] * g.n[1] * g.n[2];
    return true;
}

// The rank of this lane's key among all ranks taken from count[key] (bumped atomically), for
// lanes with on set (-1 for the others): one atomicAdd per run of consecutive such lanes with
// the same key -- the run's first lane reserves the run's length and its lanes take
// consecutive ranks.  Where keys repeat along a wave this replaces up to 64 atomics on one
// address, which the L2 serialises, by one.  Lanes above an inactive lane must be inactive
// too (a kernel's early exit for its last indices).
__device__ inline int run_rank(bool on, unsigned key, int *__restrict__ count)
{
    const int lane = __lane_id();
    const unsigned long long om = __ballot(on);
    const unsigned prev = __shfl_up(key, 1);
    const bool head = on && (lane == 0 || !((om >> (lane - 1)) & 1) || prev != key);
    const unsigned long long heads = __ballot(head);
    const unsigned long long ends = heads | ~om;   // lanes where a run cannot continue
    int r = -1, h = 0;
    if (on) h = 63 - __clzll(heads & ((2ULL << lane) - 1));   // the run's first lane
    if (head) {
        const unsigned long long above = lane == 63 ? 0ULL : ends & ~((2ULL << lane) - 1);
        const int len = above ? __ffsll((long long)above) - 1 - lane : 64 - lane;
        r = atomicAdd(&count[key], len);
    }
    const int base = __shfl(r, h);
    return on ? base + lane - h : -1;
}

// The grid, made by every workgroup from the nb sets of bounds and left in *grid by the first; per
// tet: its cell key and its rank among the tets of its cell (count[key] is bumped
// atomically, so the order within a cell varies from call to call; the pairs do not).
__global__ __launch_bounds__(256) void k_bp_cell(const double *__restrict__ lo, int nT,
                                                 const double *__restrict__ bounds, int nb, int capG, int capC,
                                                 BpGrid *__restrict__ grid, unsigned *__restrict__ key,
                                                 int *__restrict__ rank, int *__restrict__ count, Report rep)
{
    __shared__ double part[4][BP_NBOUNDS];
    __shared__ BpGrid g;
    double b[BP_NBOUNDS] = {0, 1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
    if ((int)threadIdx.x < nb) {
#pragma unroll
        for (int k = 0; k < BP_NBOUNDS; k++) b[k] = bounds[(size_t)threadIdx.x * BP_NBOUNDS + k];
    }
    bp_bounds256(b, part);
    if (threadIdx.x == 0) {
        const bool bad = rep.was(BP_BAD), finite = !bad && bp_make_grid(b, g);
        g.ok = finite && g.G <= capG && g.ncell <= capC;
        if (blockIdx.x == 0) {
            *grid = g;
            if (!bad && !finite) rep.set(BP_NONFINITE);
            if (finite && !g.ok) rep.set(BP_BIG);
            if (finite) {
                rep.put(BP_G, (unsigned)g.G);
                rep.put(BP_NCELL, (unsigned)g.ncell);
            }
        }
    }
    __syncthreads();
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (!g.ok || t >= nT) return;
    int c[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double f = floor((lo[(size_t)a * nT + t] - g.org[a]) / g.cs);
        c[a] = f < 0 ? 0 : (f > (double)(g.n[a] - 1) ? g.n[a] - 1 : (int)f);
    }
    const unsigned k = (unsigned)(c[0] + 1) + (unsigned)g.gx * ((unsigned)(c[1] + 1) + (unsigned)g.gy * (unsigned)(c[2] + 1));
    key[t] = k;
    rank[t] = run_rank(true, k, count);   // neighbouring tets of a mesh often share a cell
}

// out[0 .. n] = exclusive scan of v[0 .. n) in two launches (n: the grid's cells when grid is given, which
// the launches cover); the second puts the sum into word `word` of the report when not negative.
constexpr int BP_ITEMS = 8, BP_TILE = 256 * BP_ITEMS;
__global__ __launch_bounds__(256) void k_bp_tiles(const int *__restrict__ v, int n, const BpGrid *__restrict__ grid,
                                                  Tiles tiles)
{
    __shared__ unsigned part[4];
    if (!grid->ok) return;
    if (n < 0) n = grid->G;
    if ((int)blockIdx.x * BP_TILE >= n) return;
    const int k0 = (int)blockIdx.x * BP_TILE + (int)threadIdx.x * BP_ITEMS;
    unsigned x = 0;
#pragma unroll
    for (int r = 0; r < BP_ITEMS; r++)
        if (k0 + r < n) x += (unsigned)v[k0 + r];
    x = sum256(x, part);
    if (threadIdx.x == 0) tiles.put(blockIdx.x, x);
}
__global__ __launch_bounds__(256) void k_bp_scan(const int *__restrict__ v, int n, const BpGrid *__restrict__ grid,
                                                 Tiles tiles, int *__restrict__ out, int word, Report rep)
{
    __shared__ unsigned part[4];
    if (!grid->ok) return;
    if (n < 0) n = grid->G;
    if ((int)blockIdx.x * BP_TILE >= n) return;
    const int k0 = (int)blockIdx.x * BP_TILE + (int)threadIdx.x * BP_ITEMS;
    unsigned c[BP_ITEMS], x = 0, total;
#pragma unroll
    for (int r = 0; r < BP_ITEMS; r++) {
        c[r] = k0 + r < n ? (unsigned)v[k0 + r] : 0u;
        x += c[r];
    }
    const unsigned run = tiles.before(blockIdx.x, part);
    unsigned at = run + scan256(x, part, total);
#pragma unroll
    for (int r = 0; r < BP_ITEMS; r++) {
        if (k0 + r < n) out[k0 + r] = (int)at;
        at += c[r];
    }
    if ((int)(blockIdx.x + 1) * BP_TILE >= n && threadIdx.x == 0) {
        out[n] = (int)(run + total);
        if (word >= 0) rep.put(word, run + total);
    }
}

// The k-DOPs and node ids in cell order (a counting sort: first[key] is the exclusive scan
// of the cell counts): tet t goes to position j = first[key[t]] + rank[t], so that the tets
// of one cell, and of neighbouring cells, are adjacent in memory for the pair search.  Per
// position: the tet (sidx), the k-DOP in steps with the node ids (srec), the k-DOP as (lo, hi) pairs
// per direction (skd) and in FP32 rounded outward, lo down and hi up (sk32: 12 lo then 12 hi): steps
// and FP32 never reject a pair whose FP64 k-DOPs overlap.  first[L] for L = 0 .. G is then the first position of the cells with keys >= L.
struct alignas(64) BpTet {
    uint4 lo, mid, hi;      // lo of directions 0-7; lo 8-11, hi 0-3; hi 4-11: two to a word
    int4 node;
};
__global__ __launch_bounds__(256) void k_bp_sorted(const double *__restrict__ dn, int ns, int nT,
                                                   const unsigned *__restrict__ key,
                                                   const int *__restrict__ rank, const int *__restrict__ first,
                                                   const int *__restrict__ ie, int es,
                                                   const BpGrid *__restrict__ grid, int *__restrict__ sidx,
                                                   BpTet *__restrict__ srec, double2 *__restrict__ skd,
                                                   float4 *__restrict__ sk32)
{
#pragma clang fp contract(off)
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nT || !grid->ok) return;
    const int j = first[key[t]] + rank[t];
    sidx[j] = t;
    double p[4][3];
    (void)bp_tet_nodes(dn, ns, ie, es, t, p);   // node ids checked by k_bp_kdop
    const double x = grid->org[0], y = grid->org[1], z = grid->org[2], invq = grid->invq;
    float f[2 * BP_DIRS];
    unsigned q[BP_DIRS];
#pragma unroll
    for (int d = 0; d < BP_DIRS; d++) {
        double l, h;
        bp_extent(d, p, l, h);
        skd[(size_t)j * BP_DIRS + d] = make_double2(l, h);
        f[d] = __double2float_rd(l);
        f[BP_DIRS + d] = __double2float_ru(h);
        const double o = bp_plane(d, x, y, z);
        const unsigned ql = bp_step(l, o, invq), qh = bp_step(h, o, invq);
        q[d / 2] = d % 2 ? q[d / 2] | ql << 16 : ql;
        q[6 + d / 2] = d % 2 ? q[6 + d / 2] | qh << 16 : qh;
    }
    BpTet r;
    r.lo = make_uint4(q[0], q[1], q[2], q[3]);
    r.mid = make_uint4(q[4], q[5], q[6], q[7]);
    r.hi = make_uint4(q[8], q[9], q[10], q[11]);
    r.node = make_int4(ie[t], ie[t + (size_t)es], ie[t + 2 * (size_t)es], ie[t + 3 * (size_t)es]);
    srec[j] = r;
#pragma unroll
    for (int k = 0; k < 6; k++)
        sk32[(size_t)j * 6 + k] = make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
}

// The sign bits (0x80008000) of hi - lo over the 12 directions, both ways; 0 where all overlap.
typedef short s16x2 __attribute__((ext_vector_type(2)));
__device__ inline unsigned bp_sub(unsigned a, unsigned b)
{
    return __builtin_bit_cast(unsigned, (s16x2)(__builtin_bit_cast(s16x2, a) - __builtin_bit_cast(s16x2, b)));
}
__device__ inline unsigned bp_apart(const BpTet &a, const BpTet &b)
{
    unsigned x = bp_sub(b.mid.z, a.lo.x) | bp_sub(b.mid.w, a.lo.y) | bp_sub(b.hi.x, a.lo.z) | bp_sub(b.hi.y, a.lo.w);
    x |= bp_sub(b.hi.z, a.mid.x) | bp_sub(b.hi.w, a.mid.y) | bp_sub(a.mid.z, b.lo.x) | bp_sub(a.mid.w, b.lo.y);
    x |= bp_sub(a.hi.x, b.lo.z) | bp_sub(a.hi.y, b.lo.w) | bp_sub(a.hi.z, b.mid.x) | bp_sub(a.hi.w, b.mid.y);
    return x & 0x80008000u;
}

// A wave's LDS writes made visible to the wave's other lanes (no workgroup barrier).
__device__ inline void bp_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The pair search, first pass: one wave per cell of the grid's interior and slice of its tets; the
// waves of a workgroup meet only at its start.  The candidates are the cell's own tets and those of the 13 neighbouring cells
// with a larger key (each pair of cells visited once): 5 runs of consecutive keys -- (x, x+1)
// of the cell's own row, and the rows (x-1 .. x+1) at (y+1, z), (y-1, z+1), (y, z+1),
// (y+1, z+1) -- hence 5 ranges of sorted positions; in the first range only larger positions
// pair up.  The 64 lanes hold 64 candidates at a time, loaded coalesced; the own tets, BPW_OWN at a
// time, are staged in the wave's LDS and read by all lanes at once.  The 24 comparisons of a pair
// are 12 subtractions of two 16-bit steps each (bp_apart); the pairs that pass gather in a list
// and are taken 64 at a time, one per lane, through the node ids (most of them share a node, and
// are not wanted).  In FP32 with the ids compared for all pairs, 40 comparisons each with a ballot of
// its own, 353,000 tets (1.66M pairs pass) took 264 us; now 152.  The passing (own, candidate)
// positions collect in the wave's LDS buffer and leave in batches, one atomicAdd on the
// counter of the workgroup's buffer region per batch (positions beyond the region's capacity
// are only counted; the caller then grows the buffer and searches again).  What a wave holds at its end leaves with the rest of its workgroup's:
// the last wave of the workgroup to finish reserves space for all of them with one atomicAdd
// (the reservations on the one counter, one per wave, took a quarter of the kernel's time).
// Two waves per workgroup: a workgroup's LDS stays allocated until its slowest wave ends, and
// the work per cell varies several-fold, so with four waves the resident waves averaged about
// two per SIMD.  Where the grid has too few cells to fill the chip, several waves share a cell's
// tets, four at a time in turn (3,300 tets: 82 us with one wave per cell, now 12).  The second
// pass applies the exact FP64 test.
constexpr int BPW_WAVES = 2, BPW_OWN = 16, BPW_BUF = 128, BPW_LIST = 128;
struct BpWave {
    BpTet own[BPW_OWN];
    int4 node[64];                      // of the candidates
    unsigned long long buf[BPW_BUF];
    unsigned short list[BPW_LIST];      // own << 6 | candidate
};
// The candidate buffer is split into BP_PARTS regions of cap / BP_PARTS entries, each with its
// own counter (BP_PART_STRIDE counters apart, so that no two share a cache line): consecutive cells, or
// pairs of cells where a workgroup has two, append to one after the other, which spreads the
// reservations over as many addresses and neighbouring cells' candidates over all regions.
constexpr int BP_PARTS = 8, BP_PART_STRIDE = 64;

// The later passes run a grid row per region (blockIdx.y): this thread's position in the
// candidate buffer, or -1 beyond the region's count (its counter, capped at the capacity).
__device__ inline long long bp_slot(long long cap, const unsigned long long *__restrict__ total)
{
    const long long capP = cap / BP_PARTS;
    const long long o = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long n = (long long)total[(size_t)blockIdx.y * BP_PART_STRIDE];
    return o < (n < capP ? n : capP) ? (long long)blockIdx.y * capP + o : -1;
}

// Whether two tets overlap in FP32, lo and hi rounded outward.
__device__ inline bool bp_near32(const float4 *__restrict__ a, const float4 *__restrict__ b)
{
    bool hit = true;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const float4 al = a[q], ah = a[3 + q], bl = b[q], bh = b[3 + q];
        hit &= !(al.x > bh.x) & !(al.y > bh.y) & !(al.z > bh.z) & !(al.w > bh.w);
        hit &= !(bl.x > ah.x) & !(bl.y > ah.y) & !(bl.z > ah.z) & !(bl.w > ah.w);
    }
    return hit;
}

// One wave's cell and slice of the pair search (k_bp_cellwave): on return, cnt pairs are left in buf.
// FINE: pairs that pass the steps have to overlap in FP32 as well.
template <bool FINE>
__device__ inline void bp_cell_pairs(const BpTet *__restrict__ srec, const float4 *__restrict__ sk32,
                                     int exclude_shared, const BpGrid &g,
                                     const int *__restrict__ first, unsigned long long *__restrict__ total, unsigned long long *__restrict__ out,
                                     long long cap, int i, int slice, int slices, int chunk, BpWave &W, int lane,
                                     unsigned long long below, int &cnt)
{
    const int x = i % g.n[0] + 1, y = (i / g.n[0]) % g.n[1] + 1, z = i / (g.n[0] * g.n[1]) + 1;
    const int L = x + g.gx * (y + g.gy * z);
    const int s0 = first[L], s1 = first[L + 1];
    if (s0 + slice * chunk >= s1) return;
    const int gxy = g.gx * g.gy;
    const int r_lo[5] = {s0, first[L - 1 + g.gx], first[L - 1 - g.gx + gxy], first[L - 1 + gxy],
                         first[L - 1 + g.gx + gxy]};
    const int r_hi[5] = {first[L + 2], first[L + 2 + g.gx], first[L + 2 - g.gx + gxy], first[L + 2 + gxy],
                         first[L + 2 + g.gx + gxy]};
    int r_pre[6];
    r_pre[0] = 0;
#pragma unroll
    for (int r = 0; r < 5; r++) r_pre[r + 1] = r_pre[r] + r_hi[r] - r_lo[r];
    const int K = r_pre[5];
    auto flush = [&]() {
        bp_wave_sync();
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(total, (unsigned long long)cnt);
        base = __shfl(base, 0);
        for (int q = lane; q < cnt; q += 64)
            if (base + q < (unsigned long long)cap) out[base + q] = W.buf[q];
        bp_wave_sync();
        cnt = 0;
    };
    for (int a0 = s0 + slice * chunk; a0 < s1; a0 += slices * chunk) {
        const int na = min(chunk, s1 - a0);
        bp_wave_sync();   // the previous own tets are no longer read
        if (lane < na) W.own[lane] = srec[a0 + lane];
        for (int k0 = 0; k0 < K; k0 += 64) {
            const int k = k0 + lane;
            const bool valid = k < K;
            int jb = s0, own_row = 0;
#pragma unroll
            for (int r = 0; r < 5; r++)
                if (k >= r_pre[r] && k < r_pre[r + 1]) {
                    jb = r_lo[r] + (k - r_pre[r]);
                    own_row = r == 0;
                }
            // what comes after the positions of the candidate is larger than every own tet's but the
            // first range's
            const int after = own_row ? jb : INT_MAX;
            const BpTet c = srec[jb];
            W.node[lane] = c.node;
            bp_wave_sync();
            int nlist = 0;
            auto take = [&](int m) {      // the list's first m <= 64 pairs
                bp_wave_sync();
                const unsigned e = W.list[lane < m ? lane : 0];
                const int ia = (int)(e >> 6), l = (int)(e & 63);
                const int pb = __shfl(jb, l);
                bool hit = lane < m;
                if (exclude_shared) {
                    const int4 p = W.own[ia].node, q = W.node[l];
                    const int an[4] = {p.x, p.y, p.z, p.w}, bn[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                    for (int j2 = 0; j2 < 4; j2++)
#pragma unroll
                        for (int j1 = 0; j1 < 4; j1++) hit &= bn[j2] != an[j1];
                }
                if (FINE && hit) hit = bp_near32(sk32 + (size_t)(a0 + ia) * 6, sk32 + (size_t)pb * 6);
                const unsigned long long mk = __ballot(hit);
                if (hit) W.buf[cnt + __popcll(mk & below)] = ((unsigned long long)(a0 + ia) << 32) | (unsigned)pb;
                cnt += __popcll(mk);
                // the rest of the list to its front
                const unsigned short rest = W.list[min(m + lane, BPW_LIST - 1)];
                bp_wave_sync();
                nlist -= m;
                if (lane < nlist) W.list[lane] = rest;
                if (cnt > BPW_BUF - 64) flush();
            };
            for (int ia = 0; ia < na; ia++) {
                const bool near = valid & (after > a0 + ia) & (bp_apart(W.own[ia], c) == 0);
                const unsigned long long mk = __ballot(near);
                if (mk == 0) continue;
                if (near) W.list[nlist + __popcll(mk & below)] = (unsigned short)(ia << 6 | lane);
                nlist += __popcll(mk);
                if (nlist >= 64) take(64);
            }
            if (nlist) take(nlist);
            bp_wave_sync();   // the candidates are no longer read
        }
    }
}

template <bool FINE>
__global__ __launch_bounds__(64 * BPW_WAVES) void k_bp_cellwave(const BpTet *__restrict__ srec,
                                                                const float4 *__restrict__ sk32, int exclude_shared,
                                                                const BpGrid *__restrict__ grid, int slices, int chunk,
                                                                const int *__restrict__ first,
                                                                unsigned long long *__restrict__ total,
                                                                unsigned long long *__restrict__ out, long long cap)
{
    __shared__ BpWave waves[BPW_WAVES];
    __shared__ int wcnt[BPW_WAVES], done;
    if (!grid->ok) return;
    const BpGrid g = *grid;
    const int wave = threadIdx.x >> 6, lane = __lane_id();
    if (threadIdx.x == 0) done = 0;
    __syncthreads();
    const unsigned long long below = (1ULL << lane) - 1;
    int cnt = 0;
    // the slices of a cell are neighbouring waves; runs of 64 workgroups stay on one XCD, whose L2 then
    // holds the tets of neighbouring cells
    const int run = (int)blockIdx.x / 512 * 512, in = (int)blockIdx.x - run;
    const int group = run + in % 8 * 64 + in / 8;
    const int w = group * BPW_WAVES + wave, i = w / slices;
    const long long capP = cap / BP_PARTS;
    // by the group's cells (slices: 1 or an even number), not by blockIdx, whose eighths are runs of cells:
    // candidates crowd into neighbouring cells, and the fullest region decides how large the buffer has
    // to be.  All slices of a cell go to one region, which then counts the same in a repeated search,
    // whatever the order of the tets in their cells.
    const int part = (slices > 1 ? i : group) % BP_PARTS;
    total += (size_t)part * BP_PART_STRIDE;
    out += (size_t)part * capP;
    if (i < g.ncell) bp_cell_pairs<FINE>(srec, sk32, exclude_shared, g, first, total, out, capP, i, w % slices, slices, chunk,
                                         waves[wave], lane, below, cnt);
    // the workgroup's last wave out writes every wave's remaining pairs
    if (lane == 0) wcnt[wave] = cnt;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    int last = 0;
    if (lane == 0) last = atomicAdd(&done, 1) == BPW_WAVES - 1;
    if (!__shfl(last, 0)) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    int pre[BPW_WAVES + 1];
    pre[0] = 0;
#pragma unroll
    for (int v = 0; v < BPW_WAVES; v++) pre[v + 1] = pre[v] + wcnt[v];
    if (pre[BPW_WAVES] == 0) return;
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(total, (unsigned long long)pre[BPW_WAVES]);
    base = __shfl(base, 0);
#pragma unroll
    for (int v = 0; v < BPW_WAVES; v++)
        for (int q = lane; q < wcnt[v]; q += 64)
            if (base + pre[v] + q < (unsigned long long)capP) out[base + pre[v] + q] = waves[v].buf[q];
}

// The pair search, second pass: per candidate (own, candidate) position pair of the first
// pass, the exact test -- the FP64 12-direction overlap, the predicate of the reference's
// k-DOP test.  The FP32 copies decide first where they can: the outward-rounded
// values, each moved one step inward (nextafter), still overlap only if the FP64 values do
// (lo <= nextafter(lo rounded down, +inf) and hi >= nextafter(hi rounded up, -inf)), so the
// FP64 k-DOPs are read only for the pairs that are within an FP32 step of touching.  A pair
// that passes becomes (a, b), a < b its original indices (io[i] = a << 32 | b), and takes its
// rank among the pairs of the same a (count[a] bumped atomically); rank[i] = -1 for a pair
// that fails.
__global__ __launch_bounds__(256) void k_bp_exact(const double2 *__restrict__ skd, const float4 *__restrict__ sk32,
                                                  const int *__restrict__ sidx,
                                                  const unsigned long long *__restrict__ ncand, long long cap,
                                                  unsigned long long *__restrict__ io, int *__restrict__ rank,
                                                  int *__restrict__ count)
{
    const long long i = bp_slot(cap, ncand);
    if (i < 0) return;   // the region's used positions come first, so only a wave's top lanes leave
    const unsigned long long v = io[i];
    const int ja = (int)(v >> 32), jb = (int)(v & 0xffffffffULL);
    float fa[2 * BP_DIRS], fb[2 * BP_DIRS];
#pragma unroll
    for (int q = 0; q < 6; q++) {
        const float4 x = sk32[(size_t)ja * 6 + q], y = sk32[(size_t)jb * 6 + q];
        fa[4 * q] = x.x, fa[4 * q + 1] = x.y, fa[4 * q + 2] = x.z, fa[4 * q + 3] = x.w;
        fb[4 * q] = y.x, fb[4 * q + 1] = y.y, fb[4 * q + 2] = y.z, fb[4 * q + 3] = y.w;
    }
    bool sure = true;
#pragma unroll
    for (int d = 0; d < BP_DIRS; d++) {
        sure = sure & (nextafterf(fa[d], INFINITY) <= nextafterf(fb[BP_DIRS + d], -INFINITY)) &
               (nextafterf(fb[d], INFINITY) <= nextafterf(fa[BP_DIRS + d], -INFINITY));
    }
    bool hit = sure;
    if (!sure) {
        hit = true;
#pragma unroll
        for (int d = 0; d < BP_DIRS; d++) {
            const double2 u = skd[(size_t)ja * BP_DIRS + d], w = skd[(size_t)jb * BP_DIRS + d];
            hit = hit & !(u.x > w.y) & !(u.y < w.x);
        }
    }
    unsigned a = 0xffffffffu;
    if (hit) {
        const unsigned oa = (unsigned)sidx[ja], ob = (unsigned)sidx[jb];
        const unsigned b = oa < ob ? ob : oa;
        a = oa < ob ? oa : ob;
        io[i] = ((unsigned long long)a << 32) | b;
    }
    // the first pass emits the candidates of one own tet together, so a repeats along the wave
    rank[i] = run_rank(hit, a, count);
}

// The pairs grouped by a, in no particular order within a group: pair i goes to
// start[a] + rank[i] (start = exclusive scan of the counts).
__global__ __launch_bounds__(256) void k_bp_scatter(const unsigned long long *__restrict__ io,
                                                    const int *__restrict__ rank,
                                                    const unsigned long long *__restrict__ ncand, long long cap,
                                                    const int *__restrict__ start,
                                                    unsigned long long *__restrict__ grp, Report rep)
{
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        // the fullest region decides whether the buffer held every candidate
        unsigned long long most = 0;
        for (int q = 0; q < BP_PARTS; q++) most = max(most, ncand[(size_t)q * BP_PART_STRIDE]);
        rep.put(BP_CAND, (unsigned)min(most, 0xffffffffULL));
    }
    const long long i = bp_slot(cap, ncand);
    if (i < 0) return;
    const int r = rank[i];
    if (r < 0) return;
    const unsigned long long v = io[i];
    grp[start[v >> 32] + r] = v;
}

// Each grouped pair's final place: its group's start plus the number of b's in the group
// smaller than its own (the b's of a group are distinct), so the pairs come out in (a, b)
// order; those below max_pairs are written.
__global__ __launch_bounds__(256) void k_bp_place(const unsigned long long *__restrict__ grp,
                                                  const int *__restrict__ start, int nT,
                                                  const BpGrid *__restrict__ grid, long long max_pairs,
                                                  int *__restrict__ pairs)
{
    if (!grid->ok) return;
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long long)start[nT]) return;   // at most the places of the buffer
    const unsigned long long v = grp[p];
    const int a = (int)(v >> 32), b = (int)(v & 0xffffffffULL);
    const int s = start[a], e = start[a + 1];
    int r = 0;
    for (int q = s; q < e; q++) r += (int)(grp[q] & 0xffffffffULL) < b;
    const long long at = (long long)s + r;
    if (at < max_pairs) {
        pairs[2 * at] = a;
        pairs[2 * at + 1] = b;
    }
}

// NL2set: the distinct (node, tet) tuples of the candidate pairs' masks, in the order of their first
// occurrence (pair, then bit).  Every tuple goes into an open-addressing table (linear probing)
// that keeps its smallest place 8 * pair + bit; the places that are their tuple's smallest are
// counted per 256 pairs and written behind the pairs before (Tiles).  Four launches and one wait, with
// the table as large as the last call's distinct tuples ask for (a tuple without a slot is reported,
// and the host repeats the call with a table for all).  With the tuples counted, scanned and listed
// first it took 13 launches and two waits, 166 us a call on the 384,000-tet compression (1.66M
// pairs, 416,000 bits) and 122 us on one of 3,072 tets; now 73 and 35.  Three chains of dependent
// reads (masks, pairs and node ids, table) bound it: a pair has few bits, so the set bits of 256
// pairs are gathered in LDS and taken by one thread each.
constexpr unsigned long long NL2_EMPTY = ~0ULL;   // no key: node and tet ids are >= 0
constexpr int NL2_FULL = 0, NL2_TOTAL = 17, NL2_NUM = 18;   // words of the report; the last two are values
constexpr unsigned long long NL2_MAX = 1ULL << 28;          // tuples of one call, repeated ones counted
// Four slots, read in one go: a search is one read almost always.
struct alignas(64) Nl2Bucket {
    unsigned long long key[4], place[4];
};
struct Nl2Table {
    Nl2Bucket *bucket;
    unsigned long long mask;      // buckets - 1
    unsigned *bits;               // set bits per Tiles::GROUP workgroups, as Tiles keeps them
};
__device__ inline unsigned long long nl2_hash(unsigned long long k)
{
    k ^= k >> 33;
    k *= 0xff51afd7ed558ccdULL;
    k ^= k >> 33;
    return k;
}

// bit 0-3: vertex s of B inside A; bits 4-7: vertex s-4 of A inside B
__device__ inline unsigned long long nl2_key(const int *pairs, int i, int s, const int *ie, int es)
{
    const int tA = pairs[2LL * i], tB = pairs[2LL * i + 1];
    const int node = s < 4 ? ie[tB + (size_t)es * s] : ie[tA + (size_t)es * (s - 4)];
    return ((unsigned long long)(unsigned)node << 32) | (unsigned)(s < 4 ? tA : tB);
}

// list[0 .. total) = 8 * thread + bit of the workgroup's set bits, in order; total in every thread.
__device__ inline unsigned nl2_list(unsigned bits, unsigned short *list, unsigned *part)
{
    unsigned total, at = scan256((unsigned)__popc(bits), part, total);
    for (; bits; bits &= bits - 1) list[at++] = (unsigned short)(threadIdx.x * 8 + (unsigned)__ffs(bits) - 1);
    __syncthreads();
    return total;
}

__global__ __launch_bounds__(256) void k_nl2_clear(Nl2Table t, Tiles tiles, unsigned ntiles)
{
    const unsigned long long h = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (h <= 4 * t.mask + 3) {
        t.bucket[h / 4].key[h % 4] = NL2_EMPTY;
        t.bucket[h / 4].place[h % 4] = ~0ULL;
    }
    if (blockIdx.x == 0) {
        Tiles::clear(tiles.groups, ntiles);
        Tiles::clear(t.bits, ntiles);
    }
}

// A vertex belongs to some twenty tets, so a tuple comes up as often, mostly in neighbouring pairs:
// those of the same 256 pairs are found in a small table in LDS first (a tuple that finds no slot
// in it within 8 steps is taken for a new one), and only the others go to the large one.
// firsts[i] = the bits of pair i that did.
constexpr int NL2_LOCAL = 1024;
constexpr unsigned short NL2_NONE = 0xffff;
__global__ __launch_bounds__(256) void k_nl2_emit(const int *__restrict__ masks, const int *__restrict__ pairs,
                                                  int nPairs, const int *__restrict__ ie, int es, Nl2Table t,
                                                  unsigned long long probes, unsigned char *__restrict__ firsts,
                                                  Report rep)
{
    __shared__ unsigned long long lkey[NL2_LOCAL];
    __shared__ unsigned lplace[NL2_LOCAL], part[4], first[256];
    __shared__ unsigned short list[2048], at[2048];
    const int w = xcd_remap(blockIdx.x, gridDim.x), i0 = w * 256, i = i0 + (int)threadIdx.x;
    for (int h = threadIdx.x; h < NL2_LOCAL; h += 256) {
        lkey[h] = NL2_EMPTY;
        lplace[h] = ~0u;
    }
    first[threadIdx.x] = 0u;
    const unsigned total = nl2_list(i < nPairs ? (unsigned)masks[2LL * i] & 0xffu : 0u, list, part);
    if (threadIdx.x == 0) Tiles::add(t.bits, (unsigned)w, total);
    for (unsigned e = threadIdx.x; e < total; e += 256) {
        const unsigned long long k = nl2_key(pairs, i0 + (list[e] >> 3), list[e] & 7, ie, es);
        unsigned h = (unsigned)nl2_hash(k) % NL2_LOCAL;
        unsigned short slot = NL2_NONE;
        for (int n = 0; n < 8 && slot == NL2_NONE; n++, h = (h + 1) % NL2_LOCAL) {
            const unsigned long long prev = atomicCAS(&lkey[h], NL2_EMPTY, k);
            if (prev == NL2_EMPTY || prev == k) slot = (unsigned short)h;
        }
        if (slot != NL2_NONE) atomicMin(&lplace[slot], e);
        at[e] = slot;
    }
    __syncthreads();
    for (unsigned e = threadIdx.x; e < total; e += 256) {
        const unsigned short slot = at[e];
        if (slot != NL2_NONE && lplace[slot] != e) continue;
        const int l = list[e] >> 3, s = list[e] & 7;
        atomicOr(&first[l], 1u << s);
        const unsigned long long k = slot != NL2_NONE ? lkey[slot] : nl2_key(pairs, i0 + l, s, ie, es);
        const unsigned long long place = 8ULL * (unsigned)(i0 + l) + (unsigned)s;
        unsigned long long h = nl2_hash(k) & t.mask;
        bool done = false;
        for (unsigned long long n = 0; n < probes && !done; n++, h = (h + 1) & t.mask) {
            Nl2Bucket *b = t.bucket + h;
            const Nl2Bucket was = *b;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (done) continue;
                unsigned long long key = was.key[j];
                if (key == NL2_EMPTY) {
                    key = atomicCAS(&b->key[j], NL2_EMPTY, k);
                    if (key == NL2_EMPTY) key = k;
                }
                done = key == k;
                if (done && was.place[j] > place) atomicMin(&b->place[j], place);
            }
            if (n == 4 && !done && rep.is(NL2_FULL)) break;
        }
        if (!done) rep.set(NL2_FULL);
    }
    __syncthreads();
    if (i < nPairs) firsts[i] = (unsigned char)first[threadIdx.x];
}

// kept[i], the bits of pair i that came first among their 256 pairs' -> those whose tuples occur
// there first of all
__global__ __launch_bounds__(256) void k_nl2_keep(const int *__restrict__ pairs, int nPairs,
                                                  const int *__restrict__ ie, int es, Nl2Table t,
                                                  unsigned char *__restrict__ kept, Tiles tiles, Report rep)
{
    __shared__ unsigned short list[2048];
    __shared__ unsigned part[4], keep[256];
    if (rep.was(NL2_FULL)) return;
    const int w = xcd_remap(blockIdx.x, gridDim.x), i0 = w * 256, i = i0 + (int)threadIdx.x;
    keep[threadIdx.x] = 0u;
    const unsigned total = nl2_list(i < nPairs ? kept[i] : 0u, list, part);
    unsigned num = 0;
    if (total) {
        for (unsigned e = threadIdx.x; e < total; e += 256) {
            const int l = list[e] >> 3, s = list[e] & 7;
            const unsigned long long k = nl2_key(pairs, i0 + l, s, ie, es);
            unsigned long long h = nl2_hash(k) & t.mask;
            const unsigned long long place = 8ULL * (unsigned)(i0 + l) + (unsigned)s;
            for (bool found = false; !found; h = (h + 1) & t.mask) {
                const Nl2Bucket b = t.bucket[h];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (b.key[j] != k) continue;
                    found = true;
                    if (b.place[j] == place) {
                        atomicOr(&keep[l], 1u << s);
                        num++;
                    }
                }
            }
        }
        num = sum256(num, part);
        if (i < nPairs) kept[i] = (unsigned char)keep[threadIdx.x];
    }
    if (threadIdx.x == 0) tiles.put((unsigned)w, num);
}

// nl2 rows 0-1: the kept tuples at their places; those beyond ts are left out (the caller reports
// the count).
__global__ __launch_bounds__(256) void k_nl2_write(const unsigned char *__restrict__ kept,
                                                   const int *__restrict__ pairs, int nPairs,
                                                   const int *__restrict__ ie, int es, Nl2Table t, Tiles tiles,
                                                   int *__restrict__ nl2, int ts, Report rep)
{
    __shared__ unsigned part[4];
    __shared__ unsigned long long part8[4];
    unsigned long long bits = 0, total;
    for (unsigned g = threadIdx.x; g < Tiles::ngroups(gridDim.x); g += 256) bits += t.bits[(size_t)g * Tiles::STRIDE];
    (void)scan256(bits, part8, total);
    if (blockIdx.x == 0 && threadIdx.x == 0) rep.put(NL2_TOTAL, (unsigned)(total > NL2_MAX ? NL2_MAX + 1 : total));
    if (rep.was(NL2_FULL) || total > NL2_MAX) return;
    if (blockIdx.x == 0) {
        const unsigned num = tiles.total(gridDim.x, part);
        if (threadIdx.x == 0) rep.put(NL2_NUM, num);
    }
    if (tiles.sums[blockIdx.x] == 0) return;
    const int i = blockIdx.x * 256 + (int)threadIdx.x;
    unsigned m = i < nPairs ? kept[i] : 0u, all;
    unsigned at = tiles.before(blockIdx.x, part);
    at += scan256((unsigned)__popc(m), part, all);
    for (; m; m &= m - 1, at++) {
        if (at >= (unsigned)ts) break;
        const unsigned long long k = nl2_key(pairs, i, __ffs(m) - 1, ie, es);
        nl2[at] = (int)(k >> 32);
        nl2[at + (size_t)ts] = (int)(k & 0xffffffffULL);
    }
}

}  // namespace icf
