// icf_pattern.inc.h -- BCSR pattern and pcsr slot packing on the device (included by
// icf_lib.hip).
//
// Restates, for device-resident unit buffers:
//  - the static structure of MeshCollection.UpdateStaticStructureData
//    (v3Library/Geometry/Mesh/MeshCollection.cs:91-109): for every CZ and element, every pair
//    of non-anchored vertices with altId_2 >= altId_1;
//  - the dynamic structure of ImplicitModel3._addCollidingNodesToStructure
//    (ImplicitModel3.cs:177-196): every pair of an impact's non-anchored nodes with
//    altId_2 > altId_1;
//  - CSRDictionary.CreateStructure (CSRDictionary.cs:64-97): rows 0..N-1, each row's columns
//    the sorted union of its static and dynamic neighbours, slot = position;
//  - the slot / row packing of GPU_Functionality.TransferPCSR (GPU_Functionality.cs:345-416)
//    and collisionResponse (:627-665): slot(i,j) = position of (altId_i, altId_j) when both
//    nodes are non-anchored and altId_j >= altId_i, else -1; row_i = altId_i or -1.
// The pairs of elements and CZs are emitted as 64-bit keys (row, column), sorted with hipCUB and
// de-duplicated; what the impacts add is sorted row by row and merged in.  Both give the same rows
// and sorted columns as the dictionary.
#pragma once

namespace icf {

// Keys (row << cb | column) with cb bits per index, (1 << cb) > N; the largest 2cb-bit value
// marks a pair that adds no block and sorts after every block.
__host__ __device__ inline unsigned long long pat_none(int cb) { return (1ULL << (2 * cb)) - 1; }

// One unit source of the pattern: node ids base[u + stride * (field0 + i)], i < K.
struct PatSrc {
    const int *base;
    int n, stride, field0, K;
    int strict;            // 1: only altId_j > altId_i (impacts)
};

// Number of candidate pairs per unit: K(K+1)/2, or K(K-1)/2 when strict.
__host__ __device__ inline int pat_pairs(int K, int strict) { return strict ? K * (K - 1) / 2 : K * (K + 1) / 2; }

// Words of a call's report (Report): node ids or altIds differ from those kept, or are out of range
// in the static part or the impacts; the number of blocks.
constexpr int PAT_DIFF = 0, PAT_ERR_STATIC = 1, PAT_ERR_IMPACT = 2, PAT_NNZ = 16;

// Candidate pair t of a source: false when it adds no block (err: an id is out of range).
__device__ __forceinline__ bool pat_pair(const PatSrc &s, long long t, const int *__restrict__ alt, int nNodes, int N,
                                         int &r, int &c, bool &err)
{
    const int P = pat_pairs(s.K, s.strict);
    const int u = (int)(t / P);
    int p = (int)(t % P);
    // local pair (i, j), i <= j (i < j when strict), in row-major order
    int i = 0, row_len = s.strict ? s.K - 1 : s.K;
    while (p >= row_len) {
        p -= row_len;
        i++;
        row_len--;
    }
    const int j = s.strict ? i + 1 + p : i + p;
    const int ni = s.base[u + (size_t)s.stride * (s.field0 + i)];
    const int nj = s.base[u + (size_t)s.stride * (s.field0 + j)];
    if (ni < 0 || ni >= nNodes || nj < 0 || nj >= nNodes) {
        err = true;
        return false;
    }
    const int a = alt[ni], b = alt[nj];
    if (a < 0 || b < 0 || (s.strict && a == b)) return false;
    r = a < b ? a : b;
    c = a < b ? b : a;
    err = c >= N;
    return c < N;
}

// Keys of the static part's candidate pairs, elements' then CZs'; tile counts to be taken later
// are cleared.
__global__ __launch_bounds__(256) void k_pat_emit(PatSrc el, PatSrc cz, const int *__restrict__ alt, int nNodes, int N,
                                                  int cb, unsigned long long *__restrict__ keys, Tiles tiles,
                                                  unsigned ntiles, Report rep)
{
    if (blockIdx.x == 0) Tiles::clear(tiles.groups, ntiles);
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long Me = (long long)el.n * pat_pairs(4, 0), M = Me + (long long)cz.n * pat_pairs(6, 0);
    if (t >= M) return;
    int r = 0, c = 0;
    bool err = false;
    const bool block = t < Me ? pat_pair(el, t, alt, nNodes, N, r, c, err) : pat_pair(cz, t - Me, alt, nNodes, N, r, c, err);
    if (err) rep.set(PAT_ERR_STATIC);
    keys[t] = block ? ((unsigned long long)r << cb) | (unsigned)c : pat_none(cb);
}

// The node-id fields a pattern's static part is built from, as one sequence: the altId of
// every node, then the 4 node ids of each element (field by field), then the 6 of each CZ.
struct PatFields {
    const int *alt;
    int nNodes;
    const int *ie;
    int nElems, el_stride;
    const int *icz;
    int nCZs, cz_stride;
};
__device__ inline int pat_field(const PatFields &f, long long i)
{
    if (i < f.nNodes) return f.alt[i];
    i -= f.nNodes;
    if (i < 4LL * f.nElems) return f.ie[i % f.nElems + (size_t)f.el_stride * (EL_NODES + i / f.nElems)];
    i -= 4LL * f.nElems;
    return f.icz[i % f.nCZs + (size_t)f.cz_stride * (CZI_VRTS + i / f.nCZs)];
}
__global__ __launch_bounds__(256) void k_pat_snap(PatFields f, long long n, int *__restrict__ snap)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) snap[i] = pat_field(f, i);
}

// The sorted keys' distinct blocks: counted per tile, then written in order with their columns.
constexpr int PAT_ITEMS = 8, PAT_TILE = 256 * PAT_ITEMS;
__device__ inline bool pat_first(const unsigned long long *keys, long long i, long long M, int cb)
{
    if (i >= M) return false;
    const unsigned long long k = keys[i];
    return k != pat_none(cb) && (i == 0 || keys[i - 1] != k);
}

__global__ __launch_bounds__(256) void k_pat_count(const unsigned long long *__restrict__ keys, long long M, int cb,
                                                   Tiles tiles)
{
    __shared__ unsigned part[4];
    unsigned n = 0;
    for (int k = 0; k < PAT_ITEMS; k++)
        n += pat_first(keys, (long long)blockIdx.x * PAT_TILE + k * 256 + threadIdx.x, M, cb) ? 1u : 0u;
    n = sum256(n, part);
    if (threadIdx.x == 0) tiles.put(blockIdx.x, n);
}

__global__ __launch_bounds__(256) void k_pat_compact(const unsigned long long *__restrict__ keys, long long M, int cb,
                                                     Tiles tiles, unsigned long long *__restrict__ ukeys,
                                                     int *__restrict__ cols, int *__restrict__ count)
{
    __shared__ unsigned part[4];
    unsigned run = tiles.before(blockIdx.x, part), total;
    for (int k = 0; k < PAT_ITEMS; k++) {
        const long long i = (long long)blockIdx.x * PAT_TILE + k * 256 + threadIdx.x;
        const bool first = pat_first(keys, i, M, cb);
        const unsigned at = run + scan256(first ? 1u : 0u, part, total);
        run += total;
        if (!first) continue;
        ukeys[at] = keys[i];
        cols[at] = (int)(keys[i] & ((1ULL << cb) - 1));
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *count = (int)run;
}

// rows[r] = first distinct key with row >= r (count: their number, null for none)
__global__ __launch_bounds__(256) void k_pat_rows(const unsigned long long *__restrict__ ukeys,
                                                  const int *__restrict__ count, int N, int cb, int *__restrict__ rows)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > N) return;
    int lo = 0, hi = count ? *count : 0;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)(ukeys[mid] >> cb) < r) lo = mid + 1;
        else hi = mid;
    }
    rows[r] = lo;
}

// ---- what the impacts add ---------------------------------------------------------------------
// A Newton iteration with contact builds the pattern with other impacts each time: some thousands of
// candidate pairs beside a static part of up to a million blocks that stays.  The pairs that the
// static rows lack are listed row by row, each row's sorted and de-duplicated, and the rows
// written from both lists: five launches and one wait, in which the comparison of the static part's
// node ids with the kept copy is made too (the result is written only if it holds).  Sorting
// the keys, merging them with all static keys and compacting the result took about 20 launches and
// four waits: 301 us a call in the 384,000-tet compression and 176 us in one of 3,072 tets, now 62
// and 45; the launches and the wait themselves bound it.
struct PatExtra {
    int2 *item;            // candidate pair: row (-1: adds nothing), column
    int *rank;             // its place among its row's, in no particular order
    int *cnt;              // candidates per row, zero before and after the call
    int *off, *len;        // each row's first column in `raw` and `cols`, its distinct columns
    int *raw, *cols;
    unsigned *cursor;
};

// Workgroups below nsnap compare the static part's fields with their copy, the others take the
// impacts' pairs.
__global__ __launch_bounds__(256) void k_pat_extra(PatFields f, long long nfields, const int *__restrict__ snap,
                                                   unsigned nsnap, PatSrc s, int nNodes, int N,
                                                   const int *__restrict__ srow, const int *__restrict__ scol,
                                                   PatExtra x, Tiles tiles, unsigned ntiles, Report rep)
{
    if (blockIdx.x < nsnap) {
        const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
        if (i < nfields && snap[i] != pat_field(f, i)) rep.set(PAT_DIFF);
        return;
    }
    if (blockIdx.x == nsnap) {
        Tiles::clear(tiles.groups, ntiles);
        if (threadIdx.x == 0) *x.cursor = 0u;
    }
    const long long t = (long long)(blockIdx.x - nsnap) * blockDim.x + threadIdx.x;
    if (t >= (long long)s.n * pat_pairs(4, 1)) return;
    int r = -1, c = 0;
    bool err = false;
    if (!pat_pair(s, t, f.alt, nNodes, N, r, c, err)) r = -1;
    if (err) rep.set(PAT_ERR_IMPACT);
    if (r >= 0) {
        int lo = srow[r], hi = srow[r + 1];
        while (lo < hi) {
            const int mid = (lo + hi) >> 1, v = scol[mid];
            if (v < c) lo = mid + 1;
            else if (v > c) hi = mid;
            else {
                r = -1;
                break;
            }
        }
    }
    x.item[t] = make_int2(r, c);
    if (r >= 0) x.rank[t] = atomicAdd(x.cnt + r, 1);
}

// Room for the columns of 256 rows at a time.
__global__ __launch_bounds__(256) void k_pat_reserve(int N, PatExtra x)
{
    __shared__ unsigned part[4], base;
    const int r = blockIdx.x * 256 + (int)threadIdx.x;
    unsigned total;
    const unsigned at = scan256(r < N ? (unsigned)x.cnt[r] : 0u, part, total);
    if (threadIdx.x == 0) base = total ? atomicAdd(x.cursor, total) : 0u;
    __syncthreads();
    if (r < N) x.off[r] = (int)(base + at);
}

__global__ __launch_bounds__(256) void k_pat_fill(long long n, PatExtra x)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int2 e = x.item[t];
    if (e.x >= 0) x.raw[x.off[e.x] + x.rank[t]] = e.y;
}

// c[0 .. n) sorted without repetitions, in place; their number.
__device__ inline int sort_distinct(int *c, int n)
{
    int d = 0;
    for (int k = 0; k < n; k++) {
        const int v = c[k];
        int p = d;
        while (p > 0 && c[p - 1] > v) p--;
        if (p > 0 && c[p - 1] == v) continue;
        for (int q = d; q > p; q--) c[q] = c[q - 1];
        c[p] = v;
        d++;
    }
    return d;
}

// Each row's columns: rows of up to PAT_SHORT candidates by one thread each, in LDS where the 256
// rows' fit; longer ones (a node that hundreds of impacts share) by the workgroup, every candidate
// finding its place among all of them.
constexpr int PAT_SHORT = 64, PAT_LDS = 8192;
__global__ __launch_bounds__(256) void k_pat_distinct(int N, PatExtra x, Tiles tiles)
{
    __shared__ int lds[PAT_LDS], list[256];
    __shared__ unsigned part[4], nlist;
    const int r = blockIdx.x * 256 + (int)threadIdx.x;
    const int n = r < N ? x.cnt[r] : 0, o = r < N ? x.off[r] : 0;
    if (n) x.cnt[r] = 0;
    if (threadIdx.x == 0) nlist = 0;
    unsigned total, d = 0;
    const unsigned at = scan256((unsigned)n, part, total);      // ends with a barrier
    if (total == 0) {
        if (r < N) x.len[r] = 0;
        if (threadIdx.x == 0) tiles.put(blockIdx.x, 0u);
        return;
    }
    const bool fits = total <= PAT_LDS;
    if (n > PAT_SHORT) list[atomicAdd(&nlist, 1u)] = (int)threadIdx.x;
    if (fits) {
        // the 256 rows' candidates are one run
        if (threadIdx.x == 0) part[0] = (unsigned)o;
        __syncthreads();
        const int *raw = x.raw + part[0];
        for (unsigned i = threadIdx.x; i < total; i += 256) lds[i] = raw[i];
        __syncthreads();
    }
    if (n && n <= PAT_SHORT) {
        int *c = fits ? lds + at : x.raw + o;
        d = (unsigned)sort_distinct(c, n);
        for (unsigned k = 0; k < d; k++) x.cols[o + k] = c[k];
        x.len[r] = (int)d;
    } else if (n == 0 && r < N) x.len[r] = 0;
    __syncthreads();
    for (unsigned l = 0; l < nlist; l++) {
        const int rl = (int)blockIdx.x * 256 + list[l];
        __shared__ int ln;
        if (list[l] == (int)threadIdx.x) ln = n;
        __syncthreads();
        const int m = ln, lo = x.off[rl];
        int *raw = x.raw + lo, *cols = x.cols + lo;
        unsigned kept = 0;
        for (int i = threadIdx.x; i < m; i += 256) {      // repetitions out
            const int v = raw[i];
            int j = 0;
            while (raw[j] != v) j++;
            cols[i] = j == i ? v : INT_MAX;
            kept += j == i ? 1u : 0u;
        }
        kept = sum256(kept, part);
        for (int i = threadIdx.x; i < m; i += 256) {
            const int v = cols[i];
            if (v == INT_MAX) continue;
            int p = 0;
            for (int j = 0; j < m; j++) p += cols[j] < v ? 1 : 0;
            raw[p] = v;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < (int)kept; i += 256) cols[i] = raw[i];
        if (list[l] == (int)threadIdx.x) {
            d = kept;
            x.len[r] = (int)kept;
        }
        __syncthreads();
    }
    d = sum256(d, part);
    if (threadIdx.x == 0) tiles.put(blockIdx.x, d);
}

// First i of a[0 .. n), ascending, with a[i] >= v.
__device__ inline int lower_bound(const int *a, int n, int v)
{
    int lo = 0;
    while (lo < n) {
        const int mid = (lo + n) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else n = mid;
    }
    return lo;
}
// Last i of a[0 .. 256] with a[i] <= v, a ascending, a[0] <= v < a[256].
__device__ inline int row_of(const int *a, int v)
{
    int lo = 0;
    for (int s = 128; s > 0; s >>= 1) lo += a[lo + s] <= v ? s : 0;
    return lo;
}

// The pattern: 256 rows per workgroup, whose static blocks are one run (read and written in order);
// nothing is written when the kept part proved stale, an id out of range or max_nnz too small.
__global__ __launch_bounds__(256) void k_pat_write(const int *__restrict__ srow, const int *__restrict__ scol, int N,
                                                   bool extra, PatExtra x, Tiles tiles, unsigned ntiles, int max_nnz,
                                                   int *__restrict__ rows, int *__restrict__ cols, Report rep)
{
    __shared__ int so[257], xo[257], xoff[256];
    __shared__ unsigned part[4];
    if (rep.was(PAT_DIFF) || rep.was(PAT_ERR_STATIC) || rep.was(PAT_ERR_IMPACT)) return;
    const unsigned nnz = (unsigned)srow[N] + (extra ? tiles.total(ntiles, part) : 0u);
    if (blockIdx.x == 0 && threadIdx.x == 0) rep.put(PAT_NNZ, nnz);
    if (nnz > (unsigned)max_nnz) return;
    const int tid = (int)threadIdx.x, r = (int)blockIdx.x * 256 + tid;
    unsigned total = 0, at = 0, before = 0;
    if (extra) {
        before = tiles.before(blockIdx.x, part);
        at = scan256(r < N ? (unsigned)x.len[r] : 0u, part, total);
    }
    so[tid] = srow[min(r, N)];
    xo[tid] = (int)at;
    if (extra && r < N) xoff[tid] = x.off[r];
    if (tid == 255) {
        so[256] = srow[min(r + 1, N)];
        xo[256] = (int)total;
    }
    if (r <= N) rows[r] = so[tid] + (int)(before + at);
    __syncthreads();
    for (int i = so[0] + tid; i < so[256]; i += 256) {
        const int l = row_of(so, i), c = scol[i], nx = xo[l + 1] - xo[l];
        cols[i + (int)before + xo[l] + (nx ? lower_bound(x.cols + xoff[l], nx, c) : 0)] = c;
    }
    for (int i = tid; i < (int)total; i += 256) {
        const int l = row_of(xo, i), c = x.cols[xoff[l] + i - xo[l]];
        cols[so[l] + (int)before + i + lower_bound(scol + so[l], so[l + 1] - so[l], c)] = c;
    }
}

// One launch packs every unit kind: part k's waves follow part k-1's.  A wave takes one local
// row i of 64 consecutive units, and the waves of one group of units are neighbours, so that the
// node ids and altIds they share are read from memory once.
struct PackPart {
    int *base;
    int n, stride;
    // copies of the slot and row fields that a slot map was built from (field after field, n units
    // each), or null
    const int *slots, *rows;
};
struct PackAll {
    PackPart part[3];      // elements, CZs, impacts
    long long wave1[3];    // end of the part's waves
};
__host__ __device__ inline long long pack_waves(int n, int K) { return ((long long)n + 63) / 64 * K; }

// Words of a call's report (Report): an error; fields that are not what their slot map was built from.
constexpr int PACK_ERR = 0, PACK_CHANGED = 1;   // PACK_CHANGED + 2 part + (0: slots, 1: rows)

// Slot and row fields of local row i of unit u.  A slot that already names its pair -- a position
// inside row altId_i of the pattern whose column is altId_j, or -1 where there is no block -- is
// the slot the search would find (a row's columns are distinct), and is left alone: between two
// iterations with the same pattern nothing is searched or written.  Whether the maps still hold is
// another matter: a slot may be right because another context or a kernel of the caller's wrote it
// since, so what is in the fields at the end is held against the copy that the map was built from,
// written here or not.  For the 830,320 CZs of 256 batched specimens the call took 319 us with a
// search per pair, 118 without, 135 with the comparison (and the assembly that follows
// no longer compares 0.5 GB of fields with their copies, 1,360 instead of 1,810 us); what is left is
// the reading of 36 slots, their copies and 21 columns per CZ.  Where a slot differs, the K searches
// of the row go down together, one column load each per step.
template <int K>
__device__ __forceinline__ void pack_row(const PackPart &s, int u, int i, int node0, int slot0, int row0,
                                         const int *__restrict__ alt, int nNodes, const int *__restrict__ rows,
                                         const int *__restrict__ cols, int N, bool &err, bool &slots, bool &rowf)
{
    int nd[K], a[K], cur[K];
#pragma unroll
    for (int j = 0; j < K; j++) nd[j] = s.base[u + (size_t)s.stride * (node0 + j)];
    int *slot = s.base + u + (size_t)s.stride * (slot0 + i * K);
#pragma unroll
    for (int j = 0; j < K; j++) cur[j] = slot[(size_t)s.stride * j];
    int *row = s.base + u + (size_t)s.stride * (row0 + i);
    const int cur_row = *row;
    int was[K];                            // no copy: nothing to differ from
#pragma unroll
    for (int j = 0; j < K; j++) was[j] = s.slots ? s.slots[u + (size_t)s.n * (i * K + j)] : cur[j];
    const int was_row = s.rows ? s.rows[u + (size_t)s.n * i] : cur_row;
    int ai = -1;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < K; j++) {
        const bool out = nd[j] < 0 || nd[j] >= nNodes;
        a[j] = out ? -1 : alt[nd[j]];
        bad |= out || a[j] >= N;
        if (a[j] >= N) a[j] = -1;
        if (j == i) ai = a[j];
    }
    err |= bad;
    const int want_row = ai >= 0 ? ai : -1;
    if (cur_row != want_row) *row = want_row;
    rowf |= was_row != want_row;
    const int r0 = ai >= 0 ? rows[ai] : 0, r1 = ai >= 0 ? rows[ai + 1] : 0;
    bool need[K], keep = true;
#pragma unroll
    for (int j = 0; j < K; j++) {
        need[j] = ai >= 0 && a[j] >= ai;
        const bool in = need[j] && cur[j] >= r0 && cur[j] < r1;
        const int c = in ? cols[cur[j]] : -1;
        keep &= need[j] ? in && c == a[j] : cur[j] == -1;
    }
    if (keep) {
#pragma unroll
        for (int j = 0; j < K; j++) slots |= was[j] != cur[j];
        return;
    }
    int at[K];
#pragma unroll
    for (int j = 0; j < K; j++) at[j] = r0;
    for (int len = r1 - r0; len > 1;) {      // the last position whose column is <= a[j]
        const int half = len >> 1;
#pragma unroll
        for (int j = 0; j < K; j++) at[j] += cols[at[j] + half] <= a[j] ? half : 0;
        len -= half;
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
        int v = -1;
        if (need[j]) {
            if (r1 > r0 && cols[at[j]] == a[j]) v = at[j];
            else err = true;
        }
        if (v != cur[j]) slot[(size_t)s.stride * j] = v;
        slots |= was[j] != v;
    }
}

// Also resets the CZ flags that TransferPCSR resets (GPU_Functionality.cs:384-386): current
// failed, tentative failed, tentative damaged.
__global__ __launch_bounds__(256) void k_pack_pcsr(PackAll s, const int *__restrict__ alt, int nNodes,
                                                   const int *__restrict__ rows, const int *__restrict__ cols, int N,
                                                   Report rep)
{
    long long w = (long long)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (w >= s.wave1[2]) return;
    const int k = w < s.wave1[0] ? 0 : w < s.wave1[1] ? 1 : 2;
    if (k) w -= s.wave1[k - 1];
    const PackPart &p = s.part[k];
    const int K = k == 1 ? 6 : 4;
    const int u = (int)(w / K) * 64 + (int)__lane_id(), i = (int)(w % K);
    bool err = false, slots = false, rowf = false;
    if (u < p.n) {
        if (k == 1) {
            pack_row<6>(p, u, i, CZI_VRTS, CZI_SLOTS, CZI_ROWS, alt, nNodes, rows, cols, N, err, slots, rowf);
            if (i < 3) {
                const int f = i == 0 ? CZI_FAILED : i == 1 ? CZI_TFAILED : CZI_TDAMAGED;
                p.base[u + (size_t)p.stride * f] = 0;
            }
        } else {
            static_assert(EL_NODES == CR_NODES && EL_SLOTS == CR_SLOTS && EL_ROWS == CR_ROWS, "same fields");
            pack_row<4>(p, u, i, EL_NODES, EL_SLOTS, EL_ROWS, alt, nNodes, rows, cols, N, err, slots, rowf);
        }
    }
    if (err) rep.set(PACK_ERR);
    if (slots) rep.set(PACK_CHANGED + 2 * k);
    if (rowf) rep.set(PACK_CHANGED + 2 * k + 1);
}

}  // namespace icf
