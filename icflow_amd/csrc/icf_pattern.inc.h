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
// Pairs are emitted as 64-bit keys (row << 32 | column), sorted and de-duplicated with
// hipCUB, which gives the same rows and sorted columns as the dictionary.
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
    long long out0;        // first output position of this source
};

// Number of candidate pairs per unit: K(K+1)/2, or K(K-1)/2 when strict.
__host__ __device__ inline int pat_pairs(int K, int strict) { return strict ? K * (K - 1) / 2 : K * (K + 1) / 2; }

__global__ __launch_bounds__(256) void k_pat_emit(PatSrc s, const int *__restrict__ alt, int nNodes, int N,
                                                  int cb, unsigned long long *__restrict__ keys,
                                                  int *__restrict__ err)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int P = pat_pairs(s.K, s.strict);
    if (t >= (long long)s.n * P) return;
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
    unsigned long long key = pat_none(cb);
    if (ni < 0 || ni >= nNodes || nj < 0 || nj >= nNodes) {
        atomicOr(err, 1);
    } else {
        const int a = alt[ni], b = alt[nj];
        if (a >= 0 && b >= 0 && !(s.strict && a == b)) {
            const int r = a < b ? a : b, c = a < b ? b : a;
            if (c >= N) atomicOr(err, 1);
            else key = ((unsigned long long)r << cb) | (unsigned)c;
        }
    }
    keys[s.out0 + t] = key;
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
// compare == 0: snap = the fields; else *diff = 1 if any field differs from snap.
__global__ __launch_bounds__(256) void k_pat_snap(PatFields f, long long n, int *__restrict__ snap, int compare,
                                                  int *__restrict__ diff)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int v = pat_field(f, i);
    if (!compare) snap[i] = v;
    else if (snap[i] != v) atomicOr(diff, 1);
}

// The sorted keys' distinct blocks: flag[i] = 1 where key i differs from key i-1 and is a
// block (flag[M] = 0 is set by the caller); then each flagged key goes to its scan position.
__global__ __launch_bounds__(256) void k_pat_flag(const unsigned long long *__restrict__ keys, int M, int cb,
                                                  int *__restrict__ flag)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    const unsigned long long k = keys[i];
    flag[i] = (k != pat_none(cb) && (i == 0 || keys[i - 1] != k)) ? 1 : 0;
}

__global__ __launch_bounds__(256) void k_pat_compact(const unsigned long long *__restrict__ keys, int M,
                                                     const int *__restrict__ flag, const int *__restrict__ pos,
                                                     unsigned long long *__restrict__ ukeys)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M && flag[i]) ukeys[pos[i]] = keys[i];
}

// csr_cols[k] = column of unique key k (k < nnz); csr_rows[r] = first k with row >= r.
__global__ __launch_bounds__(256) void k_pat_cols(const unsigned long long *__restrict__ ukeys, int nnz, int cb,
                                                  int *__restrict__ cols)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nnz) cols[k] = (int)(ukeys[k] & ((1ULL << cb) - 1));
}

__global__ __launch_bounds__(256) void k_pat_rows(const unsigned long long *__restrict__ ukeys, int nnz, int N, int cb,
                                                  int *__restrict__ rows)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > N) return;
    int lo = 0, hi = nnz;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)(ukeys[mid] >> cb) < r) lo = mid + 1;
        else hi = mid;
    }
    rows[r] = lo;
}

// One launch packs every unit kind: part k's waves follow part k-1's.  A wave takes one local
// row i of 64 consecutive units, and the waves of one group of units are neighbours, so that the
// node ids and altIds they share are read from memory once.
struct PackPart {
    int *base;
    int n, stride;
};
struct PackAll {
    PackPart part[3];      // elements, CZs, impacts
    long long wave1[3];    // end of the part's waves
};
__host__ __device__ inline long long pack_waves(int n, int K) { return ((long long)n + 63) / 64 * K; }

// Words of a call's report (Report).
constexpr int PACK_ERR = 0, PACK_CHANGED = 1;   // PACK_CHANGED + 2 part + (0: slots, 1: rows)

// Slot and row fields of local row i of unit u.  A slot that already names its pair -- a position
// inside row altId_i of the pattern whose column is altId_j, or -1 where there is no block -- is
// the slot the search would find (a row's columns are distinct), and is left alone: between two
// iterations with the same pattern nothing is searched or written, and the report tells the host
// that the maps built from the fields still hold.  For the 830,320 CZs of 256 batched specimens
// the call takes 118 us instead of 319 with a search per pair (and the assembly that follows no
// longer compares 0.5 GB of fields with their copies, 1,360 instead of 1,810 us); what is left is
// the reading of 36 slots and 21 columns per CZ.  Where a slot differs, the K searches of the row
// go down together, one column load each per step.
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
    if (cur_row != want_row) {
        *row = want_row;
        rowf = true;
    }
    const int r0 = ai >= 0 ? rows[ai] : 0, r1 = ai >= 0 ? rows[ai + 1] : 0;
    bool need[K], keep = true;
#pragma unroll
    for (int j = 0; j < K; j++) {
        need[j] = ai >= 0 && a[j] >= ai;
        const bool in = need[j] && cur[j] >= r0 && cur[j] < r1;
        const int c = in ? cols[cur[j]] : -1;
        keep &= need[j] ? in && c == a[j] : cur[j] == -1;
    }
    if (keep) return;
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
        if (v != cur[j]) {
            slot[(size_t)s.stride * j] = v;
            slots = true;
        }
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
