// icf_reduce.inc.h -- deterministic scatter-free assembly (included by icf_lib.hip).
//
// The reference scatters every unit's blocks with a CAS-loop atomicAdd2
// (elem_kernels9/atomic_add.h:1-13, AssembleBCSR12/18), so the summation order in each BCSR
// slot is arbitrary.  Here assembly is a gather:
//
//   slot map  (built when a pcsr array changes): for every key (BCSR slot, rhs row or node)
//             the sorted list of 32-bit codes (kind, unit, local index) that contribute to it.
//             Sorting by code orders contributions exactly like a sequential loop over
//             kinds (elements, CZs, contacts), units and the reference's local loops.
//   phase 2   one thread per key walks its list, rebuilds each contribution from the unit's
//             staged record and adds it into an FP64 accumulator, then writes the key once.
//
// Results are therefore bitwise reproducible and independent of launch order.
#pragma once

namespace icf {

// One pcsr-style key source: keys are base[u + stride * (field0 + q)], q < nq, u < n.
struct MapSrc {
    const int *base;
    int n, stride, field0, nq;
    uint32_t kind;
};

// Largest key of a source: grid-stride over the q-major enumeration (adjacent threads read
// adjacent units of one field), block maximum, one atomic per block.
__global__ __launch_bounds__(256) void k_map_maxkey(MapSrc s, int *__restrict__ maxkey)
{
    __shared__ int part[4];
    const long long tot = (long long)s.n * s.nq;
    int key = -1;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += (long long)gridDim.x * blockDim.x) {
        const int q = (int)(i / s.n), u = (int)(i % s.n);
        key = max(key, s.base[u + (size_t)s.stride * (s.field0 + q)]);
    }
    for (int off = 32; off > 0; off >>= 1) key = max(key, __shfl_xor(key, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = key;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int m = max(max(part[0], part[1]), max(part[2], part[3]));
        if (m >= 0) atomicMax(maxkey, m);
    }
}

// ---- building slot maps ----------------------------------------------------------------------
// The maps a call needs and does not have are built together, in five launches and without a word
// from the host in between: count (each contribution also takes its rank among its key's), block
// sums, their scan, offsets with the lists of keys that have contributions, fill, sort.  Every
// buffer is sized by what it could hold, so nothing waits for a count; the host reads the number
// of keys to visit and the errors from the report, after one wait.  A Newton loop with contact
// builds the impacts' three maps in each iteration (the impacts change), and the first one of a step in
// which CZs failed those of the elements and CZs: with the chunk tables of the value reductions
// laid out on the host and allocations in between the collision response of the 384,000-tet
// compression took 6.7 ms, 0.18 ms as it is, the assembly after CZs failed on the 15,360-tet beam 1.0
// ms, now 0.17.  The atomics of the count bound large maps, the five launches small ones.
constexpr int MAX_JOBS = 3, MAX_MAP_SRCS = 6;
constexpr int SCAN_ITEMS = 8, SCAN_TILE = 256 * SCAN_ITEMS;
struct MapJobs {
    int njob, nsrc;
    MapSrc src[MAX_MAP_SRCS];
    int job[MAX_MAP_SRCS];              // the map a source belongs to
    unsigned blk0[MAX_MAP_SRCS + 1];    // first workgroup of a source: nq for each 256 units
    long long at[MAX_MAP_SRCS];         // the source's place in `rank`
    int *snap[MAX_MAP_SRCS];            // copy of the source's fields, as they are counted
    int nkeys[MAX_JOBS];
    bool vals[MAX_JOBS];                // keys are BCSR blocks
    long long cnt0[MAX_JOBS];           // the map's place in `cnt` (nkeys counts)
    unsigned tile0[MAX_JOBS + 1];       // first scan tile of a map (one at least)
    unsigned sort0[MAX_JOBS + 1];       // first sorting workgroup of a map
    int *off[MAX_JOBS];                 // nkeys + 1: first code of each key
    uint32_t *codes[MAX_JOBS];
    int *keys[MAX_JOBS], *loff[MAX_JOBS];   // the keys with contributions and their first codes, or null
};
// words of the report (MAP_NLIST holds values: no other call's words are there)
constexpr int MAP_ERR = 0, LINK_ERR = 8, SNAP_DIFF = 10, MAP_NLIST = 13;
static_assert(MAP_NLIST + MAX_JOBS <= REPORT_WORDS, "report words");

// Source, unit and field of this thread; false beyond the units.  All fields of 256 units are taken
// by neighbouring workgroups of one XCD, which so keeps the lines of their keys in its L2 (fields after
// fields, dealt over all XCDs, the count took 254 us for 5.8M contributions, now 229, the fill 98, now 62).
__device__ inline bool map_place(const MapJobs &J, int &k, int &u, int &q, unsigned nb = gridDim.x)
{
    unsigned b = (unsigned)xcd_remap(blockIdx.x, (int)nb);
    k = 0;
    while (k + 1 < J.nsrc && b >= J.blk0[k + 1]) k++;
    b -= J.blk0[k];
    q = (int)(b % (unsigned)J.src[k].nq);
    u = (int)(b / (unsigned)J.src[k].nq) * 256 + (int)threadIdx.x;
    return u < J.src[k].n;
}

// cnt (zero on entry) += the contributions of each key; rank[i] = the contribution's place among
// its key's, in no particular order.
__global__ __launch_bounds__(256) void k_map_count(MapJobs J, int *__restrict__ cnt, int *__restrict__ rank, Report rep)
{
    int k, u, q;
    if (!map_place(J, k, u, q)) return;
    const MapSrc &s = J.src[k];
    const int key = s.base[u + (size_t)s.stride * (s.field0 + q)];
    const size_t i = (size_t)q * s.n + u;
    J.snap[k][i] = key;
    if (key < 0) return;
    const int j = J.job[k];
    if (key >= J.nkeys[j]) rep.set(MAP_ERR + j);
    else rank[J.at[k] + i] = atomicAdd(&cnt[J.cnt0[j] + key], 1);
}

// Counts and keys with contributions travel through the scan together: (keys << 32) + count.
__device__ inline unsigned long long scan_item(int c) { return c > 0 ? (1ULL << 32) + (unsigned)c : 0ULL; }

// The map a scan tile belongs to, and the first key of the tile.
__device__ inline int tile_job(const MapJobs &J, int &k0)
{
    int j = 0;
    while (j + 1 < J.njob && blockIdx.x >= J.tile0[j + 1]) j++;
    k0 = (int)(blockIdx.x - J.tile0[j]) * SCAN_TILE;
    return j;
}

// Eight consecutive keys per thread, so that a tile takes one scan over its threads.
__global__ __launch_bounds__(256) void k_map_tiles(MapJobs J, const int *__restrict__ cnt,
                                                   unsigned long long *__restrict__ sums)
{
    __shared__ unsigned long long part[4];
    int k0;
    const int j = tile_job(J, k0);
    k0 += (int)threadIdx.x * SCAN_ITEMS;
    unsigned long long v = 0, total;
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; r++)
        if (k0 + r < J.nkeys[j]) v += scan_item(cnt[J.cnt0[j] + k0 + r]);
    (void)scan256(v, part, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// First code of every key, the list of keys with contributions; cnt is left zero for the next maps.
// Every tile adds up the map's tiles before it; its last one ends the offsets and reports the length
// of the list.
__global__ __launch_bounds__(256) void k_map_offsets(MapJobs J, int *__restrict__ cnt,
                                                     const unsigned long long *__restrict__ sums, Report rep)
{
    __shared__ unsigned long long part[4];
    int k0;
    const int j = tile_job(J, k0);
    k0 += (int)threadIdx.x * SCAN_ITEMS;
    int c[SCAN_ITEMS];
    unsigned long long v = 0, before = 0, run, total;
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; r++) {
        c[r] = k0 + r < J.nkeys[j] ? cnt[J.cnt0[j] + k0 + r] : 0;
        v += scan_item(c[r]);
    }
    for (unsigned t = J.tile0[j] + threadIdx.x; t < blockIdx.x; t += 256) before += sums[t];
    (void)scan256(before, part, run);
    unsigned long long x = run + scan256(v, part, total);
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; r++) {
        const int k = k0 + r;
        if (k >= J.nkeys[j]) break;
        const int first = (int)(x & 0xffffffffULL);
        J.off[j][k] = first;
        if (c[r]) {
            cnt[J.cnt0[j] + k] = 0;
            if (J.keys[j]) {
                const int p = (int)(x >> 32);
                J.keys[j][p] = k;
                J.loff[j][p] = first;
            }
        }
        x += scan_item(c[r]);
    }
    if (blockIdx.x + 1 == J.tile0[j + 1] && threadIdx.x == 0) {
        const unsigned long long all = run + total;
        const int n = (int)(all >> 32), e = (int)(all & 0xffffffffULL);
        J.off[j][J.nkeys[j]] = e;
        if (J.loff[j]) J.loff[j][n] = e;
        rep.put(MAP_NLIST + j, (unsigned)n);
    }
}

__global__ __launch_bounds__(256) void k_map_fill(MapJobs J, const int *__restrict__ rank)
{
    int k, u, q;
    if (!map_place(J, k, u, q)) return;
    const size_t i = (size_t)q * J.src[k].n + u;
    const int key = J.snap[k][i], j = J.job[k];
    if (key < 0 || key >= J.nkeys[j]) return;
    const uint32_t kind = J.src[k].kind;
    const uint32_t local = J.vals[j] && kind == KIND_CZ ? czv_code((uint32_t)q) : (uint32_t)q;
    J.codes[j][J.off[j][key] + rank[J.at[k] + i]] = make_code(kind, (uint32_t)u, local);
}

__device__ inline void sort_codes(uint32_t *c, int b, int e)
{
    for (int i = b + 1; i < e; i++) {
        const uint32_t v = c[i];
        int p = i - 1;
        while (p >= b && c[p] > v) {
            c[p + 1] = c[p];
            p--;
        }
        c[p + 1] = v;
    }
}

// Each key's codes ascending: 256 consecutive keys per workgroup, whose codes are one run, sorted
// in LDS by one thread per key (insertion: a block receives a few tens of contributions at most);
// in place where the run does not fit, a chain of dependent loads and stores per key.  256 rhs rows have
// some 4,400 contributions, 4,954 at most in the meshes measured; with room for 4,096 four
// fifths of their workgroups sorted in place: the three maps of the 15,360-tet beam took 62 us, now 34,
// those of the 384,000-tet compression 140, now 92.  6,144 and 8,192 take 100 and 131 there: less of the chip's LDS is left for other workgroups.
constexpr int SORT_CAP = 5120;
__global__ __launch_bounds__(256) void k_map_sort(MapJobs J)
{
    __shared__ uint32_t lds[SORT_CAP];
    int j = 0;
    while (j + 1 < J.njob && blockIdx.x >= J.sort0[j + 1]) j++;
    const int n = J.nkeys[j], k0 = (int)(blockIdx.x - J.sort0[j]) * 256, k1 = min(k0 + 256, n);
    const int *off = J.off[j];
    uint32_t *codes = J.codes[j];
    const int c0 = off[k0], c1 = off[k1], k = k0 + (int)threadIdx.x;
    const int b = k < k1 ? off[k] : 0, e = k < k1 ? off[k + 1] : 0;
    if (c1 - c0 > SORT_CAP) {
        sort_codes(codes, b, e);
        return;
    }
    for (int i = threadIdx.x; i < c1 - c0; i += 256) lds[i] = codes[c0 + i];
    __syncthreads();
    if (e > b) sort_codes(lds, b - c0, e - c0);
    __syncthreads();
    for (int i = threadIdx.x; i < c1 - c0; i += 256) codes[c0 + i] = lds[i];
}

// ---- slots that only moved -------------------------------------------------------------------
// A Newton iteration with contact has the units of the last one, but other impacts' blocks between
// theirs: every slot moves up or down, their order stays, and with it the codes.  Then the map needs
// new offsets alone: moved[old slot] = new slot is taken from the fields, all fields are held
// against it, the lengths of the runs go to the new slots, and their scan has to put each run
// where it was (which also shows that no two slots became one); anything else is reported, and the map is
// built from the fields.  No atomics, no sort, and the codes are not written: the assembly of an
// iteration of the 384,000-tet compression takes 254 us instead of 492, of one with 44,574 tets 96
// instead of 157.  Two passes over 5.8M fields bound it.
constexpr int MAP_MOVED = 3;        // word of the report: not so
__global__ __launch_bounds__(256) void k_map_move(MapJobs J, int *__restrict__ moved, Report rep)
{
    int k, u, q;
    if (!map_place(J, k, u, q)) return;
    const MapSrc &s = J.src[k];
    const int old = J.snap[k][(size_t)q * s.n + u], key = s.base[u + (size_t)s.stride * (s.field0 + q)];
    if ((old < 0) != (key < 0) || key >= J.nkeys[0]) rep.set(MAP_MOVED);
    else if (old >= 0 && moved[old] != key) moved[old] = key;
}

// Workgroups below `places` compare the fields and copy them; the others take the runs of the old slots.
__global__ __launch_bounds__(256) void k_map_moved(MapJobs J, unsigned places, const int *__restrict__ moved,
                                                   const int *__restrict__ off, int nold, int *__restrict__ cnt,
                                                   Report rep)
{
    if (rep.was(MAP_MOVED)) return;
    if (blockIdx.x >= places) {
        const int k = (int)(blockIdx.x - places) * 256 + (int)threadIdx.x;
        const int n = k < nold ? off[k + 1] - off[k] : 0;
        if (n) cnt[moved[k]] = n;
        return;
    }
    int k, u, q;
    if (!map_place(J, k, u, q, places)) return;
    const MapSrc &s = J.src[k];
    const size_t i = (size_t)q * s.n + u;
    const int old = J.snap[k][i], key = s.base[u + (size_t)s.stride * (s.field0 + q)];
    if (old < 0) return;
    if (moved[old] != key) rep.set(MAP_MOVED);
    if (old != key) J.snap[k][i] = key;
}

__global__ __launch_bounds__(256) void k_map_runs(const int *__restrict__ moved, const int *__restrict__ off, int nold,
                                                  const int *__restrict__ now, Report rep)
{
    if (rep.was(MAP_MOVED)) return;
    const int k = blockIdx.x * 256 + (int)threadIdx.x;
    if (k >= nold || off[k] == off[k + 1]) return;
    if (now[moved[k]] != off[k] || now[moved[k] + 1] != off[k + 1]) rep.set(MAP_MOVED);
}

// Whether a source's fields still are what the map was built from.
__global__ __launch_bounds__(256) void k_snap_cmp(MapJobs J, Report rep)
{
    int k, u, q;
    if (!map_place(J, k, u, q)) return;
    const MapSrc &s = J.src[k];
    if (J.snap[k][(size_t)q * s.n + u] != s.base[u + (size_t)s.stride * (s.field0 + q)]) rep.set(SNAP_DIFF + J.job[k]);
}

// Chunk shape of the staged BCSR-value reduction: keys per workgroup (one thread each; the
// workgroup size) and contributions staged in LDS at a time, STAGE FP32 or STAGE/2 FP64 values x 9
// per key.  STAGE = 2 is the least that still holds the chunk's output blocks (9 doubles per key)
// when they leave through the same LDS; a smaller buffer lets more workgroups share a CU, a
// larger one takes the contributions (about 5 per key) in fewer rounds.  The library's autotuner
// picks the shape per role (overwrite or accumulate map, FP32 or FP64 staging) by timing the
// candidates.  Every shape gives the same values: each key's contributions are added in list
// order whatever the chunking.
constexpr int NKC = 4, NSC = 2, NCAND = NKC * NSC;       // candidate key limits x stagings
constexpr int KEY_CANDS[NKC] = {64, 128, 256, 512};
constexpr int STAGE_CANDS[NSC] = {2, 3};
__host__ __device__ constexpr int cand_keys(int c) { return KEY_CANDS[c / NSC]; }
__host__ __device__ constexpr int cand_stage(int c) { return STAGE_CANDS[c % NSC]; }
constexpr int CAND_FP32 = 2 * NSC + 0, CAND_FP64 = 2 * NSC + 1;   // a context's shape until tuned or set
// Launches of roles that are neither tuned nor set take 128 keys, 3 FP32 or 1.5 FP64 contributions
// per key.  Time of the fused value launch, and of the other shapes of 64 to 256 keys (us): 256
// batched specimens mixed 584 (604-653), 787,000 tets FP64 176 (173-196), 24 specimens FP64 60.6
// (60.1-72.4), 146,000 tets mixed 28.3 (25.9-30.4).
constexpr int CAND_UNTUNED = 1 * NSC + 1;
// ... and where that leaves most of the chip idle, up to 98,304 blocks to overwrite, one wave of 64
// keys with room for all of their contributions: 14.5 against 16.5 us with 128 keys (7,900 blocks), 17.8
// against 20.8 (33,800), 18.0 against 19.8 (93,800).  Beyond, its LDS (37 KB a wave) leaves the rest
// waiting: 20.9 against 21.2 us in FP64 and 24.8 against 20.6 mixed at 109,800, 32.3 against 22.5 and 30.2
// against 21.0 at 130,800.  In such launches both candidates of 64 keys take that room, whatever their
// staging, so that the tuner and the callers that set a shape have it too (with 2 or 3 a key they
// took 16.1 to 17.4 us, 20.5 and 21.5, 22.2 and 23.7).  (Impacts add few to a block, which any shape takes in
// one round.)
constexpr int CAND_SMALL = 0 * NSC + 1, SMALL_KEYS = cand_keys(CAND_SMALL), SMALL_STAGE = 16, VALS_SMALL = 3 << 15;
template <typename L, int KEYS, int STAGE>
__host__ __device__ constexpr int flat_cap() { return sizeof(L) == 4 ? STAGE * KEYS : STAGE * KEYS / 2; }
// bytes of LDS of a value reduction: the staged contributions, then the list of long keys
template <typename L, int KEYS, int STAGE>
__host__ __device__ constexpr int vals_stage() { return flat_cap<L, KEYS, STAGE>() * 9 * (int)sizeof(L); }
template <typename L, int KEYS, int STAGE>
__host__ __device__ constexpr int vals_lds() { return vals_stage<L, KEYS, STAGE>() + 2 * KEYS + 4 * (KEYS / 64); }

// Staged per-unit records of the current call.
struct Stage {
    const double *tet_rhs;  // node part i of tet u at (i * tplane + u) * 3
    const void *tan;        // tangent records: tets (isotropic: node i's (g~, V) of tet u at record
                            // i * tplane + u), and from 8-byte word cz_word on the CZs'
    uint32_t cz_word;
    int tplane;             // tet plane stride (the staged tet count, rounded up to 64)
    const double *cz_rhs;
    const void *ct_tan;     // impact tangent blocks (float in mixed mode)
    const double *ct_f;     // impact forces
    double stiff, mcoef;   // tet LHS coefficients (element_kernels2.h:239-240)
};

// One contribution to a node force or rhs row.
struct Part {
    double x, y, z;
};
__device__ inline Part part_of(const Stage &sv, uint32_t code)
{
    const uint32_t kind = code_kind(code), u = code_unit(code), q = code_q(code);
    const double *p;
    bool neg = false;
    if (kind == KIND_TET) p = sv.tet_rhs + ((size_t)q * sv.tplane + u) * 3;
    else if (kind == KIND_CZ) {
        neg = q >= 3;
        p = sv.cz_rhs + (size_t)u * CZ_RHS_REC + 3 * (neg ? q - 3 : q);
    } else p = sv.ct_f + (size_t)u * CT_F_REC + 3 * q;
    const f64x2 v = *(const f64x2 *)p;
    const double z = p[2];
    return neg ? Part{-v.x, -v.y, -z} : Part{v.x, v.y, z};
}

// The values of one isotropic tet or CZ contribution, loaded by the same instructions whichever it
// is (a wave usually has both).  Places are counted in 8-byte words from the start of the tangent
// records, tets' then CZs' (Stage::tan): 32 bits hold them for 2^24 units of each, and a place is a
// few 24-bit products and one select.
template <typename T>
struct TanLoad;
__device__ inline const double *tan_word(const Stage &sv, uint32_t at) { return (const double *)sv.tan + at; }
// i * tplane + u, node i's place in the planes of tet u (tplane is a multiple of 64 up to 2^24)
__device__ inline uint32_t tet_at(const Stage &sv, uint32_t i, uint32_t u)
{
    return (__umul24(i, (uint32_t)sv.tplane >> 6) << 6) + u;
}
template <>
struct TanLoad<float> {
    f32x4 a, b;      // tet: (g~_i, V), (g~_j, V); CZ: values 0-3 and 2-5 of the pair's six
    __device__ inline void load(const Stage &sv, uint32_t code)
    {
        const uint32_t u = code_unit(code), cz = sv.cz_word + __umul24(u, CZ_TAN_REC / 2) + 3 * czv_pair(code);
        const bool tet = code_kind(code) == KIND_TET;
        a = *(const f32x4 *)tan_word(sv, tet ? 2 * tet_at(sv, code_q(code) >> 2, u) : cz);
        b = *(const f32x4 *)tan_word(sv, tet ? 2 * tet_at(sv, code_q(code) & 3, u) : cz + 1);
    }
    __device__ inline void values(float w[9], uint32_t code, float stiff, float mcoef) const
    {
        if (code_kind(code) == KIND_TET) {
            TetIso<float> t;
            t.gi = make_float4(a.x, a.y, a.z, a.w);
            t.gj = make_float4(b.x, b.y, b.z, b.w);
            t.ij = (int)code_q(code);
            t.values(w, stiff, mcoef);
        } else {
            const float c[6] = {a.x, a.y, a.z, a.w, b.z, b.w};
            cz_spread(c, czv_neg(code), w);
        }
    }
};
template <>
struct TanLoad<double> {
    f64x2 a, b, c, d;   // tet: (g~_i, V), (g~_j, V); CZ: the pair's six values in a, b, c
    __device__ inline void load(const Stage &sv, uint32_t code)
    {
        const uint32_t u = code_unit(code), cz = sv.cz_word + __umul24(u, CZ_TAN_REC) + 6 * czv_pair(code);
        const bool tet = code_kind(code) == KIND_TET;
        const double *p0 = tan_word(sv, tet ? 4 * tet_at(sv, code_q(code) >> 2, u) : cz);
        const double *p1 = tan_word(sv, tet ? 4 * tet_at(sv, code_q(code) & 3, u) : cz + 2);
        a = *(const f64x2 *)p0;
        b = *(const f64x2 *)(p0 + 2);
        c = *(const f64x2 *)p1;
        d = *(const f64x2 *)(p1 + 2);
    }
    __device__ inline void values(double w[9], uint32_t code, double stiff, double mcoef) const
    {
        if (code_kind(code) == KIND_TET) {
            TetIso<double> t;
            t.i0 = make_double2(a.x, a.y);
            t.i1 = make_double2(b.x, b.y);
            t.j0 = make_double2(c.x, c.y);
            t.j1 = make_double2(d.x, d.y);
            t.ij = (int)code_q(code);
            t.values(w, stiff, mcoef);
        } else {
            const double z[6] = {a.x, a.y, b.x, b.y, d.x, d.y};
            cz_spread(z, czv_neg(code), w);
        }
    }
};

// One contribution's 3x3 block where tets have general records or the units are impacts, as the
// values that are added into the slot's FP64 accumulator.
template <bool MIXED, typename L>
__device__ inline void contrib9(const Stage &sv, uint32_t code, L v[9])
{
    using T = typename std::conditional<MIXED, float, double>::type;
    const T stiff = (T)sv.stiff, mcoef = (T)sv.mcoef;
    const uint32_t kind = code_kind(code), u = code_unit(code), q = code_q(code);
    if (kind == KIND_CZ) {
        const T *rec = (const T *)((const double *)sv.tan + sv.cz_word) + (size_t)u * CZ_TAN_REC + 6 * czv_pair(code);
        T c[6];
#pragma unroll
        for (int k = 0; k < 6; k++) c[k] = rec[k];
        cz_spread(c, czv_neg(code), v);
        return;
    }
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (kind == KIND_TET)
        tet_block_gen<T>(acc, (const T *)sv.tan + (size_t)u * TET_GEN_REC, q >> 2, q & 3, stiff, mcoef);
    else
        contact_block<T>(acc, (const T *)sv.ct_tan + (size_t)u * CT_TAN_REC, q >> 2, q & 3);
#pragma unroll
    for (int k = 0; k < 9; k++) v[k] = (L)acc[k];
}

// Phase 2 for BCSR values, one workgroup per KEYS consecutive list positions.  The chunk's
// contributions are contiguous in `codes` and are taken in rounds of flat_cap: every thread
// evaluates contributions (uniform work across lanes) into LDS, then one thread per key adds its
// own of the round from LDS in list order into an FP64 accumulator.  The values and their order
// are those of a sequential loop over the key's list, so the result does not depend on the
// chunking.
//   A block on the diagonal has some 16 to 40 contributions, one off it 4 to 6, and each row of
// about 8 blocks holds one of the former: a wave of one key per lane runs as long as its longest
// and was idle for three quarters of the sums, half of the kernel's VALU instructions.  Keys with
// more than VALS_LONG contributions are therefore listed and summed by teams of nine lanes, one
// component each, which keep their sums across the rounds; the rest by one lane each, in at most
// VALS_LONG steps.
//   With isotropic tets the next round's gathers are in flight while one is summed, so nothing in
// between may wait for loads (the mass factor is selected, not looked up).  Alone, the values of
// 256 batched specimens (mixed) take 420 us, from 524 without teams, prefetch and word addresses
// (1.05 GB written and read at least); those of 779,000 tets (FP64) 144 us, from 189.
//   keys   null: list positions are keys; else keys[position] (accumulate mode)
//   off    first code per list position
//   ACC    add to A (single-kernel calls); otherwise overwrite, zero where nothing contributes
// L is the staging type: float for tet and CZ blocks in mixed mode, double otherwise.
constexpr int VALS_LONG = 8;
template <bool MIXED, bool ISO, bool ACC, typename L, int KEYS, int STAGE>
__device__ __forceinline__ void reduce_vals(int bid_, int nb_, const int *__restrict__ off,
        const uint32_t *__restrict__ codes, const int *__restrict__ keys, int nlist, double *__restrict__ A, Stage sv,
        void *smem)
{
    constexpr int CAP = flat_cap<L, KEYS, STAGE>();
    static_assert(CAP * 9 * sizeof(L) >= KEYS * 9 * sizeof(double), "output staging fits the LDS");
    constexpr int PER = (CAP + KEYS - 1) / KEYS;
    L *lds = (L *)smem;
    const int p0 = xcd_remap(bid_, nb_) * KEYS;
    if (p0 >= nlist) return;
    const int p1 = min(p0 + KEYS, nlist);
    const int cb = off[p0], ce = off[p1];
    // this thread's key and its code range, loaded beside the chunk's codes
    const int p = p0 + threadIdx.x;
    const bool live = p < p1;
    int s = 0, b = 0, e = 0;
    if (live) {
        s = keys ? keys[p] : p;
        b = off[p];
        e = off[p + 1];
    }
    // the long keys, in order
    constexpr int WAVES = KEYS / 64, TEAMS = 7 * WAVES, SLOTS = 2;
    auto *longs = (unsigned short *)((char *)smem + vals_stage<L, KEYS, STAGE>());
    int *wcnt = (int *)((char *)smem + vals_stage<L, KEYS, STAGE>() + 2 * KEYS);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool lng = live && e - b > VALS_LONG;
    const unsigned long long lm = __ballot(lng);
    if (lane == 0) wcnt[wave] = __popcll(lm);
    __syncthreads();
    int at_long = __popcll(lm & ((1ULL << lane) - 1)), nlong = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        if (w < wave) at_long += wcnt[w];
        nlong += wcnt[w];
    }
    if (lng) longs[at_long] = (unsigned short)threadIdx.x;
    const bool mine = live && (!lng || at_long >= TEAMS * SLOTS);   // summed by this thread alone
    double acc[9];
#pragma unroll
    for (int i = 0; i < 9; i++) acc[i] = 0.;
    if (ACC && mine) {   // the block's current values, also loaded before the contributions
        const double *src = A + (size_t)s * 9;
#pragma unroll
        for (int i = 0; i < 9; i++) acc[i] = src[i];
    }
    __syncthreads();
    // consecutive long keys go to one wave's teams, whose ranges then fall in the same rounds
    const int team = lane / 9, comp = lane - 9 * team;
    int tkey[SLOTS], tb[SLOTS], te[SLOTS];
    double tacc[SLOTS];
#pragma unroll
    for (int q = 0; q < SLOTS; q++) {
        const int j = (q * WAVES + wave) * 7 + team;
        const bool on = team < 7 && j < nlong;
        tkey[q] = on ? (int)longs[j] : -1;
        tb[q] = on ? off[p0 + tkey[q]] : 0;
        te[q] = on ? off[p0 + tkey[q] + 1] : 0;
        tacc[q] = 0.;
        if (ACC && on) tacc[q] = A[(size_t)keys[p0 + tkey[q]] * 9 + comp];
    }
    auto sum = [&](int c0, int c1) {      // the contributions of the round, each key's in order
        if (mine) {
            const int hi = min(e, c1) - c0;
            for (int c = max(b, c0) - c0; c < hi; c++) {
#pragma unroll
                for (int k = 0; k < 9; k++) acc[k] += (double)lds[c * 9 + k];
            }
        }
#pragma unroll
        for (int q = 0; q < SLOTS; q++) {
            const int hi = min(te[q], c1) - c0;
#pragma unroll 4
            for (int c = max(tb[q], c0) - c0; c < hi; c++) tacc[q] += (double)lds[c * 9 + comp];
        }
    };
    uint32_t cd[PER];
    auto fetch = [&](int c0) {            // codes of the round at c0 (coalesced)
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int i = c0 + (int)threadIdx.x + r * KEYS;
            cd[r] = i < min(c0 + CAP, ce) ? codes[i] : CODE_NONE;
        }
    };
    if constexpr (ISO) {
        // the next round's gathers are under way while this one is summed, and the codes of the
        // one after that
        using T = typename std::conditional<MIXED, float, double>::type;
        const T stiff = (T)sv.stiff, mcoef = (T)sv.mcoef;
        TanLoad<T> ld[PER];
        uint32_t at[PER];
        auto gather = [&]() {
#pragma unroll
            for (int r = 0; r < PER; r++) {
                at[r] = cd[r];
                if (at[r] != CODE_NONE) ld[r].load(sv, at[r]);
            }
        };
        fetch(cb);
        gather();
        fetch(cb + CAP);
        for (int c0 = cb; c0 < ce; c0 += CAP) {
            if (c0 != cb) __syncthreads();   // the previous round's values have been added
#pragma unroll
            for (int r = 0; r < PER; r++) {
                if (at[r] == CODE_NONE) continue;
                T w[9];
                ld[r].values(w, at[r], stiff, mcoef);
                L *v = lds + ((int)threadIdx.x + r * KEYS) * 9;
#pragma unroll
                for (int k = 0; k < 9; k++) v[k] = (L)w[k];
            }
            __syncthreads();
            gather();
            fetch(c0 + 2 * CAP);
            sum(c0, min(c0 + CAP, ce));
        }
    } else {
        for (int c0 = cb; c0 < ce; c0 += CAP) {
            fetch(c0);
            if (c0 != cb) __syncthreads();   // the previous round's values have been added
#pragma unroll
            for (int r = 0; r < PER; r++) {
                if (cd[r] == CODE_NONE) continue;
                L v[9];
                contrib9<MIXED, L>(sv, cd[r], v);
#pragma unroll
                for (int k = 0; k < 9; k++) lds[((int)threadIdx.x + r * KEYS) * 9 + k] = v[k];
            }
            __syncthreads();
            sum(c0, min(c0 + CAP, ce));
        }
    }
    if (ACC) {
        if (mine) {
            double *dst = A + (size_t)s * 9;
#pragma unroll
            for (int i = 0; i < 9; i++) dst[i] = acc[i];
        }
#pragma unroll
        for (int q = 0; q < SLOTS; q++)
            if (tkey[q] >= 0) A[(size_t)keys[p0 + tkey[q]] * 9 + comp] = tacc[q];
        return;
    }
    // overwrite mode: the chunk's blocks A[p0 .. p1) are contiguous; write them through LDS
    // as consecutive doubles (coalesced) instead of one 72-byte block per thread, as
    // nontemporal stores: A is written once and not read again here, so it need not take L2
    // lines from the staged records the other chunks still gather
    double *out = reinterpret_cast<double *>(lds);
    __syncthreads();
    if (mine) {
#pragma unroll
        for (int k = 0; k < 9; k++) out[threadIdx.x * 9 + k] = acc[k];
    }
#pragma unroll
    for (int q = 0; q < SLOTS; q++)
        if (tkey[q] >= 0) out[tkey[q] * 9 + comp] = tacc[q];
    __syncthreads();
    const int nout = (p1 - p0) * 9;
    double *dst = A + (size_t)p0 * 9;
    for (int i = threadIdx.x; i < nout; i += KEYS) __builtin_nontemporal_store(out[i], &dst[i]);
}

template <bool MIXED, bool ISO, bool ACC, typename L, int KEYS, int STAGE>
__global__ __launch_bounds__(KEYS) void k_reduce_vals(const int *__restrict__ off, const uint32_t *__restrict__ codes,
                                                      const int *__restrict__ keys, int nlist, double *__restrict__ A,
                                                      Stage sv)
{
    __shared__ __align__(16) char lds[vals_lds<L, KEYS, STAGE>()];
    reduce_vals<MIXED, ISO, ACC, L, KEYS, STAGE>(blockIdx.x, gridDim.x, off, codes, keys, nlist, A, sv, lds);
}

// Phase 2 for rhs rows (b[row*3+k]) or node forces (dn[node + ns*(F+k)]): one thread per list
// position (off: first code per position).
// TSUM (node forces of the fused call): the sum of the key's contributions from zero is also
// written to tsum[3 key .. 3 key + 2], from which k_reduce_rhs_tsum starts the rhs rows.
template <bool ACC, bool TSUM>
__device__ __forceinline__ void reduce_vec3(int bid_, int nb_, const int *__restrict__ off,
        const uint32_t *__restrict__ codes, const int *__restrict__ keys, int nkeys, double *__restrict__ out,
        int comp_stride, int elem_stride, Stage sv, double *__restrict__ tsum)
{
    const int t = xcd_remap(bid_, nb_) * blockDim.x + threadIdx.x;
    if (t >= nkeys) return;
    const int s = keys ? keys[t] : t;
    const int b = off[t], e = off[t + 1];
    double *dst = out + (size_t)s * elem_stride;
    double a0, a1, a2, t0 = 0., t1 = 0., t2 = 0.;
    if (ACC) {
        if (b == e) return;
        a0 = dst[0]; a1 = dst[comp_stride]; a2 = dst[2 * comp_stride];
    } else {
        a0 = a1 = a2 = 0.;
    }
    auto add = [&](const Part &v) {
        a0 += v.x; a1 += v.y; a2 += v.z;
        if (TSUM) { t0 += v.x; t1 += v.y; t2 += v.z; }
    };
    int c = b;
    for (; c + 4 <= e; c += 4) {          // loads of four contributions in flight, added in order
        const Part p0 = part_of(sv, codes[c]), p1 = part_of(sv, codes[c + 1]);
        const Part p2 = part_of(sv, codes[c + 2]), p3 = part_of(sv, codes[c + 3]);
        add(p0);
        add(p1);
        add(p2);
        add(p3);
    }
    for (; c < e; c++) add(part_of(sv, codes[c]));
    dst[0] = a0; dst[comp_stride] = a1; dst[2 * comp_stride] = a2;
    if (TSUM) {
        double *o = tsum + (size_t)s * 3;
        o[0] = t0; o[1] = t1; o[2] = t2;
    }
}

// Node forces and rhs rows of the fused call in one pass, one thread per node key: F[node] gets
// the node's tet contributions added in list order (as reduce_vec3<true, TSUM>), and the node's
// rhs row -- node_row[node], when not negative -- is the sum of the same contributions from zero
// followed by the row's CZ contributions in list order (as reduce_rhs_tsum from that tet sum).
// Used when every rhs row's tet contributions are its node's force list and every row has such
// a node (the host checks both once per pair of maps).
// The contributions of the workgroup's nodes are one run of codes; they come through LDS in rounds
// of BYTES / 24, like those of reduce_vals: codes read as they lie, three or more gathers in
// flight per lane, neighbouring lanes in neighbouring tets.  A lane walking its own node's list
// fetched every line for 24 of its bytes: alone on 256 batched specimens 242 us and 67 for the rows,
// 205 for both this way.
template <int KEYS, int BYTES>
__device__ __forceinline__ void reduce_force_rhs(int bid_, int nb_, const int *__restrict__ foff,
        const uint32_t *__restrict__ fcodes, const int *__restrict__ fkeys, int nfkeys, double *__restrict__ F,
        int ns, const int *__restrict__ node_row, const int *__restrict__ roff, const uint32_t *__restrict__ rcodes,
        const int *__restrict__ cz_begin, double *__restrict__ rhs, Stage sv, void *smem)
{
    constexpr int PER = BYTES / 24 / KEYS < 12 ? BYTES / 24 / KEYS : 12, CAP = PER * KEYS;
    static_assert(PER >= 1, "a contribution per lane");
    double *lds = (double *)smem;
    const int p0 = xcd_remap(bid_, nb_) * KEYS;
    if (p0 >= nfkeys) return;
    const int p1 = min(p0 + KEYS, nfkeys), cb = foff[p0], ce = foff[p1];
    const int t = p0 + (int)threadIdx.x;
    const bool live = t < p1;
    int s = 0, b = 0, e = 0, r = -1;
    double a0 = 0., a1 = 0., a2 = 0., t0 = 0., t1 = 0., t2 = 0.;
    double *dst = F;
    if (live) {
        s = fkeys ? fkeys[t] : t;
        b = foff[t];
        e = foff[t + 1];
        r = node_row[s];
        dst = F + s;
        a0 = dst[0]; a1 = dst[ns]; a2 = dst[2 * (size_t)ns];
    }
    for (int c0 = cb; c0 < ce; c0 += CAP) {
        const int c1 = min(c0 + CAP, ce);
        Part v[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = c0 + (int)threadIdx.x + k * KEYS;
            if (i < c1) v[k] = part_of(sv, fcodes[i]);
        }
        if (c0 != cb) __syncthreads();   // the previous round's parts have been added
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = (int)threadIdx.x + k * KEYS;
            if (c0 + i < c1) {
                lds[3 * i] = v[k].x;
                lds[3 * i + 1] = v[k].y;
                lds[3 * i + 2] = v[k].z;
            }
        }
        __syncthreads();
        const int hi = min(e, c1) - c0;
#pragma unroll 4
        for (int c = max(b, c0) - c0; c < hi; c++) {
            const double x = lds[3 * c], y = lds[3 * c + 1], z = lds[3 * c + 2];
            a0 += x; a1 += y; a2 += z;
            t0 += x; t1 += y; t2 += z;
        }
    }
    if (!live) return;
    dst[0] = a0; dst[ns] = a1; dst[2 * (size_t)ns] = a2;
    if (r < 0) return;
    // six contributions of CZs in flight, as many as a row mostly has
    constexpr int CZS = 6;
    const int re = roff[r + 1];
    for (int k = cz_begin[r]; k < re; k += CZS) {
        uint32_t cd[CZS];
        Part q[CZS];
#pragma unroll
        for (int i = 0; i < CZS; i++) cd[i] = rcodes[min(k + i, re - 1)];
#pragma unroll
        for (int i = 0; i < CZS; i++) q[i] = part_of(sv, cd[i]);
#pragma unroll
        for (int i = 0; i < CZS; i++)
            if (k + i < re) {
                t0 += q[i].x; t1 += q[i].y; t2 += q[i].z;
            }
    }
    double *o = rhs + (size_t)r * 3;
    o[0] = t0; o[1] = t1; o[2] = t2;
}

template <bool ACC, bool TSUM = false>
__global__ __launch_bounds__(256) void k_reduce_vec3(const int *__restrict__ off, const uint32_t *__restrict__ codes,
                                                     const int *__restrict__ keys, int nkeys, double *__restrict__ out,
                                                     int comp_stride, int elem_stride, Stage sv,
                                                     double *__restrict__ tsum = nullptr)
{
    reduce_vec3<ACC, TSUM>(blockIdx.x, gridDim.x, off, codes, keys, nkeys, out, comp_stride, elem_stride, sv, tsum);
}

// For each rhs row r of the fused call: the length of its leading run of tet codes and the
// node those tets share; node_row (-1 before) gets the row of each such node.  The row's tet
// contributions must be exactly the force key's list of that node (same codes, same order), else
// LINK_ERR is set; a row without a tet node, or a node with two rows, sets LINK_ERR + 1.
__global__ __launch_bounds__(256) void k_rhs_check(const int *__restrict__ roff, const uint32_t *__restrict__ rcodes,
                                                   int N, const int *__restrict__ foff,
                                                   const uint32_t *__restrict__ fcodes, int nfkeys, MapSrc tet,
                                                   int *__restrict__ row_node, int *__restrict__ cz_begin,
                                                   int *__restrict__ node_row, Report rep)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= N) return;
    const int b = roff[r], e = roff[r + 1];
    int L = 0;
    while (b + L < e && code_kind(rcodes[b + L]) == KIND_TET) L++;
    cz_begin[r] = b + L;
    if (L == 0) {
        row_node[r] = -1;
        rep.set(LINK_ERR + 1);
        return;
    }
    const uint32_t c0 = rcodes[b];
    const int u = (int)code_unit(c0), q = (int)code_q(c0);
    const int n = (u < tet.n && q < 4) ? tet.base[u + (size_t)tet.stride * (tet.field0 + q)] : -1;
    bool ok = n >= 0 && n < nfkeys && foff[n + 1] - foff[n] == L;
    const int fb = ok ? foff[n] : 0;
    for (int k = 0; ok && k < L; k++) ok = fcodes[fb + k] == rcodes[b + k];
    if (!ok) {
        rep.set(LINK_ERR);
        return;
    }
    row_node[r] = n;
    if (atomicExch(node_row + n, r) != -1) rep.set(LINK_ERR + 1);
}

// rhs rows of the fused call: the node's tet sum (k_reduce_vec3 TSUM), then the row's CZ
// contributions in order -- the sequential sum over the row's list.
__device__ __forceinline__ void reduce_rhs_tsum(int bid_, int nb_, const int *__restrict__ off,
        const uint32_t *__restrict__ codes, const int *__restrict__ cz_begin, const int *__restrict__ row_node,
        const double *__restrict__ tsum, int N, double *__restrict__ out, Stage sv)
{
    const int r = xcd_remap(bid_, nb_) * blockDim.x + threadIdx.x;
    if (r >= N) return;
    const int n = row_node[r];
    double a0 = 0., a1 = 0., a2 = 0.;
    if (n >= 0) {
        a0 = tsum[(size_t)n * 3];
        a1 = tsum[(size_t)n * 3 + 1];
        a2 = tsum[(size_t)n * 3 + 2];
    }
    const int e = off[r + 1];
    for (int c = cz_begin[r]; c < e; c++) {
        const Part p = part_of(sv, codes[c]);
        a0 += p.x; a1 += p.y; a2 += p.z;
    }
    double *o = out + (size_t)r * 3;
    o[0] = a0; o[1] = a1; o[2] = a2;
}

__global__ __launch_bounds__(256) void k_reduce_rhs_tsum(const int *__restrict__ off, const uint32_t *__restrict__ codes,
                                                         const int *__restrict__ cz_begin, const int *__restrict__ row_node,
                                                         const double *__restrict__ tsum, int N, double *__restrict__ out,
                                                         Stage sv)
{
    reduce_rhs_tsum(blockIdx.x, gridDim.x, off, codes, cz_begin, row_node, tsum, N, out, sv);
}

// Byte copy, 16 bytes per thread where both ends allow it (icf_d2d; a kernel so that it can
// be recorded in a captured graph).
__global__ __launch_bounds__(256) void k_copy(char *__restrict__ dst, const char *__restrict__ src, size_t bytes)
{
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 16;
    if (i >= bytes) return;
    if (i + 16 <= bytes && (((uintptr_t)(dst + i) | (uintptr_t)(src + i)) & 15) == 0) {
        *(uint4 *)(dst + i) = *(const uint4 *)(src + i);
    } else {
        const size_t e = i + 16 < bytes ? i + 16 : bytes;
        for (size_t k = i; k < e; k++) dst[k] = src[k];
    }
}

// VALU issue-rate probe (icf_probe_valu): every thread runs `iters` rounds of 16 independent
// fused multiply-add chains x = x * m + c (one VALU instruction each, no memory traffic in the
// loop) and stores the sum of its chains, so that no chain can be dropped.  With enough waves
// per SIMD the loop is bound by VALU issue alone: its rate is the achievable FMA peak.
template <typename T>
__global__ __launch_bounds__(256) void k_valu_probe(T *__restrict__ out, int iters, T m, T c)
{
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    T x[16];
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = (T)(tid & 7) * (T)0.125 + (T)k;
    for (int i = 0; i < iters; i++) {
#pragma unroll
        for (int k = 0; k < 16; k++) x[k] = fma(x[k], m, c);
    }
    T s = 0;
#pragma unroll
    for (int k = 0; k < 16; k++) s += x[k];
    out[tid] = s;
}

__global__ void k_fill_int(int *__restrict__ p, int n, int v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Block-wide integer sum (256 threads), result valid in thread 0.
__device__ inline int block_sum256(int x)
{
    __shared__ int part[4];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = x;
    __syncthreads();
    int r = 0;
    if (threadIdx.x == 0) r = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    return r;
}

// Integer sum (GPU_Functionality.Sum, :93-107): grid-stride, one atomic per block.
__global__ __launch_bounds__(256) void k_sum_int(const int *__restrict__ v, int n, int *__restrict__ out)
{
    int x = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) x += v[i];
    x = block_sum256(x);
    if (threadIdx.x == 0 && x != 0) atomicAdd(out, x);
}

// The damaged and failed counts of one CZ pass in one sweep (out[0], out[1]).
__device__ __forceinline__ void count_flags(int bid_, int nb_, const int *__restrict__ damaged,
        const int *__restrict__ failed, int n, int *__restrict__ out)
{
    int d = 0, f = 0;
    for (int i = bid_ * blockDim.x + threadIdx.x; i < n; i += nb_ * blockDim.x) {
        d += damaged[i];
        f += failed[i];
    }
    d = block_sum256(d);
    f = block_sum256(f);
    if (threadIdx.x == 0) {
        if (d) atomicAdd(out, d);
        if (f) atomicAdd(out + 1, f);
    }
}

// One thread of each of nb workgroups adds its counts; the last of them reports the totals when asked to
// (rep.host; out[3] is zero before), so that the host has them after the wait of its call: a copy
// and a second wait took 15 us of a call of 50.  A thread's tickets follow its sums because it waits for them.
__device__ inline void add_counts(int *out, int d, int f, int nb, const Report &rep)
{
    if (!rep.host) {
        if (d) atomicAdd(out, d);
        if (f) atomicAdd(out + 1, f);
        return;
    }
    const int d0 = atomicAdd(out, d), f0 = atomicAdd(out + 1, f);
    int one = 1;
    asm volatile("" : "+v"(one) : "v"(d0), "v"(f0));
    if (atomicAdd(out + 3, one) != nb - 1) return;
    rep.put(CZ_DAMAGED, (unsigned)__hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    rep.put(CZ_FAILED, (unsigned)__hip_atomic_load(out + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// count_flags for workgroups of NT threads (a multiple of 64, at most 1024).
template <int NT>
__device__ __forceinline__ void count_flags_n(int bid_, int nb_, const int *__restrict__ damaged,
        const int *__restrict__ failed, int n, int *__restrict__ out, const Report &rep)
{
    __shared__ int part[2][NT / 64];
    int d = 0, f = 0;
    for (int i = bid_ * NT + threadIdx.x; i < n; i += nb_ * NT) {
        d += damaged[i];
        f += failed[i];
    }
    for (int o = 32; o > 0; o >>= 1) {
        d += __shfl_xor(d, o);
        f += __shfl_xor(f, o);
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = d;
        part[1][threadIdx.x >> 6] = f;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        d = f = 0;
        for (int w = 0; w < NT / 64; w++) {
            d += part[0][w];
            f += part[1][w];
        }
        add_counts(out, d, f, nb_, rep);
    }
}

// Per-specimen counters: workgroup bid_ takes specimens bid_, bid_ + nb_, ...; each
// specimen's damaged and failed counts are written (no atomics) and added into the totals.
template <int NT>
__device__ __forceinline__ void count_flags_spec(int bid_, int nb_, const int *__restrict__ damaged,
        const int *__restrict__ failed, const int *__restrict__ cz_off, int nspec, int *__restrict__ spec,
        int *__restrict__ out, const Report &rep)
{
    __shared__ int part[2][NT / 64];
    int td = 0, tf = 0;
    for (int s = bid_; s < nspec; s += nb_) {
        int d = 0, f = 0;
        for (int i = cz_off[s] + (int)threadIdx.x; i < cz_off[s + 1]; i += NT) {
            d += damaged[i];
            f += failed[i];
        }
        for (int o = 32; o > 0; o >>= 1) {
            d += __shfl_xor(d, o);
            f += __shfl_xor(f, o);
        }
        if ((threadIdx.x & 63) == 0) {
            part[0][threadIdx.x >> 6] = d;
            part[1][threadIdx.x >> 6] = f;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            d = f = 0;
            for (int w = 0; w < NT / 64; w++) {
                d += part[0][w];
                f += part[1][w];
            }
            spec[2 * s] = d;
            spec[2 * s + 1] = f;
            if (rep.host && nspec <= REPORT_SPECS) {
                rep.put(REPORT_WORDS + 2 * s, (unsigned)d);
                rep.put(REPORT_WORDS + 2 * s + 1, (unsigned)f);
            }
            td += d;
            tf += f;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) add_counts(out, td, tf, nb_, rep);
}

__global__ __launch_bounds__(256) void k_count_flags(const int *__restrict__ damaged, const int *__restrict__ failed,
                                                     int n, int *__restrict__ out)
{
    count_flags(blockIdx.x, gridDim.x, damaged, failed, n, out);
}

}  // namespace icf
