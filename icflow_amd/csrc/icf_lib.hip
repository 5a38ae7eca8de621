// icf_lib.hip -- libicflow_hip.so: the C ABI declared in include/icflow_hip.h.
//
// Single translation unit: the kernels of icf_*.inc.h share one __constant__ DevConsts.
// Device memory for staging records and slot maps is owned by the context and grows on
// demand; the caller's buffers (nodes, pcsr arrays, BCSR, rhs) are never retained.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>
#include <string.h>
#include <math.h>
#include <climits>
#include <string>
#include <vector>
#include <list>
#include <type_traits>
#include <atomic>
#include <algorithm>
#include <mutex>

#include "../../include/icflow_hip.h"

#include "icf_device.h"
namespace icf {
__constant__ DevConsts g_c;
}
#include "icf_elem.inc.h"
#include "icf_cz.inc.h"
#include "icf_cz_phase1.inc.h"
#include "icf_contact.inc.h"
#include "icf_contact_resp.inc.h"
#include "icf_reduce.inc.h"
#include "icf_fused.inc.h"
#include "icf_batch.inc.h"
#include "icf_nodes.inc.h"
#include "icf_pattern.inc.h"
#include "icf_broad.inc.h"

using namespace icf;

namespace {

// Device bytes a call reads or writes: up to MAXS spans, or `all` (conflicts with everything).
struct Span {
    uintptr_t lo, hi;
    bool w;
};
struct Access {
    static constexpr int MAXS = 12;
    Span s[MAXS];
    int n = 0;
    bool all = false;
    Access &add(const void *p, size_t bytes, bool w)
    {
        if (!p || !bytes) return *this;
        if (n == MAXS) {
            all = true;
            return *this;
        }
        s[n++] = {(uintptr_t)p, (uintptr_t)p + bytes, w};
        return *this;
    }
    template <typename T> Access &rd(const T *p, size_t count) { return add(p, count * sizeof(T), false); }
    template <typename T> Access &wr(const T *p, size_t count) { return add(p, count * sizeof(T), true); }
    // the whole allocation holding p, for buffers whose used extent the call does not know
    Access &alloc(const void *p, bool w)
    {
        if (!p) return *this;
        void *base = nullptr;
        size_t sz = 0;
        if (hipMemGetAddressRange(&base, &sz, const_cast<void *>(p)) == hipSuccess && sz) return add(base, sz, w);
        (void)hipGetLastError();
        all = true;
        return *this;
    }
    static Access everything()
    {
        Access a;
        a.all = true;
        return a;
    }
};

bool conflict(const Access &a, const Access &b)
{
    if (a.all || b.all) return true;
    for (int i = 0; i < a.n; i++)
        for (int j = 0; j < b.n; j++)
            if ((a.s[i].w || b.s[j].w) && a.s[i].lo < b.s[j].hi && b.s[j].lo < a.s[i].hi) return true;
    return false;
}

// A call issued on one lane, with the event recorded after its last launch.
struct LaneRec {
    Access a;
    hipEvent_t ev;
};
constexpr int LANE_EVENTS = 32, LANE_LOG = 24;   // a logged event is one of the lane's last LANE_LOG

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
};

enum Target { TGT_VALS = 0, TGT_RHS = 1, TGT_FORCE = 2 };

struct SrcKey {
    uint32_t kind;
    const int *base;
    int n, stride, field0, nq;
    bool operator==(const SrcKey &o) const
    {
        return kind == o.kind && base == o.base && n == o.n && stride == o.stride && field0 == o.field0 && nq == o.nq;
    }
};

struct SlotMap {
    int target = 0;
    int fixed_nkeys = -1;          // -1: as many keys as the fields turn out to need
    std::vector<SrcKey> srcs;
    int nkeys = 0;                 // keys counted; without fixed_nkeys at least the largest key + 1
    // grow-only buffers, kept when the map is built anew
    DevBuf b_off, b_codes, b_keys, b_loff, b_snap;
    DevBuf b_off2;                 // offsets of slots that moved; changes places with b_off
    int *off = nullptr;            // nkeys + 1
    uint32_t *codes = nullptr;
    int *keys = nullptr;           // accumulate mode: the keys with contributions (null: all keys)
    int *loff = nullptr;           // first code per list position (off when all keys are listed)
    int nlaunch = 0;               // keys a reduction visits
    int id = 0;                    // unique per map built
    // rhs maps of the fused call: the force map (by id) whose per-node tet sums seed the rows,
    // the outcome of that check, and per row the node and the first non-tet code
    int tsum_with = -1;
    bool tsum_ok = false;
    DevBuf b_row_node, b_cz_begin, b_node_row;
    int *row_node = nullptr, *cz_begin = nullptr;
    // ... and per node of the force map its rhs row (-1: none), when every row has one tet node
    // (then the node-force pass also writes the rhs rows)
    int *node_row = nullptr;
    bool merge_ok = false;
    // copies of the key fields the map was built from, per source; after a write that may have
    // touched the fields (suspect) the map is kept if they still compare equal
    std::vector<int *> snap;
    bool suspect = false;
    bool changed = false;          // suspect, and the fields are known to be others
    bool built = false;
};

std::atomic<int> g_next_ctx_id{1};
// All contexts on a device share the one __constant__ g_c.  g_const_owner[d] is the id of the
// context whose constants it holds; g_dev_mu[d] is held by every call that launches kernels
// reading g_c, from the check of the owner to its last launch, so that another context
// cannot replace the constants in between (ConstUse).
int g_const_owner[64];
std::mutex g_dev_mu[64];

// Scratch of the allocation-free entry point (icf_find_closest_face_noalloc): one array per
// GPU, reserved when the code object loads on that GPU and held until the process ends.
// Host code never passes `scratch` itself to a kernel or a copy (on the host the name is a
// stand-in, not a device address): it uses the address that hipGetSymbolAddress returned for
// the device, looked up once per device by icf_create and kept in g_scratch_ptr.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
std::mutex g_scratch_mu;
void *g_scratch_ptr[64];           // per device: device address of `scratch`, null until looked up

// With `device` current: the device address of its scratch array (looked up on first use).
hipError_t scratch_for_device(int device, void **out)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return hipSuccess;
}

}  // namespace

// Launch-shape roles besides the value reductions (icf_set_shape / icf_get_shape): the
// workgroup size (64, 128 or 256 lanes) of phase 1 of the fused call, of the narrow phase and
// of the impacts' phase 1, the lanes per (node, tet) tuple of the closest face (4, 8 or 16),
// and the order of the fused value launch's two phases (0: node forces first, then the BCSR
// values; 1: interleaved in rounds of eight workgroups).  Every candidate gives the same
// results (each unit's and key's work does not depend on the shape).
constexpr int NSHAPE = 5, NSHAPE_CAND = 3;
constexpr int shape_value(int role, int c)
{
    return role == ICF_SHAPE_CLOSEST ? 4 << c : role == ICF_SHAPE_ORDER ? c : 64 << c;
}
constexpr int shape_ncand(int role) { return role == ICF_SHAPE_ORDER ? 2 : 3; }
constexpr int SHAPE_DEFAULT[NSHAPE] = {2, 2, 1, 2, 1};   // 256, 256, 8 lanes, 256, interleaved
// What untuned launches use: the same, but node forces first.  Interleaved with the values they
// gained 40 us on 256 specimens while both waited on memory; since they do not, the order costs 6 us
// of 34 on 146,000 tets and gives 4 of 584 on 256 specimens.
constexpr int SHAPE_UNTUNED[NSHAPE] = {2, 2, 1, 2, 0};
// ... and for launches of at most so many units, whose workgroups would leave compute units empty
// while each runs through a long chain: phase 1 with 64 lanes (14.3 -> 11.9 us on 3,072 tets, 20.7 ->
// 18.9 on 48,000, 42.9 -> 41.9 on 309,000; 113.7 -> 117.7 on 779,000), 64 impacts (21.9 -> 17.8 us for
// 547, 27.0 -> 18.2 for 7,000, 25.2 -> 22.1 for 20,900; 25.3 -> 28.3 for 61,600).
constexpr int SHAPE_SMALL[NSHAPE] = {0, 2, 1, 0, 0};
constexpr long long SHAPE_SMALL_MAX[NSHAPE] = {1 << 19, 0, 0, 1 << 15, 0};
// For the same reason the closest face's candidate of 8 lanes takes 16 for at most so many tuples (9.5 ->
// 8.3 us for 547, 11.2 -> 9.9 for 7,000; 14.8 -> 14.4 for 20,900, 27.6 -> 28.4 for 61,600), tuned, set or
// neither: a candidate's launch, so that 8, which untuned contexts report, stays what they use.
constexpr int CLOSEST_SMALL = 1 << 14;

struct icf_ctx {
    int id = 0;
    int device = 0;
    int ncu = 256;                 // compute units of the device
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipStream_t cur = nullptr;       // where LAUNCH issues: `stream`, or `stream_c` (lanes)
    // lanes across calls: lane 0 is `stream`, lane 1 is `stream_c` (contact detection); each
    // lane's log holds its calls that the other lane has not yet waited for
    hipStream_t stream_c = nullptr;
    hipEvent_t lane_ev[2][LANE_EVENTS] = {};
    unsigned lane_ev_next[2] = {0, 0};
    std::vector<LaneRec> lane_log[2];
    bool lane0_unlogged = false;   // lane-0 work issued since the last lane-0 log entry
    bool has_consts = false;
    bool consts_dirty = false;     // icf_set_constants changed hc since this context's last upload
    // bumped whenever memory the context owns is freed or moved, or a slot map or the
    // adjacency lists may no longer match what they were built from: a graph captured at an
    // older epoch may point at stale memory and is refused by icf_graph_launch
    unsigned long long epoch = 1;
    // bumped with it, except where the fields in question were found unchanged: the batched
    // call's layout check holds as long as this stays (no graph is involved in it)
    unsigned long long fields_epoch = 1;
    // what kernels report to the host (Report): pinned words, their device copy, the last call's
    // sequence number
    unsigned *rep_host = nullptr, *rep_dev = nullptr, rep_seq = 0;
    int precision = ICF_FP64;
    DevConsts hc;
    DevBuf tet_rhs, tan, cz_rhs, ct, scan_tmp;
    uint32_t cz_word = 0;            // first 8-byte word of the CZs' records in `tan`
    DevBuf pat_a, pat_b;           // pattern build / broad phase / NL2set: 64-bit keys
    DevBuf pat_cnt;                // pattern build: the impacts' pairs per row (zero in between)
    // the pattern's static part (elements and CZs): its rows, kept with a copy of the node-id fields
    // and altIds they came from; reused while that copy still matches
    struct PatCache {
        bool valid = false;
        int nNodes = 0, nElems = 0, el_stride = 0, nCZs = 0, cz_stride = 0, N = 0;
        DevBuf snap, rows, cols;
    } patc;
    DevBuf bp_f, bp_i, bp_l;         // broad phase and NL2set scratch (doubles, ints, int64)
    DevBuf bp_c;                     // broad phase grid (cell counts, first sorted position per cell key)
    DevBuf bp_g;                     // broad phase pair grouping (counts and starts per tet, ranks)
    long long nl2_last = 0;          // distinct tuples of the last NL2set call
    long long bp_cells = 0, bp_inner = 0;   // cells of the last search's grid, with and without margin
    long long bp_cap = 0;            // pair keys the broad phase's buffer holds (grows with use)
    DevBuf map_cnt, map_rank, map_sums;   // building slot maps: counts (zero in between), ranks, tile sums
    DevBuf tsum;                     // per-node tet sums of the fused call
    DevBuf ct_f;                     // impact forces (the tangent blocks are in ct)
    int tplane = 64;                 // plane stride of the staged tet records (tet_plane)
    // compact adjacent-face lists of the surface tets (k_adj_*), built from `ie` on first use and
    // dropped when a library write or free touches that allocation (or icf_pattern_changed)
    struct Adj {
        const int *ie = nullptr;
        int es = 0;
        uintptr_t lo = 0, hi = 0;    // the allocation holding ie
        DevBuf off, ids;
        bool valid = false;
    } adj;
    int *small = nullptr;          // 16 ints of scratch (error flag, sums; 8-11: largest keys)
    unsigned char *noalloc = nullptr;   // this device's `scratch` array (device address)
    std::list<SlotMap> maps;       // std::list: pointers handed out by get_maps stay valid
    int next_map_id = 0;
    std::string err;
    double last_ms = -1;
    bool blocking = true;          // icf_set_blocking
    bool capturing = false;        // between icf_graph_begin and icf_graph_end
    bool overlap = true;           // icf_set_overlap: independent kernels on more than one stream
    // autotuned launch shapes.  tune: the chunk shape (workgroup size, staging) of the BCSR-value
    // reductions, per role [accumulate map][FP64 staging]; shape: the workgroup size of phase 1,
    // the narrow phase and the impacts' phase 1, and the lanes per tuple of the closest face.
    // Per role: the candidate in use and, while tuning, the timings
    struct Tune {
        int ncand = NCAND;
        int sel = CAND_FP32;       // candidate in use
        bool tuned = false;        // a tuning has chosen it
        int untuned = CAND_UNTUNED;    // what launches use when it is neither tuned nor set
        int small = CAND_SMALL;        // ... where they have at most small_max units
        long long small_max = 0;
        bool active = false;       // timing the candidates in turn
        bool fixed = false;        // chosen by the caller (icf_set_chunk_keys / icf_set_shape)
        int turn = 0;              // launches started while tuning
        int samples = 0;           // launches timed
        int cand = -1;             // candidate of the launch being timed, -1: none
        int last = -1;             // candidate of the role's last launch
        // the shape that the role's launches use, as far as the caller can be told: a launch that is
        // neither tuned nor set goes by its size
        int in_use() const { return active || fixed || tuned || last < 0 ? sel : last; }
        int bucket = -1;           // size class of the launches timed (the shape cache's key)
        float best[NCAND] = {};    // fastest launch per candidate (ms), 0: not timed
        hipEvent_t ev[2] = {nullptr, nullptr};
    } tune[2][2], shape[NSHAPE];
    int tune_rounds = 0;           // timed launches per candidate (icf_set_autotune)
    // icf_assemble_batched: the last offsets (host copy; device copy followed by 2 counts per
    // specimen) and the value and rhs maps whose units were last checked against them
    struct Batch {
        std::vector<int> off;      // 4 (n + 1): tets, CZs, rows, blocks
        int n = 0;
        DevBuf d;
        // the units and epoch whose block-diagonal layout was last checked against `off`
        std::vector<long long> checked;
        // set by icf_assemble_batched for its assembly: the fused value launch then also writes
        // the per-specimen CZ counts (spec_counted reports that it did)
        const int *cz_off = nullptr;
        int *spec_counts = nullptr;
        bool spec_counted = false;
    } batch;
    // per-kernel profiling (icf_set_profiling)
    bool profiling = false;
    struct Pending {
        const char *name;
        hipEvent_t a, b;
    };
    std::vector<Pending> pending;
    std::vector<hipEvent_t> ev_pool;
    std::vector<std::string> prof_names;
    std::vector<double> prof_ms;
    std::vector<long long> prof_n;
};

namespace {

int fail(icf_ctx *ctx, int code, const std::string &msg)
{
    if (ctx) ctx->err = msg;
    return code;
}

#define HIPCHK(ctx, x)                                                                             \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess)                                                                      \
            return fail((ctx), (int)e_, std::string(#x) + ": " + hipGetErrorString(e_));           \
    } while (0)

void bump(icf_ctx *ctx)
{
    ctx->epoch++;
    ctx->fields_epoch++;
}

// A new report for the launches of one call; its words read as not set until a kernel sets them.
Report new_report(icf_ctx *ctx) { return Report{ctx->rep_dev, ctx->rep_host, ++ctx->rep_seq}; }
// After the stream has been waited for.
bool reported(const Report &r, int k) { return ((volatile unsigned *)r.host)[k] == r.seq; }

int grow(icf_ctx *ctx, DevBuf &b, size_t bytes)
{
    if (b.bytes >= bytes) return 0;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "an internal buffer must grow: run the call once uncaptured");
    if (b.p) {
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream_c));
        HIPCHK(ctx, hipFree(b.p));
        b.p = nullptr;
        b.bytes = 0;
    }
    size_t want = bytes + bytes / 4 + 256;
    bump(ctx);
    HIPCHK(ctx, hipMalloc(&b.p, want));
    b.bytes = want;
    return 0;
}

void free_map(SlotMap &m)
{
    for (DevBuf *b : {&m.b_off, &m.b_off2, &m.b_codes, &m.b_keys, &m.b_loff, &m.b_snap, &m.b_row_node, &m.b_cz_begin, &m.b_node_row}) {
        if (b->p) (void)hipFree(b->p);
        *b = DevBuf();
    }
}

// Maps whose key fields overlap [lo, hi): dropped when the memory goes away (erase), else
// marked suspect, to be compared against their snapshot before the next use (or not, where the
// fields are known to have changed).
bool map_keys_overlap(const SlotMap &m, uintptr_t lo, uintptr_t hi)
{
    if (!m.built) return false;
    for (const SrcKey &s : m.srcs) {
        uintptr_t a = (uintptr_t)(s.base + (size_t)s.stride * s.field0);
        uintptr_t b = (uintptr_t)(s.base + (size_t)s.stride * (s.field0 + s.nq));
        if (a < hi && lo < b) return true;
    }
    return false;
}

void invalidate_range(icf_ctx *ctx, uintptr_t lo, uintptr_t hi, bool erase = false)
{
    if (ctx->adj.valid && ctx->adj.lo < hi && lo < ctx->adj.hi) {
        ctx->adj.valid = false;
        bump(ctx);
    }
    for (auto it = ctx->maps.begin(); it != ctx->maps.end();) {
        const bool hit = map_keys_overlap(*it, lo, hi);
        if (hit) bump(ctx);
        if (hit && erase) {
            (void)hipStreamSynchronize(ctx->stream);
            free_map(*it);
            it = ctx->maps.erase(it);
        } else {
            if (hit) it->suspect = true;
            ++it;
        }
    }
}

// The built map that has one of its sources over these fields of a unit array; a map not in doubt
// rather than one that is.
SlotMap *map_over(icf_ctx *ctx, const int *base, int n, int stride, int field0, int nq, const int **snap)
{
    SlotMap *found = nullptr;
    for (SlotMap &m : ctx->maps) {
        if (!m.built || (found && (!found->suspect || m.suspect))) continue;
        for (size_t i = 0; i < m.srcs.size(); i++) {
            const SrcKey &s = m.srcs[i];
            if (s.base != base || s.n != n || s.stride != stride || s.field0 != field0 || s.nq != nq) continue;
            found = &m;
            *snap = m.snap[i];
        }
    }
    return found;
}

// Fields in [lo, hi) were packed.  `held`, the map whose copy they were compared with, stays as it
// is if they are still its own (same); every other map over them is compared with its copy before its
// next use.  Graphs captured before are refused either way, as after any write to such fields.
void packed_range(icf_ctx *ctx, uintptr_t lo, uintptr_t hi, const SlotMap *held, bool same, bool changed)
{
    if (ctx->adj.valid && ctx->adj.lo < hi && lo < ctx->adj.hi) {
        ctx->adj.valid = false;
        bump(ctx);
    }
    for (SlotMap &m : ctx->maps) {
        if (!map_keys_overlap(m, lo, hi)) continue;
        if (&m == held && same && !m.suspect) {
            ctx->epoch++;
            continue;
        }
        bump(ctx);
        m.suspect = true;
        if (&m == held && changed) m.changed = true;
    }
}

// A write by the library into caller memory [p, p + bytes) (copies, kernels that write int
// fields in place).  Outside capture: slot maps and adjacency lists built from those bytes
// are checked again before their next use.  During capture such a write is refused: every
// replay would change what the maps were built from behind their back.
int note_write(icf_ctx *ctx, const void *p, size_t bytes, const char *what)
{
    const uintptr_t lo = (uintptr_t)p, hi = lo + bytes;
    if (!bytes) return 0;
    if (!ctx->capturing) {
        invalidate_range(ctx, lo, hi);
        return 0;
    }
    bool hit = ctx->adj.valid && ctx->adj.lo < hi && lo < ctx->adj.hi;
    for (const SlotMap &m : ctx->maps) hit = hit || map_keys_overlap(m, lo, hi);
    if (hit)
        return fail(ctx, ICF_E_CAPTURE, std::string(what) +
                                            " would write fields that a slot map or the adjacency lists were built "
                                            "from: it cannot be captured");
    return 0;
}

// The context's constants in g_c for the lifetime of this object: takes the device's lock,
// and when another context's constants are loaded, waits for all work on the device (its
// queued kernels read them) before loading ours.  During capture nothing is loaded: a replay
// loads them in icf_graph_launch.
struct ConstUse {
    std::unique_lock<std::mutex> lk;
    int err = 0;
    explicit ConstUse(icf_ctx *ctx)
    {
        if (!ctx->has_consts) {
            err = fail(ctx, ICF_E_NOCONST, "icf_set_constants has not been called");
            return;
        }
        if (ctx->capturing) return;
        lk = std::unique_lock<std::mutex>(g_dev_mu[ctx->device]);
        int &owner = g_const_owner[ctx->device];
        if (owner == ctx->id && !ctx->consts_dirty) return;
        hipError_t e = hipSuccess;
        if (owner != ctx->id && owner != 0) e = hipDeviceSynchronize();
        if (e == hipSuccess)
            e = hipMemcpyToSymbolAsync(HIP_SYMBOL(g_c), &ctx->hc, sizeof(DevConsts), 0, hipMemcpyHostToDevice,
                                       ctx->stream);
        if (e != hipSuccess) {
            owner = 0;
            err = fail(ctx, (int)e, std::string("loading the constants: ") + hipGetErrorString(e));
            return;
        }
        owner = ctx->id;
        ctx->consts_dirty = false;
    }
};

unsigned blocks_for(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipEvent_t prof_begin(icf_ctx *ctx)
{
    if (!ctx->profiling || ctx->capturing) return nullptr;
    hipEvent_t e = nullptr;
    if (!ctx->ev_pool.empty()) {
        e = ctx->ev_pool.back();
        ctx->ev_pool.pop_back();
    } else if (hipEventCreate(&e) != hipSuccess) {
        return nullptr;
    }
    (void)hipEventRecord(e, ctx->cur);
    return e;
}

void prof_end(icf_ctx *ctx, const char *name, hipEvent_t a)
{
    if (!a) return;
    hipEvent_t b = prof_begin(ctx);
    if (!b) {
        ctx->ev_pool.push_back(a);
        return;
    }
    ctx->pending.push_back({name, a, b});
}

// After the stream has drained: fold pending event pairs into the per-kernel totals.
void prof_flush(icf_ctx *ctx)
{
    for (auto &p : ctx->pending) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
            size_t i = 0;
            while (i < ctx->prof_names.size() && ctx->prof_names[i] != p.name) i++;
            if (i == ctx->prof_names.size()) {
                ctx->prof_names.push_back(p.name);
                ctx->prof_ms.push_back(0);
                ctx->prof_n.push_back(0);
            }
            ctx->prof_ms[i] += ms;
            ctx->prof_n[i] += 1;
        }
        ctx->ev_pool.push_back(p.a);
        ctx->ev_pool.push_back(p.b);
    }
    ctx->pending.clear();
}

// Kernel launch on the context's stream, bracketed by events when profiling is on.
#define LAUNCH(ctx, name, kern, g, b, ...)                                   \
    do {                                                                     \
        hipEvent_t ea_ = prof_begin(ctx);                                    \
        hipLaunchKernelGGL(kern, g, b, 0, (ctx)->cur, __VA_ARGS__);          \
        prof_end(ctx, name, ea_);                                            \
    } while (0)

int lane_barrier(icf_ctx *ctx);

// A slot map that a call needs.
struct MapReq {
    int target, fixed_nkeys;
    std::vector<SrcKey> srcs;
    SlotMap *map = nullptr;
};

MapSrc map_src(const SrcKey &k) { return MapSrc{k.base, k.n, k.stride, k.field0, k.nq, k.kind}; }
long long src_fields(const SrcKey &k) { return (long long)k.n * k.nq; }

// The workgroups of k_map_count, k_map_fill and k_snap_cmp over one more map's sources.
void add_srcs(MapJobs &J, int job, const SlotMap &m)
{
    for (size_t i = 0; i < m.srcs.size(); i++) {
        const SrcKey &k = m.srcs[i];
        if (k.n == 0) continue;
        const int n = J.nsrc++;
        J.src[n] = map_src(k);
        J.job[n] = job;
        J.snap[n] = m.snap[i];
        J.at[n] = n ? J.at[n - 1] + (long long)J.src[n - 1].n * J.src[n - 1].nq : 0;
        J.blk0[n + 1] = J.blk0[n] + blocks_for(k.n, 256) * (unsigned)k.nq;
    }
}

// Rows of the rhs map starting from the per-node tet sums of the force map (k_rhs_check); the
// outcome is in the report after the wait.
int launch_link(icf_ctx *ctx, SlotMap *mr, const SlotMap *mf, const MapSrc &tet, const Report &rep)
{
    mr->tsum_ok = mr->merge_ok = false;
    mr->tsum_with = -1;
    if (int r = grow(ctx, mr->b_row_node, sizeof(int) * (size_t)mr->nkeys)) return r;
    if (int r = grow(ctx, mr->b_cz_begin, sizeof(int) * (size_t)mr->nkeys)) return r;
    if (int r = grow(ctx, mr->b_node_row, sizeof(int) * (size_t)mf->nkeys)) return r;
    mr->row_node = (int *)mr->b_row_node.p;
    mr->cz_begin = (int *)mr->b_cz_begin.p;
    mr->node_row = (int *)mr->b_node_row.p;
    if (mf->nkeys)
        hipLaunchKernelGGL(k_fill_int, dim3(blocks_for(mf->nkeys, 256)), dim3(256), 0, ctx->stream, mr->node_row,
                           mf->nkeys, -1);
    if (mr->nkeys)
        hipLaunchKernelGGL(k_rhs_check, dim3(blocks_for(mr->nkeys, 256)), dim3(256), 0, ctx->stream, mr->off,
                           mr->codes, mr->nkeys, mf->off, mf->codes, mf->nkeys, tet, mr->row_node, mr->cz_begin,
                           mr->node_row, rep);
    return 0;
}

// Launches that build the maps `todo` (at most MAX_JOBS) into their buffers, and the link of rhs
// map `mr` to force map `mf` when given; then one wait.  A map without fixed_nkeys is counted over
// the keys its buffers hold; `over` tells where that was too few.
int build_maps(icf_ctx *ctx, const std::vector<SlotMap *> &todo, SlotMap *mr, const SlotMap *mf, const MapSrc *tet,
               bool over[MAX_JOBS])
{
    MapJobs J{};
    long long keys = 0, fields = 0;
    for (SlotMap *m : todo) {
        const int j = J.njob++;
        long long codes = 0;
        m->snap.assign(m->srcs.size(), nullptr);
        for (const SrcKey &k : m->srcs) codes += src_fields(k);
        if (int r = grow(ctx, m->b_off, sizeof(int) * ((size_t)m->nkeys + 1))) return r;
        if (int r = grow(ctx, m->b_codes, sizeof(uint32_t) * (size_t)(codes + 1))) return r;
        if (int r = grow(ctx, m->b_snap, sizeof(int) * (size_t)(codes + 1))) return r;
        const bool list = m->fixed_nkeys < 0;
        if (list) {
            const size_t most = (size_t)std::min<long long>(m->nkeys, codes) + 1;
            if (int r = grow(ctx, m->b_keys, sizeof(int) * most)) return r;
            if (int r = grow(ctx, m->b_loff, sizeof(int) * most)) return r;
        }
        m->off = (int *)m->b_off.p;
        m->codes = (uint32_t *)m->b_codes.p;
        m->keys = list ? (int *)m->b_keys.p : nullptr;
        m->loff = list ? (int *)m->b_loff.p : m->off;
        int *snap = (int *)m->b_snap.p;
        for (size_t i = 0; i < m->srcs.size(); i++) {
            m->snap[i] = snap;
            snap += src_fields(m->srcs[i]);
        }
        add_srcs(J, j, *m);
        J.nkeys[j] = m->nkeys;
        J.vals[j] = m->target == TGT_VALS;
        J.cnt0[j] = keys;
        J.tile0[j + 1] = J.tile0[j] + std::max(blocks_for(m->nkeys, SCAN_TILE), 1u);
        J.sort0[j + 1] = J.sort0[j] + blocks_for(m->nkeys, 256);
        J.off[j] = m->off;
        J.codes[j] = m->codes;
        J.keys[j] = m->keys;
        J.loff[j] = list ? m->loff : nullptr;
        keys += m->nkeys;
        fields += codes;
    }
    const size_t cnt_bytes = sizeof(int) * (size_t)std::max(keys, 1LL);
    if (ctx->map_cnt.bytes < cnt_bytes) {
        if (int r = grow(ctx, ctx->map_cnt, cnt_bytes)) return r;
        HIPCHK(ctx, hipMemsetAsync(ctx->map_cnt.p, 0, ctx->map_cnt.bytes, ctx->stream));
    }
    if (int r = grow(ctx, ctx->map_rank, sizeof(int) * (size_t)std::max(fields, 1LL))) return r;
    const unsigned tiles = J.tile0[J.njob], sorts = J.sort0[J.njob], places = J.nsrc ? J.blk0[J.nsrc] : 0;
    if (int r = grow(ctx, ctx->map_sums, sizeof(unsigned long long) * std::max(tiles, 1u))) return r;
    int *cnt = (int *)ctx->map_cnt.p, *rank = (int *)ctx->map_rank.p;
    auto *sums = (unsigned long long *)ctx->map_sums.p;
    const Report rep = new_report(ctx);
    if (J.njob) {
        const dim3 b(256);
        if (places) hipLaunchKernelGGL(k_map_count, dim3(places), b, 0, ctx->stream, J, cnt, rank, rep);
        hipLaunchKernelGGL(k_map_tiles, dim3(tiles), b, 0, ctx->stream, J, cnt, sums);
        hipLaunchKernelGGL(k_map_offsets, dim3(tiles), b, 0, ctx->stream, J, cnt, sums, rep);
        if (places) hipLaunchKernelGGL(k_map_fill, dim3(places), b, 0, ctx->stream, J, rank);
        if (sorts) hipLaunchKernelGGL(k_map_sort, dim3(sorts), b, 0, ctx->stream, J);
    }
    if (mr)
        if (int r = launch_link(ctx, mr, mf, *tet, rep)) return r;
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    for (int j = 0; j < J.njob; j++) {
        SlotMap *m = todo[j];
        over[j] = reported(rep, MAP_ERR + j);
        m->nlaunch = m->fixed_nkeys < 0 ? (int)((volatile unsigned *)rep.host)[MAP_NLIST + j] : m->nkeys;
        m->id = ++ctx->next_map_id;
        m->suspect = m->changed = false;
        m->built = !over[j];
    }
    if (mr) {
        mr->tsum_with = mf->id;
        mr->tsum_ok = mr->nkeys > 0 && !reported(rep, LINK_ERR);
        mr->merge_ok = mr->tsum_ok && mf->nkeys > 0 && !reported(rep, LINK_ERR + 1);
    }
    return 0;
}

// The new offsets of an overwrite value map (m.nkeys keys, nold before) whose slots may only have
// moved (k_map_move); one wait.  `moved` tells whether they had; if not, the map is to be built.
int move_map(icf_ctx *ctx, SlotMap &m, int nold, bool &moved)
{
    MapJobs J{};
    J.njob = 1;
    add_srcs(J, 0, m);
    J.nkeys[0] = m.nkeys;
    J.tile0[1] = std::max(blocks_for(m.nkeys, SCAN_TILE), 1u);
    if (int r = grow(ctx, m.b_off2, sizeof(int) * ((size_t)m.nkeys + 1))) return r;
    if (int r = grow(ctx, ctx->map_rank, sizeof(int) * (size_t)std::max(nold, 1))) return r;
    if (int r = grow(ctx, ctx->map_sums, sizeof(unsigned long long) * std::max(J.tile0[1], 1u))) return r;
    const size_t cnt_bytes = sizeof(int) * (size_t)std::max(m.nkeys, 1);
    if (ctx->map_cnt.bytes < cnt_bytes) {
        if (int r = grow(ctx, ctx->map_cnt, cnt_bytes)) return r;
        HIPCHK(ctx, hipMemsetAsync(ctx->map_cnt.p, 0, ctx->map_cnt.bytes, ctx->stream));
    }
    int *cnt = (int *)ctx->map_cnt.p, *to = (int *)ctx->map_rank.p, *now = (int *)m.b_off2.p;
    auto *sums = (unsigned long long *)ctx->map_sums.p;
    J.off[0] = now;
    const unsigned places = J.nsrc ? J.blk0[J.nsrc] : 0, olds = blocks_for(nold, 256);
    const Report rep = new_report(ctx);
    const dim3 b(256);
    if (places) hipLaunchKernelGGL(k_map_move, dim3(places), b, 0, ctx->stream, J, to, rep);
    if (places + olds)
        hipLaunchKernelGGL(k_map_moved, dim3(places + olds), b, 0, ctx->stream, J, places, to, m.off, nold, cnt, rep);
    hipLaunchKernelGGL(k_map_tiles, dim3(J.tile0[1]), b, 0, ctx->stream, J, cnt, sums);
    hipLaunchKernelGGL(k_map_offsets, dim3(J.tile0[1]), b, 0, ctx->stream, J, cnt, sums, rep);
    if (olds) hipLaunchKernelGGL(k_map_runs, dim3(olds), b, 0, ctx->stream, to, m.off, nold, now, rep);
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    moved = !reported(rep, MAP_MOVED);
    if (!moved) return 0;
    std::swap(m.b_off, m.b_off2);
    m.off = m.loff = now;
    m.nlaunch = m.nkeys;
    m.id = ++ctx->next_map_id;
    m.suspect = m.changed = false;
    m.built = true;
    return 0;
}

void drop_map(icf_ctx *ctx, SlotMap *m)
{
    for (auto it = ctx->maps.begin(); it != ctx->maps.end(); ++it)
        if (&*it == m) {
            (void)hipStreamSynchronize(ctx->stream);
            free_map(*it);
            ctx->maps.erase(it);
            return;
        }
}

// Finds or builds the slot maps of one call (at most MAX_JOBS): one wait when any had to be
// compared with its fields, one when any had to be built.  `link`: requests 1 (rhs rows) and 2
// (node forces, over the tets `tet`) are the fused call's, whose rows may start from the forces'
// tet sums.  A map whose fields were written since is built anew in its own buffers, also for
// another number of units: the unit lists of a Newton loop change from call to call.
int get_maps(icf_ctx *ctx, std::vector<MapReq> &req, const MapSrc *tet = nullptr)
{
    const int nreq = (int)req.size();
    MapJobs S{};
    bool checked = false;
    for (int i = 0; i < nreq; i++) {
        MapReq &r = req[i];
        for (SlotMap &m : ctx->maps)
            if (m.target == r.target && m.fixed_nkeys == r.fixed_nkeys && m.srcs == r.srcs) r.map = &m;
        if (r.map && r.map->suspect) {
            if (ctx->capturing)
                return fail(ctx, ICF_E_CAPTURE, "a slot map must be checked during capture: run the call once uncaptured");
        }
    }
    // Suspect maps are compared with their fields, except those known to have changed and, beside
    // those, maps of fewer fields than they have: building them too costs less than a wait of its own
    // (15 us a call).
    long long changed = 0, unsure = 0;
    for (MapReq &r : req) {
        if (!r.map || !r.map->suspect) continue;
        long long n = 0;
        for (const SrcKey &s : r.srcs) n += src_fields(s);
        (r.map->changed ? changed : unsure) += n;
    }
    for (int i = 0; i < nreq; i++) {
        SlotMap *m = req[i].map;
        if (!m || !m->suspect || m->changed || unsure < changed) continue;
        add_srcs(S, i, *m);
        checked = true;
    }
    if (!ctx->capturing && (!std::all_of(req.begin(), req.end(), [](const MapReq &r) { return r.map && !r.map->suspect; })))
        if (int r = lane_barrier(ctx)) return r;      // fields may have been written on the other lane
    if (checked) {
        const Report rep = new_report(ctx);
        if (S.nsrc) hipLaunchKernelGGL(k_snap_cmp, dim3(S.blk0[S.nsrc]), dim3(256), 0, ctx->stream, S, rep);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        for (int i = 0; i < nreq; i++)
            if (req[i].map && req[i].map->suspect && !reported(rep, SNAP_DIFF + i) && !req[i].map->changed)
                req[i].map->suspect = false;
    }
    std::vector<SlotMap *> todo, first;
    int nold = -1;                     // keys of the last of them if its slots may only have moved
    for (MapReq &r : req) {
        if (r.map && !r.map->suspect) continue;
        if (ctx->capturing)
            return fail(ctx, ICF_E_CAPTURE, "a slot map would be built during capture: run the call once uncaptured");
        for (const SrcKey &s : r.srcs)
            if ((uint32_t)s.n > CODE_UNIT_MAX + 1u)
                return fail(ctx, ICF_E_CAPACITY, "more than 2^24 units in one pcsr array");
        if (!r.map) {
            // a map over the same arrays whose fields were written since
            auto same = [&](const SlotMap &m) {
                if (m.target != r.target || (m.fixed_nkeys < 0) != (r.fixed_nkeys < 0) || !m.suspect ||
                    m.srcs.size() != r.srcs.size())
                    return false;
                for (size_t k = 0; k < r.srcs.size(); k++)
                    if (m.srcs[k].base != r.srcs[k].base || m.srcs[k].kind != r.srcs[k].kind) return false;
                return std::none_of(req.begin(), req.end(), [&](const MapReq &q) { return q.map == &m; });
            };
            for (SlotMap &m : ctx->maps)
                if (!r.map && same(m)) r.map = &m;
            if (!r.map) {
                ctx->maps.emplace_back();
                r.map = &ctx->maps.back();
            }
        }
        SlotMap &m = *r.map;
        nold = m.built && m.target == TGT_VALS && m.fixed_nkeys >= 0 && m.srcs == r.srcs ? m.nkeys : -1;
        if (m.built) bump(ctx);
        m.built = false;
        m.suspect = true;              // until it is built
        m.changed = true;
        m.tsum_with = -1;
        m.target = r.target;
        m.fixed_nkeys = r.fixed_nkeys;
        m.srcs = r.srcs;
        if (r.fixed_nkeys >= 0) m.nkeys = r.fixed_nkeys;
        else if (m.nkeys == 0) first.push_back(&m);
        todo.push_back(&m);
    }
    auto drop = [&](int code, const char *msg) {
        for (SlotMap *m : todo) drop_map(ctx, m);
        return fail(ctx, code, msg);
    };
    // maps that count as many keys as their fields need: the largest key, with room for more
    auto size_keys = [&](const std::vector<SlotMap *> &ms) -> int {
        int *d_max = ctx->small + 8, init[4] = {-1, -1, -1, -1}, mx[4];
        HIPCHK(ctx, hipMemcpyAsync(d_max, init, sizeof(init), hipMemcpyHostToDevice, ctx->stream));
        for (size_t j = 0; j < ms.size(); j++)
            for (const SrcKey &s : ms[j]->srcs) {
                if (s.n == 0) continue;
                const unsigned nb = blocks_for(src_fields(s), 256);
                hipLaunchKernelGGL(k_map_maxkey, dim3(nb < 1024 ? nb : 1024), dim3(256), 0, ctx->stream, map_src(s),
                                   d_max + j);
            }
        HIPCHK(ctx, hipMemcpyAsync(mx, d_max, sizeof(mx), hipMemcpyDeviceToHost, ctx->stream));
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        for (size_t j = 0; j < ms.size(); j++)
            ms[j]->nkeys = (int)std::min<long long>(mx[j] + 1LL + (mx[j] + 1LL) / 8, INT_MAX - 1);
        return 0;
    };
    SlotMap *mr = nullptr, *mf = nullptr;
    if (tet && nreq == 3 &&
        (!req[1].map->built || !req[2].map->built || req[1].map->tsum_with != req[2].map->id)) {
        if (ctx->capturing)
            return fail(ctx, ICF_E_CAPTURE, "a slot map would be built during capture: run the call once uncaptured");
        mr = req[1].map;
        mf = req[2].map;
    }
    if (todo.empty() && !mr) return 0;
    bool over[MAX_JOBS] = {};
    int err = first.empty() ? 0 : size_keys(first);
    if (!err && todo.size() == 1 && !mr && nold >= 0) {
        bool moved = false;
        err = move_map(ctx, *todo[0], nold, moved);
        if (moved) return 0;
    }
    if (!err) err = build_maps(ctx, todo, mr, mf, tet, over);
    std::vector<SlotMap *> again;
    bool bad = false;
    for (size_t j = 0; j < todo.size() && !err; j++)
        if (over[j]) {
            if (todo[j]->fixed_nkeys >= 0) bad = true;
            else again.push_back(todo[j]);
        }
    if (!err && !bad && !again.empty()) {
        err = size_keys(again);
        bool over2[MAX_JOBS] = {};
        if (!err) err = build_maps(ctx, again, mr, mf, tet, over2);
        for (bool o : over2) bad = bad || o;
    }
    if (bad) return drop(ICF_E_INDEX, "a slot/row/node index exceeds the declared size");
    if (err) {
        const std::string why = ctx->err;
        return drop(err, why.c_str());
    }
    return 0;
}

int check_ctx(icf_ctx *ctx)
{
    if (!ctx) return ICF_E_INVALID;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    return 0;
}

struct Timer {
    icf_ctx *ctx;
    bool sync;
    explicit Timer(icf_ctx *c) : ctx(c), sync(c->blocking && !c->capturing)
    {
        ctx->last_ms = -1;
        if (sync) (void)hipEventRecord(ctx->ev0, ctx->stream);
    }
    int finish()
    {
        if (!sync) {
            HIPCHK(ctx, hipGetLastError());
            return 0;
        }
        HIPCHK(ctx, hipEventRecord(ctx->ev1, ctx->stream));
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        float ms = 0;
        HIPCHK(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        ctx->last_ms = ms;
        prof_flush(ctx);
        HIPCHK(ctx, hipGetLastError());
        return 0;
    }
};

// ---- launch helpers ---------------------------------------------------------------------------

// ---- lanes across calls -----------------------------------------------------------------------
// When calls are enqueued without waiting (icf_set_blocking(0), outside capture, overlap on), the
// contact-detection work -- narrow phase, closest face, the per-impact phase of the collision
// response -- runs on lane 1 (`stream_c`) beside the assembly on lane 0 (`stream`).  Every call
// declares the device bytes it reads and writes; before issuing, it waits for the latest call of
// the other lane whose bytes conflict with its own (one of the two writes bytes the other
// touches).  Blocking calls finish before they return, and captured calls replay as one graph
// (whose independent branches the HIP runtime was measured to run one after the other), so
// both use lane 0 only; lane-0 work that was not logged is waited for in full by the next
// lane-1 call.

bool lanes_on(const icf_ctx *ctx) { return ctx->overlap && !ctx->profiling && !ctx->blocking && !ctx->capturing; }

hipStream_t lane_stream(const icf_ctx *ctx, int l) { return l ? ctx->stream_c : ctx->stream; }

// lane for a call that may run on lane 1
int contact_lane(const icf_ctx *ctx) { return lanes_on(ctx) ? 1 : 0; }

hipEvent_t next_lane_event(icf_ctx *ctx, int l) { return ctx->lane_ev[l][ctx->lane_ev_next[l]++ % LANE_EVENTS]; }

// `access` returns the call's Access; it is only evaluated when the other lane has logged calls
template <typename G> int lane_enter(icf_ctx *ctx, int l, G &&access)
{
    if (l == 1 && ctx->lane0_unlogged) {
        hipEvent_t ev = next_lane_event(ctx, 0);
        HIPCHK(ctx, hipEventRecord(ev, ctx->stream));
        HIPCHK(ctx, hipStreamWaitEvent(ctx->stream_c, ev, 0));
        ctx->lane_log[0].clear();
        ctx->lane0_unlogged = false;
    }
    std::vector<LaneRec> &other = ctx->lane_log[1 - l];
    if (!other.empty()) {
        auto &&a = access();
        for (int i = (int)other.size() - 1; i >= 0; i--) {
            if (!conflict(a, other[i].a)) continue;
            HIPCHK(ctx, hipStreamWaitEvent(lane_stream(ctx, l), other[i].ev, 0));
            // the other lane's calls up to i are now ordered before everything later on this lane
            other.erase(other.begin(), other.begin() + i + 1);
            break;
        }
    }
    ctx->cur = lane_stream(ctx, l);
    return 0;
}

template <typename G> int lane_exit(icf_ctx *ctx, int l, G &&access)
{
    ctx->cur = ctx->stream;
    if (l == 0 && !lanes_on(ctx)) {
        ctx->lane0_unlogged = true;
        return 0;
    }
    hipEvent_t ev = next_lane_event(ctx, l);
    HIPCHK(ctx, hipEventRecord(ev, lane_stream(ctx, l)));
    std::vector<LaneRec> &log = ctx->lane_log[l];
    if ((int)log.size() + 1 >= LANE_LOG) {
        // the latest event stands for every earlier call of the lane
        log.clear();
        log.push_back({Access::everything(), ev});
    } else {
        log.push_back({access(), ev});
    }
    return 0;
}

Access everything() { return Access::everything(); }

// A call that touches unknown memory, or returns host data: after all lane-1 work.
int lane_barrier(icf_ctx *ctx) { return lane_enter(ctx, 0, everything); }

// Both lanes idle, logs empty.
int sync_lanes(icf_ctx *ctx)
{
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream_c));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    ctx->lane_log[0].clear();
    ctx->lane_log[1].clear();
    ctx->lane0_unlogged = false;
    return 0;
}

// One call's lane: enters on construction (check `err`), done() logs it.  `make` builds the
// call's Access when a lane needs it.
template <typename F> struct OnLane {
    icf_ctx *ctx;
    int lane;
    F make;
    Access acc;
    bool have = false;
    int err = 0;
    OnLane(icf_ctx *c, int l, F f) : ctx(c), lane(l), make(f)
    {
        err = lane_enter(ctx, lane, [this]() -> const Access & { return get(); });
    }
    const Access &get()
    {
        if (!have) {
            acc = make();
            have = true;
        }
        return acc;
    }
    int done() { return lane_exit(ctx, lane, [this]() -> const Access & { return get(); }); }
    ~OnLane() { ctx->cur = ctx->stream; }
};

// Plane stride of the tet staging records for n tets.
int tet_plane(long long n) { return (int)((std::max(n, 1LL) + 63) / 64 * 64); }

// Staged tet records of more than this many bytes are written with nontemporal stores: they
// would not stay in the caches until phase 2 reads them anyway (measured: 3.5M tets faster
// with them, 384k tets faster without).
constexpr size_t STREAM_STAGING_BYTES = 128u << 20;
bool stream_tet_staging(const icf_ctx *ctx, int n)
{
    const size_t rec = (ctx->hc.iso ? TET_ISO_REC : TET_GEN_REC) * (ctx->precision == ICF_MIXED ? 4 : 8);
    return (size_t)tet_plane(n) * (rec + sizeof(double) * TET_RHS_REC) > STREAM_STAGING_BYTES;
}

// Staging buffers of a call over nt tets and nc CZs; their tangent records share one buffer.
int reserve_stage(icf_ctx *ctx, int nt, int nc)
{
    const size_t val = ctx->precision == ICF_MIXED ? 4 : 8, rec = ctx->hc.iso ? TET_ISO_REC : TET_GEN_REC;
    const size_t cap = (size_t)tet_plane(nt), tets = val * rec * cap;
    if (int r = grow(ctx, ctx->tet_rhs, sizeof(double) * TET_RHS_REC * cap)) return r;
    if (int r = grow(ctx, ctx->cz_rhs, sizeof(double) * CZ_RHS_REC * (size_t)std::max(nc, 1))) return r;
    if (int r = grow(ctx, ctx->tan, tets + val * CZ_TAN_REC * (size_t)nc)) return r;
    ctx->cz_word = (uint32_t)(tets / 8);
    return 0;
}
void *cz_records(const icf_ctx *ctx) { return (double *)ctx->tan.p + ctx->cz_word; }

void stage_tets(icf_ctx *ctx, const int *ie, const double *dn, int n, int es, int ns)
{
    const bool mixed = ctx->precision == ICF_MIXED, iso = ctx->hc.iso != 0;
    if (n == 0) return;
    const int tp = ctx->tplane = tet_plane(n);
    dim3 g(blocks_for(n, 256)), b(256);
    double *sr = (double *)ctx->tet_rhs.p;
    void *st = ctx->tan.p;
    const bool so = stream_tet_staging(ctx, n);
#define ICF_T1(MX, IS, NAME)                                                                                   \
    do {                                                                                                      \
        if (so) LAUNCH(ctx, NAME, (k_tet_phase1<MX, IS, true>), g, b, ie, dn, n, tp, es, ns, sr, st);         \
        else LAUNCH(ctx, NAME, (k_tet_phase1<MX, IS, false>), g, b, ie, dn, n, tp, es, ns, sr, st);           \
    } while (0)
    if (mixed && iso) ICF_T1(true, true, "k_tet_phase1<mixed,iso>");
    else if (mixed) ICF_T1(true, false, "k_tet_phase1<mixed,gen>");
    else if (iso) ICF_T1(false, true, "k_tet_phase1<fp64,iso>");
    else ICF_T1(false, false, "k_tet_phase1<fp64,gen>");
#undef ICF_T1
}

void stage_czs(icf_ctx *ctx, double *dcz, int *icz, const double *dn, int n, int cs, int ns)
{
    const bool mixed = ctx->precision == ICF_MIXED;
    if (n == 0) return;
    const long long waves = (n + CZ_PER_WAVE - 1) / CZ_PER_WAVE;   // three lanes per CZ
    dim3 g(blocks_for(waves * 64, 256)), b(256);
    if (mixed)
        LAUNCH(ctx, "k_cz_phase1<mixed>", (k_cz_phase1<true>), g, b, dcz, icz, dn, n, cs, ns, (double *)ctx->cz_rhs.p,
               cz_records(ctx));
    else
        LAUNCH(ctx, "k_cz_phase1<fp64>", (k_cz_phase1<false>), g, b, dcz, icz, dn, n, cs, ns, (double *)ctx->cz_rhs.p,
               cz_records(ctx));
}

// ---- autotuner of the launch shapes -----------------------------------------------------------
// While a role is being tuned, its launches cycle through the role's candidates, each timed
// with a pair of events around the launch; the next launch of the role reads the previous
// timing (waiting for it if it has not finished), and after tune_rounds timings per candidate
// the fastest launch decides.  Captured calls are not timed; they use the current choice.
// Roles: the value reductions' chunk shape per (accumulate map, FP64 staging) (eight
// candidates), and the shape roles (three candidates each).  A finished tuning is also kept in
// a cache held by the library, per device, role, precision and size class (the launch's units,
// to the next power of two): contexts whose role is neither being tuned nor set by the caller
// take the cached choice for launches of that size class.

struct ShapeCache {
    std::mutex mu;
    std::map<std::array<int, 4>, int> choice;   // (device, role id, precision, size class) -> candidate
};
ShapeCache g_shape_cache;

int size_class(long long n)
{
    int b = 0;
    while (b < 62 && (1LL << b) < n) b++;
    return b;
}

void tune_fold(icf_ctx *ctx, icf_ctx::Tune &t, int role_id)
{
    if (t.cand >= 0) {
        float ms = 0;
        if (hipEventSynchronize(t.ev[1]) == hipSuccess && hipEventElapsedTime(&ms, t.ev[0], t.ev[1]) == hipSuccess &&
            ms > 0) {
            if (t.best[t.cand] == 0 || ms < t.best[t.cand]) t.best[t.cand] = ms;
            t.samples++;
        }
        t.cand = -1;
    }
    if (t.active && (t.samples >= ctx->tune_rounds * t.ncand || t.turn >= 4 * ctx->tune_rounds * t.ncand)) {
        t.active = false;
        t.tuned = true;
        for (int c = 0; c < t.ncand; c++)
            if (t.best[c] > 0 && (t.best[t.sel] == 0 || t.best[c] < t.best[t.sel])) t.sel = c;
        if (t.bucket >= 0) {
            std::lock_guard<std::mutex> lk(g_shape_cache.mu);
            g_shape_cache.choice[{ctx->device, role_id, ctx->precision, t.bucket}] = t.sel;
        }
    }
}

// The candidate for the next launch of a role with `units` units; starts its timing if tuning
// (not when `peek`).
int tune_begin(icf_ctx *ctx, icf_ctx::Tune &t, int role_id, long long units, bool peek = false)
{
    const int bucket = size_class(units) + (units <= t.small_max ? 64 : 0);   // small launches are apart
    if (!t.active || ctx->capturing || peek) {
        t.last = t.sel;
        if (!t.active && !t.fixed) {
            std::lock_guard<std::mutex> lk(g_shape_cache.mu);
            auto it = g_shape_cache.choice.find({ctx->device, role_id, ctx->precision, bucket});
            if (it != g_shape_cache.choice.end()) t.last = it->second;
            else if (!t.tuned) t.last = units <= t.small_max ? t.small : t.untuned;
        }
        return t.last;
    }
    tune_fold(ctx, t, role_id);
    if (!t.active) return t.last = t.sel;
    t.bucket = bucket;
    t.last = t.cand = t.turn++ % t.ncand;
    (void)hipEventRecord(t.ev[0], ctx->cur);
    return t.cand;
}

void tune_end(icf_ctx *ctx, icf_ctx::Tune &t)
{
    if (t.cand >= 0 && !ctx->capturing) (void)hipEventRecord(t.ev[1], ctx->cur);
}

// value-reduction roles: ids 0-3
int tune_begin(icf_ctx *ctx, bool acc, bool fp64, long long keys)
{
    return tune_begin(ctx, ctx->tune[acc][fp64], 2 * acc + fp64, keys);
}
void tune_end(icf_ctx *ctx, bool acc, bool fp64) { tune_end(ctx, ctx->tune[acc][fp64]); }

// shape roles: ids 4-7; returns the role's value (workgroup size or lanes per tuple)
int shape_begin(icf_ctx *ctx, int role, long long units, bool peek = false)
{
    return shape_value(role, tune_begin(ctx, ctx->shape[role], 4 + role, units, peek));
}
void shape_end(icf_ctx *ctx, int role) { tune_end(ctx, ctx->shape[role]); }

// ---- fused launches (icf_fused.inc.h) ----------------------------------------------------------

int round8(long long n) { return (int)((n + 7) / 8 * 8); }

// Phase 1 of the fused call as one launch; the staging buffers have already grown.
void phase1_fused(icf_ctx *ctx, const int *ie, const double *dn, int nt, int es, int ns, double *dcz, int *icz, int nc,
                  int cs, int *counts)
{
    const bool mixed = ctx->precision == ICF_MIXED, iso = ctx->hc.iso != 0;
    const int B = shape_begin(ctx, ICF_SHAPE_PHASE1, (long long)nt + nc);
    const int nbt = nt ? round8(blocks_for(nt, B)) : 0;
    const int nbc = nc ? (int)blocks_for((long long)(nc + CZ_PER_WAVE - 1) / CZ_PER_WAVE * 64, B) : 0;
    const dim3 g(std::max(interleave2_grid(nbt, nbc), 1)), b(B);
    double *tr = (double *)ctx->tet_rhs.p, *cr = (double *)ctx->cz_rhs.p;
    void *tt = ctx->tan.p, *ct = cz_records(ctx);
    const int tp = ctx->tplane = tet_plane(nt);
    const bool so = stream_tet_staging(ctx, nt);
#define ICF_P1(MX, IS, NAME)                                                                                      \
    do {                                                                                                          \
        if (so)                                                                                                   \
            LAUNCH(ctx, NAME, (k_phase1_fused<MX, IS, true>), g, b, nbt, nbc, ie, dn, nt, tp, es, ns, tr, tt, dcz, \
                   icz, nc, cs, cr, ct, counts);                                                                  \
        else                                                                                                      \
            LAUNCH(ctx, NAME, (k_phase1_fused<MX, IS, false>), g, b, nbt, nbc, ie, dn, nt, tp, es, ns, tr, tt, dcz, \
                   icz, nc, cs, cr, ct, counts);                                                                  \
    } while (0)
    if (mixed && iso) ICF_P1(true, true, "k_phase1<mixed,iso>");
    else if (mixed) ICF_P1(true, false, "k_phase1<mixed,gen>");
    else if (iso) ICF_P1(false, true, "k_phase1<fp64,iso>");
    else ICF_P1(false, false, "k_phase1<fp64,gen>");
#undef ICF_P1
    shape_end(ctx, ICF_SHAPE_PHASE1);
}

// Calls f(integral_constant<cand_keys(c)>, integral_constant<cand_stage(c)>); OVER: for a launch that
// overwrites `keys` blocks, where few of them give the candidates of 64 keys more room.
template <bool OVER, typename F>
void with_cand(int c, long long keys, F &&f)
{
    static_assert(NCAND == 8, "one case per candidate");
    using std::integral_constant;
    if constexpr (OVER) {
        if (cand_keys(c) == SMALL_KEYS && keys <= VALS_SMALL)
            return f(integral_constant<int, SMALL_KEYS>(), integral_constant<int, SMALL_STAGE>());
    }
    switch (c) {
    case 0: f(integral_constant<int, cand_keys(0)>(), integral_constant<int, cand_stage(0)>()); break;
    case 1: f(integral_constant<int, cand_keys(1)>(), integral_constant<int, cand_stage(1)>()); break;
    case 2: f(integral_constant<int, cand_keys(2)>(), integral_constant<int, cand_stage(2)>()); break;
    case 3: f(integral_constant<int, cand_keys(3)>(), integral_constant<int, cand_stage(3)>()); break;
    case 4: f(integral_constant<int, cand_keys(4)>(), integral_constant<int, cand_stage(4)>()); break;
    case 5: f(integral_constant<int, cand_keys(5)>(), integral_constant<int, cand_stage(5)>()); break;
    case 6: f(integral_constant<int, cand_keys(6)>(), integral_constant<int, cand_stage(6)>()); break;
    default: f(integral_constant<int, cand_keys(7)>(), integral_constant<int, cand_stage(7)>()); break;
    }
}

// BCSR values (overwrite) and node forces with their tet sums as one launch.  False when the
// value map is an accumulate map: the caller launches them apart.
bool vals_force_fused(icf_ctx *ctx, const SlotMap *mv, double *A, const SlotMap *mf, double *F, int ns,
                      const Stage &st)
{
    if (mv->keys) return false;
    if (mv->nlaunch == 0 && mf->nlaunch == 0) return true;
    const bool mixed = ctx->precision == ICF_MIXED, iso = ctx->hc.iso != 0;
    double *ts = (double *)ctx->tsum.p;
    const int c = tune_begin(ctx, false, !mixed, mv->nlaunch);
    const int ilv = shape_begin(ctx, ICF_SHAPE_ORDER, mv->nlaunch);
    with_cand<true>(c, mv->nlaunch, [&](auto kc, auto sc) {
        constexpr int K = decltype(kc)::value, S = decltype(sc)::value;
        const int nch = (int)blocks_for(mv->nlaunch, K);
        const int nbf = mf->nlaunch ? round8(blocks_for(mf->nlaunch, K)) : 0;
        const dim3 g(interleave2_grid(nbf, nch)), b(K);   // not empty: at least one map has keys
#define ICF_VF(MX, IS, L, NAME)                                                                                   \
    LAUNCH(ctx, NAME, (k_vals_force_fused<MX, IS, L, K, S>), g, b, nbf, mv->loff, mv->codes, mv->nlaunch, nch, A, \
           mf->loff, mf->codes, mf->keys, mf->nlaunch, F, ns, st, ts, ilv)
        if (mixed && iso) ICF_VF(true, true, float, "k_vals_force<mixed,iso>");
        else if (mixed) ICF_VF(true, false, float, "k_vals_force<mixed,gen>");
        else if (iso) ICF_VF(false, true, double, "k_vals_force<fp64,iso>");
        else ICF_VF(false, false, double, "k_vals_force<fp64,gen>");
#undef ICF_VF
    });
    shape_end(ctx, ICF_SHAPE_ORDER);
    tune_end(ctx, false, !mixed);
    return true;
}

// The second half of the fused call as one launch: node forces with the rhs rows, the CZ
// counters and the BCSR values (overwrite).  False unless the rhs map's rows each have their
// tet node (merge_ok) and the value map is an overwrite map.  The counters go to `rep` too unless its
// host words are null.
bool vals_force_rhs_fused(icf_ctx *ctx, const SlotMap *mv, double *A, const SlotMap *mf, double *F, int ns,
                          const SlotMap *mr, double *b, const int *dmg, const int *fld, int nCZs, int *counts,
                          const Stage &st, const Report &rep)
{
    if (mv->keys || !mr->merge_ok || !mr->node_row) return false;
    if (mv->nlaunch == 0 && mf->nlaunch == 0 && nCZs == 0) return true;
    const bool mixed = ctx->precision == ICF_MIXED, iso = ctx->hc.iso != 0;
    const int c = tune_begin(ctx, false, !mixed, mv->nlaunch);
    const int ilv = shape_begin(ctx, ICF_SHAPE_ORDER, mv->nlaunch);
    with_cand<true>(c, mv->nlaunch, [&](auto kc, auto sc) {
        constexpr int K = decltype(kc)::value, S = decltype(sc)::value;
        const int nch = (int)blocks_for(mv->nlaunch, K);
        const int nbf = mf->nlaunch ? round8(blocks_for(mf->nlaunch, K)) : 0;
        // the CZ counters' workgroups: per specimen in a batched call (one or more specimens
        // each), else strided over all CZs
        const auto &bt = ctx->batch;
        const bool per_spec = bt.cz_off && nCZs;
        const int nbc = per_spec ? round8(std::min(bt.n, 64))
                                 : nCZs ? round8(std::min<long long>(blocks_for(nCZs, K), 64)) : 0;
        const dim3 g(nbc + interleave2_grid(nbf, nch)), bl(K);   // not empty: something has keys or CZs
#define ICF_VFR(MX, IS, L, NAME)                                                                                   \
    LAUNCH(ctx, NAME, (k_vals_force_rhs_fused<MX, IS, L, K, S>), g, bl, nbf, nbc, mv->loff, mv->codes, mv->nlaunch, \
           nch, A, mf->loff, mf->codes, mf->keys, mf->nlaunch, F, ns, mr->node_row, mr->off, mr->codes, mr->cz_begin, \
           b, dmg, fld, nCZs, counts, per_spec ? bt.cz_off : nullptr, bt.n, bt.spec_counts, st, ilv, rep)
        if (mixed && iso) ICF_VFR(true, true, float, "k_vals_force_rhs<mixed,iso>");
        else if (mixed) ICF_VFR(true, false, float, "k_vals_force_rhs<mixed,gen>");
        else if (iso) ICF_VFR(false, true, double, "k_vals_force_rhs<fp64,iso>");
        else ICF_VFR(false, false, double, "k_vals_force_rhs<fp64,gen>");
#undef ICF_VFR
        ctx->batch.spec_counted = per_spec;
    });
    shape_end(ctx, ICF_SHAPE_ORDER);
    tune_end(ctx, false, !mixed);
    return true;
}

// The collision response's sums into node forces, BCSR blocks and rhs rows as one launch.
// False when the value map is an overwrite map.
bool contact_sums_fused(icf_ctx *ctx, const SlotMap *mf, double *F, int ns, const SlotMap *mv, double *A,
                        const SlotMap *mr, double *b, const Stage &st)
{
    if (!mv->keys) return false;
    if (mf->nlaunch == 0 && mv->nlaunch == 0 && mr->nlaunch == 0) return true;
    const bool mixed = ctx->precision == ICF_MIXED;
    const int c = tune_begin(ctx, true, !mixed, mv->nlaunch);
    with_cand<false>(c, mv->nlaunch, [&](auto kc, auto sc) {
        constexpr int K = decltype(kc)::value, S = decltype(sc)::value;
        const int nch = (int)blocks_for(mv->nlaunch, K);
        const int nb0 = mf->nlaunch ? round8(blocks_for(mf->nlaunch, K)) : 0, nb1 = round8(nch);
        const int nb2 = mr->nlaunch ? (int)blocks_for(mr->nlaunch, K) : 0;
        const dim3 g(nb0 + nb1 + nb2), bl(K);
#define ICF_CS(MX, L, NAME)                                                                                       \
    LAUNCH(ctx, NAME, (k_contact_sums<MX, L, K, S>), g, bl, nb0, nb1, mf->loff, mf->codes, mf->keys, mf->nlaunch, F, ns, \
           mv->loff, mv->codes, mv->keys, mv->nlaunch, A, mr->loff, mr->codes, mr->keys, mr->nlaunch, b, st)
        if (mixed) ICF_CS(true, float, "k_contact_sums<mixed>");
        else ICF_CS(false, double, "k_contact_sums<fp64>");
#undef ICF_CS
    });
    tune_end(ctx, true, !mixed);
    return true;
}

Stage make_stage(icf_ctx *ctx, double h)
{
    Stage sv;
    sv.tet_rhs = (const double *)ctx->tet_rhs.p;
    sv.tan = ctx->tan.p;
    sv.cz_word = ctx->cz_word;
    sv.tplane = ctx->tplane;
    sv.cz_rhs = (const double *)ctx->cz_rhs.p;
    sv.ct_tan = ctx->ct.p;
    sv.ct_f = (const double *)ctx->ct_f.p;
    const DevConsts &c = ctx->hc;
    sv.stiff = 1.0 + c.dampK * c.ngamma / (h * c.nbeta);
    sv.mcoef = (1.0 / (h * h) + c.dampM * c.ngamma / h) / c.nbeta;
    return sv;
}

template <bool MX, bool IS, bool ACC, typename L>
void vals_kernel(icf_ctx *ctx, const char *name, const SlotMap *m, double *A, const Stage &sv)
{
    const int k = sizeof(L) == 4 ? 0 : 1;
    if (m->nlaunch == 0) return;
    const int c = tune_begin(ctx, ACC, k == 1, m->nlaunch);
    with_cand<!ACC>(c, m->nlaunch, [&](auto kc, auto sc) {
        constexpr int K = decltype(kc)::value, S = decltype(sc)::value;
        LAUNCH(ctx, name, (k_reduce_vals<MX, IS, ACC, L, K, S>), dim3(blocks_for(m->nlaunch, K)), dim3(K), m->loff,
               m->codes, m->keys, m->nlaunch, A, sv);
    });
    tune_end(ctx, ACC, k == 1);
}

// Phase 2 of BCSR values for map m.  accumulate: add into A over the keys with contributions
// (single-kernel entry points); otherwise overwrite every block.  contact: the map's units
// are impacts, whose FP64 records are staged as FP64 in both modes.
void launch_vals(icf_ctx *ctx, const SlotMap *m, double *A, int accumulate, const Stage &sv, bool contact = false)
{
    if (m->nlaunch == 0) return;
    const bool mixed = ctx->precision == ICF_MIXED, iso = ctx->hc.iso != 0;
    if (contact) {
        // impact records are FP64; in mixed mode their blocks are staged (and added) as FP32
        // values, like the other tangent blocks of that mode
        if (mixed) vals_kernel<true, false, true, float>(ctx, "k_reduce_vals<contact,mixed,acc>", m, A, sv);
        else vals_kernel<false, false, true, double>(ctx, "k_reduce_vals<contact,fp64,acc>", m, A, sv);
        return;
    }
#define ICF_VALS(MX, IS, L, NAME)                                                                              \
    do {                                                                                                       \
        if (accumulate)                                                                                        \
            vals_kernel<MX, IS, true, L>(ctx, "k_reduce_vals<" NAME ",acc>", m, A, sv);                        \
        else                                                                                                   \
            vals_kernel<MX, IS, false, L>(ctx, "k_reduce_vals<" NAME ">", m, A, sv);                           \
    } while (0)
    if (mixed && iso) ICF_VALS(true, true, float, "mixed,iso");
    else if (mixed) ICF_VALS(true, false, float, "mixed,gen");
    else if (iso) ICF_VALS(false, true, double, "fp64,iso");
    else ICF_VALS(false, false, double, "fp64,gen");
#undef ICF_VALS
}

void launch_vec3(icf_ctx *ctx, const SlotMap *m, double *out, int comp_stride, int elem_stride, int accumulate,
                 const Stage &sv)
{
    const int *keys = m->keys;
    const int n = m->nlaunch;
    if (n == 0) return;
    dim3 g(blocks_for(n, 256)), b(256);
    const bool force = elem_stride == 1;
    if (accumulate)
        LAUNCH(ctx, force ? "k_reduce_vec3<force,acc>" : "k_reduce_vec3<rhs,acc>", k_reduce_vec3<true>, g, b, m->loff,
               m->codes, keys, n, out, comp_stride, elem_stride, sv);
    else
        LAUNCH(ctx, force ? "k_reduce_vec3<force>" : "k_reduce_vec3<rhs>", k_reduce_vec3<false>, g, b, m->loff,
               m->codes, keys, n, out, comp_stride, elem_stride, sv);
}

bool bad_units(int n, int stride) { return n < 0 || stride < 0 || (n > 0 && stride < n); }

}  // namespace

// =================================================================================================
// C ABI
// =================================================================================================
extern "C" {

int icf_create(int device, icf_ctx **out)
{
    if (!out || device < 0 || device >= 64) return ICF_E_INVALID;
    *out = nullptr;
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess) return (int)e;
    if (device >= ndev) return ICF_E_INVALID;
    icf_ctx *ctx = new icf_ctx();
    for (auto &row : ctx->tune) row[1].sel = CAND_FP64;   // FP64 staging roles
    for (auto &t : ctx->tune[0]) t.small_max = VALS_SMALL;
    for (int r = 0; r < NSHAPE; r++) {
        ctx->shape[r].ncand = shape_ncand(r);
        ctx->shape[r].sel = SHAPE_DEFAULT[r];
        ctx->shape[r].untuned = SHAPE_UNTUNED[r];
        ctx->shape[r].small = SHAPE_SMALL[r];
        ctx->shape[r].small_max = SHAPE_SMALL_MAX[r];
    }
    ctx->id = g_next_ctx_id++;
    ctx->device = device;
    memset(&ctx->hc, 0, sizeof(ctx->hc));
    e = hipSetDevice(device);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ctx->ncu, hipDeviceAttributeMultiprocessorCount, device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&ctx->stream_c, hipStreamNonBlocking);
    for (int l = 0; l < 2; l++)
        for (int k = 0; k < LANE_EVENTS && e == hipSuccess; k++)
            e = hipEventCreateWithFlags(&ctx->lane_ev[l][k], hipEventDisableTiming);


    ctx->cur = ctx->stream;
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev0);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev1);
    if (e == hipSuccess) e = hipMalloc(&ctx->small, 16 * sizeof(int));
    const size_t rep_bytes = (REPORT_WORDS + 2 * REPORT_SPECS) * sizeof(unsigned);
    if (e == hipSuccess) e = hipMalloc(&ctx->rep_dev, REPORT_WORDS * sizeof(unsigned));
    if (e == hipSuccess) e = hipMemset(ctx->rep_dev, 0, REPORT_WORDS * sizeof(unsigned));
    if (e == hipSuccess) e = hipHostMalloc((void **)&ctx->rep_host, rep_bytes, hipHostMallocMapped);
    if (e == hipSuccess) memset(ctx->rep_host, 0, rep_bytes);
    if (e == hipSuccess) e = scratch_for_device(device, (void **)&ctx->noalloc);
    if (e != hipSuccess) {
        delete ctx;
        return (int)e;
    }
    *out = ctx;
    return 0;
}

int icf_destroy(icf_ctx *ctx)
{
    if (!ctx) return ICF_E_INVALID;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream_c) (void)hipStreamSynchronize(ctx->stream_c);
    (void)hipStreamSynchronize(ctx->stream);
    for (SlotMap &m : ctx->maps) free_map(m);
    DevBuf *bufs[] = {&ctx->tet_rhs, &ctx->tan, &ctx->cz_rhs, &ctx->ct,   &ctx->scan_tmp,
                      &ctx->pat_a,   &ctx->pat_b,   &ctx->bp_f,   &ctx->bp_i, &ctx->bp_l, &ctx->bp_c,
                      &ctx->tsum,    &ctx->ct_f,    &ctx->adj.off, &ctx->adj.ids, &ctx->batch.d,
                      &ctx->patc.snap, &ctx->patc.rows, &ctx->patc.cols, &ctx->pat_cnt, &ctx->bp_g, &ctx->map_cnt, &ctx->map_rank, &ctx->map_sums};
    for (DevBuf *b : bufs)
        if (b->p) (void)hipFree(b->p);
    if (ctx->small) (void)hipFree(ctx->small);
    if (ctx->rep_dev) (void)hipFree(ctx->rep_dev);
    if (ctx->rep_host) (void)hipHostFree(ctx->rep_host);
    (void)hipEventDestroy(ctx->ev0);
    (void)hipEventDestroy(ctx->ev1);
    for (auto &p : ctx->pending) {
        ctx->ev_pool.push_back(p.a);
        ctx->ev_pool.push_back(p.b);
    }
    for (hipEvent_t e : ctx->ev_pool) (void)hipEventDestroy(e);
    for (auto &row : ctx->tune)
        for (auto &t : row)
            for (hipEvent_t e : t.ev)
                if (e) (void)hipEventDestroy(e);
    for (auto &t : ctx->shape)
        for (hipEvent_t e : t.ev)
            if (e) (void)hipEventDestroy(e);
    for (int l = 0; l < 2; l++)
        for (int k = 0; k < LANE_EVENTS; k++)
            if (ctx->lane_ev[l][k]) (void)hipEventDestroy(ctx->lane_ev[l][k]);
    if (ctx->stream_c) (void)hipStreamDestroy(ctx->stream_c);
    (void)hipStreamDestroy(ctx->stream);
    {
        std::lock_guard<std::mutex> lk(g_dev_mu[ctx->device]);
        if (g_const_owner[ctx->device] == ctx->id) g_const_owner[ctx->device] = 0;
    }
    delete ctx;
    return 0;
}

const char *icf_last_error_string(const icf_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int icf_set_constants(icf_ctx *ctx, const icf_consts *c)
{
    if (!ctx || !c) return ICF_E_INVALID;
    // E symmetric
    for (int i = 0; i < 6; i++)
        for (int j = 0; j < 6; j++)
            if (c->E[i * 6 + j] != c->E[j * 6 + i]) return fail(ctx, ICF_E_CONSTANTS, "E is not symmetric");
    // B must be [s (x) I3, -s (x) I3] built from sf (ModelPrms.k_Bmatrix)
    for (int gp = 0; gp < 3; gp++)
        for (int p = 0; p < 3; p++)
            for (int k = 0; k < 18; k++) {
                int node = k / 3;
                double want = 0;
                if (k % 3 == p) want = node < 3 ? c->sf[node * 3 + gp] : -c->sf[(node - 3) * 3 + gp];
                if (c->B[gp * 54 + p * 18 + k] != want)
                    return fail(ctx, ICF_E_CONSTANTS, "CZ B table is not the shape-function Kronecker form");
            }
    DevConsts &d = ctx->hc;
    memset(&d, 0, sizeof(d));
    memcpy(d.E, c->E, sizeof(d.E));
    memcpy(d.M, c->M, sizeof(d.M));
    d.nbeta = c->NewmarkBeta; d.ngamma = c->NewmarkGamma;
    d.dampM = c->dampingMass; d.dampK = c->dampingStiffness;
    d.rho = c->rho; d.grav = c->gravity;
    d.G_fn = c->G_fn; d.G_ft = c->G_ft; d.f_tn = c->f_tn; d.f_tt = c->f_tt;
    d.alpha = c->alpha; d.beta = c->beta; d.rn = c->rn; d.rt = c->rt;
    d.p_m = c->p_m; d.p_n = c->p_n; d.deln = c->deln; d.delt = c->delt;
    d.pMtn = c->pMtn; d.pMnt = c->pMnt; d.gam_n = c->gam_n; d.gam_t = c->gam_t;
    memcpy(d.sf, c->sf, sizeof(d.sf));
    // isotropic split: E = lam 1 1^T (normal block) + diag(2mu,2mu,2mu,mu,mu,mu)
    {
        double lam = c->E[1], mu = c->E[3 * 6 + 3], dg = c->E[0];
        bool iso = mu > 0;
        for (int i = 0; i < 6 && iso; i++)
            for (int j = 0; j < 6 && iso; j++) {
                double v = c->E[i * 6 + j];
                if (i < 3 && j < 3) iso = (i == j) ? (v == dg) : (v == lam);
                else if (i == j) iso = (v == mu);
                else iso = (v == 0);
            }
        if (iso) iso = fabs(dg - (lam + 2 * mu)) <= 1e-12 * fabs(dg);
        // the isotropic path also takes the mass as m_ij I3 per node pair (ModelPrms.cs:239-248
        // builds it so); any other M takes the general path
        for (int i = 0; i < 4; i++)
            for (int j = 0; j < 4; j++) {
                const double mij = c->M[(3 * i) * 12 + 3 * j];
                d.m4[4 * i + j] = mij;
                d.m4f[4 * i + j] = (float)mij;
                for (int k = 0; k < 3 && iso; k++)
                    for (int l = 0; l < 3 && iso; l++)
                        iso = c->M[(3 * i + k) * 12 + 3 * j + l] == (k == l ? mij : 0.0);
            }
        d.iso = iso ? 1 : 0;
        d.m_two = 1;
        d.m_ii = d.m4[0];
        d.m_ij = d.m4[1];
        d.m_iif = d.m4f[0];
        d.m_ijf = d.m4f[1];
        for (int k = 0; k < 16; k++) d.m_two = d.m_two && d.m4[k] == (k / 4 == k % 4 ? d.m_ii : d.m_ij);
        d.lam = lam;
        d.mu = mu;
        d.lamf = (float)lam;
        d.muf = (float)mu;
    }
    auto small_int = [](double v) { return v >= 2 && v <= 16 && v == (double)(int)v ? (int)v : 0; };
    d.alpha_n = small_int(c->alpha);
    d.beta_n = small_int(c->beta);
    d.k_tn = c->gam_n / c->deln;
    d.k_tt = c->gam_t / c->delt;
    d.k_dnn = c->gam_n / (c->deln * c->deln);
    d.k_dtt = c->gam_t / (c->delt * c->delt);
    d.k_dnt = c->gam_n * c->gam_t / (c->deln * c->delt);
    d.pm_alpha = c->p_m / c->alpha;
    d.pn_beta = c->p_n / c->beta;
    d.thr_n = c->f_tn * 0.05;
    d.thr_t = c->f_tt * 0.05;
    d.lim_n = c->deln * c->rn / 5;
    d.lim_t = c->delt * c->rt / 5;
    for (int e = 0; e < 3; e++) {
        d.bn0[e] = pow(c->p_m / c->alpha, c->p_m - e);
        d.bt0[e] = pow(c->p_n / c->beta, c->p_n - e);
    }
    for (int i = 0; i < 36; i++) d.Ef[i] = (float)d.E[i];
    for (int i = 0; i < 144; i++) d.Mf[i] = (float)d.M[i];
    ctx->has_consts = true;
    ctx->consts_dirty = true;
    if (int r = check_ctx(ctx)) return r;
    ConstUse cu(ctx);
    return cu.err;
}

int icf_set_precision(icf_ctx *ctx, int mode)
{
    if (!ctx || (mode != ICF_FP64 && mode != ICF_MIXED)) return ICF_E_INVALID;
    ctx->precision = mode;
    return 0;
}

int icf_get_precision(const icf_ctx *ctx) { return ctx ? ctx->precision : ICF_E_INVALID; }

int icf_alloc(icf_ctx *ctx, size_t bytes, void **dptr)
{
    if (!ctx || !dptr) return ICF_E_INVALID;
    if (int r = check_ctx(ctx)) return r;
    *dptr = nullptr;
    HIPCHK(ctx, hipMalloc(dptr, bytes ? bytes : 1));
    return 0;
}

int icf_free(icf_ctx *ctx, void *dptr)
{
    if (!ctx) return ICF_E_INVALID;
    if (!dptr) return 0;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_free during capture");
    if (int r = check_ctx(ctx)) return r;
    if (int r = sync_lanes(ctx)) return r;
    size_t sz = 0;
    void *basep = nullptr;
    if (hipMemGetAddressRange(&basep, &sz, dptr) == hipSuccess && sz)
        invalidate_range(ctx, (uintptr_t)basep, (uintptr_t)basep + sz, true);
    else
        invalidate_range(ctx, (uintptr_t)dptr, (uintptr_t)dptr + 1, true);
    HIPCHK(ctx, hipFree(dptr));
    return 0;
}

int icf_h2d(icf_ctx *ctx, void *dst, size_t dst_off, const void *src, size_t bytes)
{
    if (!ctx || (!dst && bytes) || (!src && bytes)) return ICF_E_INVALID;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "host copies cannot be captured");
    if (int r = check_ctx(ctx)) return r;
    if (!bytes) return 0;
    char *d = (char *)dst + dst_off;
    invalidate_range(ctx, (uintptr_t)d, (uintptr_t)d + bytes);
    if (int r = lane_barrier(ctx)) return r;
    HIPCHK(ctx, hipMemcpyAsync(d, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

int icf_d2h(icf_ctx *ctx, void *dst, const void *src, size_t src_off, size_t bytes)
{
    if (!ctx || (!dst && bytes) || (!src && bytes)) return ICF_E_INVALID;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "host copies cannot be captured");
    if (int r = check_ctx(ctx)) return r;
    if (!bytes) return 0;
    if (int r = lane_barrier(ctx)) return r;
    HIPCHK(ctx, hipMemcpyAsync(dst, (const char *)src + src_off, bytes, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

int icf_memset(icf_ctx *ctx, void *dst, int value, size_t bytes)
{
    if (!ctx || (!dst && bytes)) return ICF_E_INVALID;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_memset during capture (clear buffers with a kernel)");
    if (int r = check_ctx(ctx)) return r;
    if (!bytes) return 0;
    invalidate_range(ctx, (uintptr_t)dst, (uintptr_t)dst + bytes);
    if (int r = lane_barrier(ctx)) return r;
    HIPCHK(ctx, hipMemsetAsync(dst, value, bytes, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

int icf_synchronize(icf_ctx *ctx)
{
    if (int r = check_ctx(ctx)) return r;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_synchronize during capture");
    if (int r = sync_lanes(ctx)) return r;
    prof_flush(ctx);
    return 0;
}

int icf_pattern_changed(icf_ctx *ctx)
{
    if (int r = check_ctx(ctx)) return r;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_pattern_changed during capture");
    for (SlotMap &m : ctx->maps) m.suspect = true;
    ctx->adj.valid = false;
    ctx->patc.valid = false;
    bump(ctx);
    return 0;
}

double icf_last_device_ms(const icf_ctx *ctx) { return ctx ? ctx->last_ms : -1; }

int icf_d2d(icf_ctx *ctx, void *dst, size_t dst_off, const void *src, size_t src_off, size_t bytes)
{
    if (!ctx || (!dst && bytes) || (!src && bytes)) return ICF_E_INVALID;
    if (int r = check_ctx(ctx)) return r;
    if (!bytes) return 0;
    char *d = (char *)dst + dst_off;
    if (int r = note_write(ctx, d, bytes, "icf_d2d")) return r;
    OnLane ln(ctx, 0, [&] { return Access().rd((const char *)src + src_off, bytes).wr(d, bytes); });
    if (ln.err) return ln.err;
    Timer tm(ctx);
    LAUNCH(ctx, "k_copy", k_copy, dim3(blocks_for((long long)((bytes + 15) / 16), 256)), dim3(256), d,
           (const char *)src + src_off, bytes);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_probe_valu(icf_ctx *ctx, int fp64, int workgroups, int iters, void *out)
{
    if (!ctx || !out || workgroups <= 0 || iters <= 0) return ICF_E_INVALID;
    if (int r = check_ctx(ctx)) return r;
    const size_t bytes = (size_t)workgroups * 256 * (fp64 ? 8 : 4);
    if (int r = note_write(ctx, out, bytes, "icf_probe_valu")) return r;
    OnLane ln(ctx, 0, [&] { return Access().wr((const char *)out, bytes); });
    if (ln.err) return ln.err;
    Timer tm(ctx);
    // m slightly below one and c small keep every chain finite for any iteration count
    if (fp64)
        LAUNCH(ctx, "k_valu_probe<double>", k_valu_probe<double>, dim3(workgroups), dim3(256), (double *)out, iters,
               0.999999, 1e-6);
    else
        LAUNCH(ctx, "k_valu_probe<float>", k_valu_probe<float>, dim3(workgroups), dim3(256), (float *)out, iters,
               0.9999f, 1e-4f);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_set_blocking(icf_ctx *ctx, int blocking)
{
    if (!ctx) return ICF_E_INVALID;
    ctx->blocking = blocking != 0;
    return 0;
}

int icf_cz_counts(icf_ctx *ctx, int *nCZDamaged, int *nCZFailed)
{
    if (int r = check_ctx(ctx)) return r;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_cz_counts during capture");
    if (int r = lane_barrier(ctx)) return r;
    int sums[2] = {0, 0};
    HIPCHK(ctx, hipMemcpyAsync(sums, ctx->small + 2, 2 * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    if (nCZDamaged) *nCZDamaged = sums[0];
    if (nCZFailed) *nCZFailed = sums[1];
    return 0;
}

struct icf_graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int device = 0;
    int ctx_id = 0;                  // the context that captured it ...
    unsigned long long epoch = 0;    // ... and its epoch at icf_graph_end
};

int icf_graph_begin(icf_ctx *ctx)
{
    if (int r = check_ctx(ctx)) return r;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "capture already in progress");
    if (int r = sync_lanes(ctx)) return r;
    prof_flush(ctx);
    HIPCHK(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    ctx->capturing = true;
    return 0;
}

int icf_graph_end(icf_ctx *ctx, icf_graph **out)
{
    if (!ctx || !out) return ICF_E_INVALID;
    if (!ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "no capture in progress");
    *out = nullptr;
    ctx->capturing = false;
    hipGraph_t g = nullptr;
    HIPCHK(ctx, hipStreamEndCapture(ctx->stream, &g));
    hipGraphExec_t ex = nullptr;
    hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        return fail(ctx, (int)e, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    }
    icf_graph *gr = new icf_graph();
    gr->graph = g;
    gr->exec = ex;
    gr->device = ctx->device;
    gr->ctx_id = ctx->id;
    gr->epoch = ctx->epoch;
    *out = gr;
    return 0;
}

int icf_graph_launch(icf_ctx *ctx, icf_graph *g)
{
    if (int r = check_ctx(ctx)) return r;
    if (!g || g->device != ctx->device) return fail(ctx, ICF_E_INVALID, "icf_graph_launch: bad graph");
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_graph_launch during capture");
    if (g->ctx_id != ctx->id)
        return fail(ctx, ICF_E_CAPTURE, "icf_graph_launch: the graph was captured on another context");
    if (g->epoch != ctx->epoch)
        return fail(ctx, ICF_E_CAPTURE,
                    "icf_graph_launch: the graph is stale (since its capture, memory it uses was freed or moved, or "
                    "slot fields it was built from were written): capture it again");
    ConstUse cu(ctx);
    if (cu.err) return cu.err;
    OnLane ln(ctx, 0, everything);
    if (ln.err) return ln.err;
    Timer tm(ctx);
    HIPCHK(ctx, hipGraphLaunch(g->exec, ctx->stream));
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_graph_destroy(icf_graph *g)
{
    if (!g) return ICF_E_INVALID;
    (void)hipSetDevice(g->device);
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    delete g;
    return 0;
}

int icf_set_profiling(icf_ctx *ctx, int on)
{
    if (!ctx) return ICF_E_INVALID;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_set_profiling during capture");
    ctx->profiling = on != 0;
    return 0;
}

int icf_set_overlap(icf_ctx *ctx, int on)
{
    if (!ctx) return ICF_E_INVALID;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_set_overlap during capture");
    ctx->overlap = on != 0;
    return 0;
}

int icf_set_autotune(icf_ctx *ctx, int rounds)
{
    if (!ctx || rounds < 0 || rounds > 1000) return ICF_E_INVALID;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_set_autotune during capture");
    if (int r = check_ctx(ctx)) return r;
    std::vector<std::pair<icf_ctx::Tune *, int>> all;
    for (int a = 0; a < 2; a++)
        for (int f = 0; f < 2; f++) all.push_back({&ctx->tune[a][f], 2 * a + f});
    for (int r = 0; r < NSHAPE; r++) all.push_back({&ctx->shape[r], 4 + r});
    for (auto &tr : all) {
        icf_ctx::Tune &t = *tr.first;
        if (rounds == 0) {             // stop: fold what was timed, keep the fastest so far
            if (t.active) {
                t.tuned = true;
                tune_fold(ctx, t, tr.second);
                for (int c = 0; c < t.ncand; c++)
                    if (t.best[c] > 0 && (t.best[t.sel] == 0 || t.best[c] < t.best[t.sel])) t.sel = c;
            }
            t.active = false;
            continue;
        }
        for (hipEvent_t &e : t.ev)
            if (!e) HIPCHK(ctx, hipEventCreate(&e));
        t.active = true;
        t.fixed = false;
        t.turn = t.samples = 0;
        t.cand = -1;
        t.bucket = -1;
        for (float &b : t.best) b = 0;
    }
    ctx->tune_rounds = rounds;
    return 0;
}

int icf_get_autotune(icf_ctx *ctx, int *keys, int *stage, int *tuning, float *best_ms)
{
    if (!ctx) return ICF_E_INVALID;
    for (int r = 0; r < 4; r++) {
        icf_ctx::Tune &t = ctx->tune[r >> 1][r & 1];
        if (t.active && !ctx->capturing) tune_fold(ctx, t, r);   // a finished last timing counts
        if (keys) keys[r] = cand_keys(t.in_use());
        if (stage) stage[r] = cand_stage(t.in_use());
        if (tuning) tuning[r] = t.active ? 1 : 0;
        if (best_ms)
            for (int c = 0; c < NCAND; c++) best_ms[r * NCAND + c] = t.best[c];
    }
    return 0;
}

int icf_set_chunk_keys(icf_ctx *ctx, int accumulate, int fp64, int keys, int stage)
{
    if (!ctx) return ICF_E_INVALID;
    icf_ctx::Tune &t = ctx->tune[accumulate != 0][fp64 != 0];
    if (stage == 0) stage = cand_stage(t.in_use());
    int c = 0;
    while (c < NCAND && (cand_keys(c) != keys || cand_stage(c) != stage)) c++;
    if (c == NCAND)
        return fail(ctx, ICF_E_INVALID, "icf_set_chunk_keys: keys must be 64, 128, 256 or 512 and stage 2 or 3");
    if (t.active && !ctx->capturing) tune_fold(ctx, t, 2 * (accumulate != 0) + (fp64 != 0));
    t.active = false;
    t.fixed = true;
    t.cand = -1;
    t.sel = c;
    return 0;
}

int icf_set_shape(icf_ctx *ctx, int role, int value)
{
    if (!ctx) return ICF_E_INVALID;
    if (role < 0 || role >= NSHAPE) return fail(ctx, ICF_E_INVALID, "icf_set_shape: unknown role");
    int c = 0;
    while (c < shape_ncand(role) && shape_value(role, c) != value) c++;
    if (c == shape_ncand(role))
        return fail(ctx, ICF_E_INVALID, role == ICF_SHAPE_CLOSEST ? "icf_set_shape: lanes per tuple must be 4, 8 or 16"
                                        : role == ICF_SHAPE_ORDER ? "icf_set_shape: the order must be 0 or 1"
                                                                  : "icf_set_shape: workgroup size must be 64, 128 or 256");
    icf_ctx::Tune &t = ctx->shape[role];
    if (t.active && !ctx->capturing) tune_fold(ctx, t, 4 + role);
    t.active = false;
    t.fixed = true;
    t.cand = -1;
    t.sel = c;
    return 0;
}

int icf_get_shape(icf_ctx *ctx, int role, int *value, int *tuning, float *best_ms)
{
    if (!ctx) return ICF_E_INVALID;
    if (role < 0 || role >= NSHAPE) return fail(ctx, ICF_E_INVALID, "icf_get_shape: unknown role");
    icf_ctx::Tune &t = ctx->shape[role];
    if (t.active && !ctx->capturing) tune_fold(ctx, t, 4 + role);
    if (value) *value = shape_value(role, t.in_use());
    if (tuning) *tuning = t.active ? 1 : 0;
    if (best_ms)
        for (int c = 0; c < NSHAPE_CAND; c++) best_ms[c] = c < t.ncand ? t.best[c] : 0.f;
    return 0;
}

int icf_profile_reset(icf_ctx *ctx)
{
    if (!ctx) return ICF_E_INVALID;
    ctx->prof_names.clear();
    ctx->prof_ms.clear();
    ctx->prof_n.clear();
    return 0;
}

int icf_profile_count(const icf_ctx *ctx) { return ctx ? (int)ctx->prof_names.size() : ICF_E_INVALID; }

int icf_profile_entry(const icf_ctx *ctx, int i, char *name, int cap, double *total_ms, long long *launches)
{
    if (!ctx || i < 0 || i >= (int)ctx->prof_names.size()) return ICF_E_INVALID;
    if (name && cap > 0) {
        strncpy(name, ctx->prof_names[i].c_str(), (size_t)cap - 1);
        name[cap - 1] = 0;
    }
    if (total_ms) *total_ms = ctx->prof_ms[i];
    if (launches) *launches = ctx->prof_n[i];
    return 0;
}

int icf_elem_force(icf_ctx *ctx, const int *ie, double *dn, double h, double *A, double *b, int nElems, int el_stride,
                   int nd_stride)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nElems, el_stride) || nd_stride < 0 || (nElems && (!ie || !dn || !A || !b)) || !(h > 0))
        return fail(ctx, ICF_E_INVALID, "icf_elem_force: invalid argument");
    ConstUse cu(ctx);
    if (cu.err) return cu.err;
    if (nElems == 0) return 0;
    OnLane ln(ctx, 0, everything);
    if (ln.err) return ln.err;
    std::vector<MapReq> req{{TGT_VALS, -1, {{KIND_TET, ie, nElems, el_stride, EL_SLOTS, 16}}},
                            {TGT_RHS, -1, {{KIND_TET, ie, nElems, el_stride, EL_ROWS, 4}}},
                            {TGT_FORCE, -1, {{KIND_TET, ie, nElems, el_stride, EL_NODES, 4}}}};
    if (int r = get_maps(ctx, req)) return r;
    SlotMap *mv = req[0].map, *mr = req[1].map, *mf = req[2].map;
    if (int r = reserve_stage(ctx, nElems, 0)) return r;
    Timer tm(ctx);
    stage_tets(ctx, ie, dn, nElems, el_stride, nd_stride);
    Stage st = make_stage(ctx, h);
    launch_vec3(ctx, mf, dn + (size_t)nd_stride * ND_F, nd_stride, 1, 1, st);
    launch_vals(ctx, mv, A, 1, st);
    launch_vec3(ctx, mr, b, 1, 3, 1, st);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_cz_force(icf_ctx *ctx, double *dcz, int *icz, double *dn, double *A, double *b, double h, int nCZs,
                 int cz_stride, int nd_stride)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nCZs, cz_stride) || nd_stride < 0 || (nCZs && (!dcz || !icz || !dn || !A || !b)))
        return fail(ctx, ICF_E_INVALID, "icf_cz_force: invalid argument");
    ConstUse cu(ctx);
    if (cu.err) return cu.err;
    if (nCZs == 0) return 0;
    OnLane ln(ctx, 0, everything);
    if (ln.err) return ln.err;
    std::vector<MapReq> req{{TGT_VALS, -1, {{KIND_CZ, icz, nCZs, cz_stride, CZI_SLOTS, 36}}},
                            {TGT_RHS, -1, {{KIND_CZ, icz, nCZs, cz_stride, CZI_ROWS, 6}}}};
    if (int r = get_maps(ctx, req)) return r;
    SlotMap *mv = req[0].map, *mr = req[1].map;
    if (int r = reserve_stage(ctx, 0, nCZs)) return r;
    Timer tm(ctx);
    stage_czs(ctx, dcz, icz, dn, nCZs, cz_stride, nd_stride);
    Stage st = make_stage(ctx, h);
    launch_vals(ctx, mv, A, 1, st);
    launch_vec3(ctx, mr, b, 1, 3, 1, st);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_narrow_phase(icf_ctx *ctx, int nPairs, const double *dn, const int *ie, int *narrowList, int el_all_stride,
                     int nd_stride)
{
    if (int r = check_ctx(ctx)) return r;
    if (nPairs < 0 || el_all_stride < 0 || nd_stride < 0 || (nPairs && (!dn || !ie || !narrowList)))
        return fail(ctx, ICF_E_INVALID, "icf_narrow_phase: invalid argument");
    if (nPairs == 0) return 0;
    if (int r = note_write(ctx, narrowList, sizeof(int) * 2 * (size_t)nPairs, "icf_narrow_phase")) return r;
    // reads node positions and the tets' node ids, rewrites the list
    OnLane ln(ctx, contact_lane(ctx), [&] {
        return Access()
            .rd(dn + (size_t)nd_stride * ND_XC, 3 * (size_t)nd_stride)
            .rd(ie, 4 * (size_t)el_all_stride)
            .wr(narrowList, 2 * (size_t)nPairs);
    });
    if (ln.err) return ln.err;
    Timer tm(ctx);
    const int B = shape_begin(ctx, ICF_SHAPE_NARROW, nPairs);
    LAUNCH(ctx, "k_narrow_phase", k_narrow_phase, dim3(blocks_for(nPairs, B)), dim3(B), nPairs, dn, ie,
           narrowList, el_all_stride, nd_stride);
    shape_end(ctx, ICF_SHAPE_NARROW);
    if (int r = ln.done()) return r;
    return tm.finish();
}

// The compact adjacency lists of ie (valid on return), built synchronously when missing.
int get_adjacency(icf_ctx *ctx, const int *ie, int es)
{
    icf_ctx::Adj &a = ctx->adj;
    if (a.valid && a.ie == ie && a.es == es) return 0;
    if (ctx->capturing)
        return fail(ctx, ICF_E_CAPTURE, "the adjacency lists must be built: run the call once uncaptured");
    void *base = nullptr;
    size_t sz = 0;
    HIPCHK(ctx, hipMemGetAddressRange(&base, &sz, const_cast<int *>(ie)));
    const uintptr_t end = (uintptr_t)base + sz;
    const long long rows = ((long long)(end - (uintptr_t)ie)) / (4LL * std::max(es, 1));
    if (rows < 5) return fail(ctx, ICF_E_INVALID, "icf_find_closest_face: ie holds fewer than 5 rows");
    const int max_rows = (int)std::min(rows - 5, 1LL << 20);
    if (int r = lane_barrier(ctx)) return r;
    if (int r = grow(ctx, a.off, sizeof(int) * ((size_t)es + 1))) return r;
    int *off = (int *)a.off.p;
    size_t tb = 0;
    HIPCHK(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, tb, off, off, es + 1, ctx->stream));
    if (int r = grow(ctx, ctx->scan_tmp, tb)) return r;
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, ctx->stream, off + es, 1, 0);
    hipLaunchKernelGGL(k_adj_count, dim3(blocks_for(es, 256)), dim3(256), 0, ctx->stream, ie, es, max_rows, off);
    HIPCHK(ctx, hipcub::DeviceScan::ExclusiveSum(ctx->scan_tmp.p, tb, off, off, es + 1, ctx->stream));
    int total = 0;
    HIPCHK(ctx, hipMemcpyAsync(&total, off + es, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    if (int r = grow(ctx, a.ids, sizeof(int) * (size_t)std::max(total, 1))) return r;
    hipLaunchKernelGGL(k_adj_fill, dim3(blocks_for(es, 256)), dim3(256), 0, ctx->stream, ie, es, off, (int *)a.ids.p);
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    a.ie = ie;
    a.es = es;
    a.lo = (uintptr_t)base;
    a.hi = end;
    a.valid = true;
    return 0;
}

// k_closest_face with the tuned lanes per tuple, on `stream` (the profiled launch when it is
// the context's current stream)
void launch_closest_face(icf_ctx *ctx, int nPairs, int ts, int *nl2, const double *dn, const int *adj_off,
                         const int *adj_ids, const int *faces, int ns, int fs, hipStream_t stream)
{
    const bool timed = stream == ctx->cur;   // tuning times launches on the current stream only
    int G = shape_begin(ctx, ICF_SHAPE_CLOSEST, nPairs, !timed);
    if (G == 8 && nPairs <= CLOSEST_SMALL) G = 16;
    const dim3 g(blocks_for((long long)nPairs * G, 256)), b(256);
    auto go = [&](auto kern) {
        if (stream == ctx->cur) LAUNCH(ctx, "k_closest_face", kern, g, b, nPairs, ts, nl2, dn, adj_off, adj_ids, faces, ns, fs);
        else hipLaunchKernelGGL(kern, g, b, 0, stream, nPairs, ts, nl2, dn, adj_off, adj_ids, faces, ns, fs);
    };
    if (G == 4) go(k_closest_face<4>);
    else if (G == 16) go(k_closest_face<16>);
    else go(k_closest_face<8>);
    if (timed) shape_end(ctx, ICF_SHAPE_CLOSEST);
}

int icf_find_closest_face(icf_ctx *ctx, int nPairs, int tet_stride, int *nl2, const double *dn, const int *ie,
                          const int *faces, int nd_stride, int el_all_stride, int fc_stride)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nPairs, tet_stride) || nd_stride < 0 || el_all_stride < 0 || fc_stride < 0 ||
        (nPairs && (!nl2 || !dn || !ie || !faces)))
        return fail(ctx, ICF_E_INVALID, "icf_find_closest_face: invalid argument");
    if (nPairs == 0) return 0;
    if (int r = note_write(ctx, nl2 + tet_stride, sizeof(int) * 3 * (size_t)tet_stride, "icf_find_closest_face"))
        return r;
    // the surface tets' adjacency lists, read from their compact copy
    if (int r = get_adjacency(ctx, ie, el_all_stride)) return r;
    OnLane ln(ctx, contact_lane(ctx), [&] {
        return Access()
            .wr(nl2, 4 * (size_t)tet_stride)
            .rd(dn + (size_t)nd_stride * ND_XC, 3 * (size_t)nd_stride)
            .rd((const char *)ctx->adj.off.p, ctx->adj.off.bytes)
            .rd((const char *)ctx->adj.ids.p, ctx->adj.ids.bytes)
            .rd(faces, 3 * (size_t)fc_stride);
    });
    if (ln.err) return ln.err;
    Timer tm(ctx);
    launch_closest_face(ctx, nPairs, tet_stride, nl2, dn, (const int *)ctx->adj.off.p, (const int *)ctx->adj.ids.p,
                        faces, nd_stride, fc_stride, ctx->cur);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_find_closest_face_noalloc(icf_ctx *ctx, int nPairs, int tet_stride, int *nl2, const double *dn,
                                  const int *ie, const int *faces, int nd_stride, int el_all_stride, int fc_stride)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nPairs, tet_stride) || nd_stride < 0 || el_all_stride < 0 || fc_stride < 0 ||
        (nPairs && (!nl2 || !dn || !ie || !faces)))
        return fail(ctx, ICF_E_INVALID, "icf_find_closest_face_noalloc: invalid argument");
    if (nPairs == 0) return 0;
    if (!ctx->noalloc) return fail(ctx, ICF_E_INVALID, "icf_find_closest_face_noalloc: no scratch on this device");
    if (int r = note_write(ctx, nl2 + tet_stride, sizeof(int) * 3 * (size_t)tet_stride,
                           "icf_find_closest_face_noalloc"))
        return r;
    const int es = el_all_stride;
    // adjacent-face rows of ie, from the extent of its allocation (as icf_find_closest_face)
    void *base = nullptr;
    size_t sz = 0;
    HIPCHK(ctx, hipMemGetAddressRange(&base, &sz, const_cast<int *>(ie)));
    const long long rows = ((long long)((uintptr_t)base + sz - (uintptr_t)ie)) / (4LL * std::max(es, 1));
    if (rows < 5) return fail(ctx, ICF_E_INVALID, "icf_find_closest_face_noalloc: ie holds fewer than 5 rows");
    const int max_rows = (int)std::min(rows - 5, 1LL << 20);
    // scratch layout: list offsets [es + 1], the scan's temporary storage, the lists (at most
    // max_rows faces per tet: k_adj_count clamps the counts)
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    size_t tb = 0;
    HIPCHK(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (int *)nullptr, (int *)nullptr, es + 1, ctx->stream));
    const size_t tmp_at = up(sizeof(int) * ((size_t)es + 1)), ids_at = tmp_at + up(tb);
    const size_t need = ids_at + sizeof(int) * (size_t)es * (size_t)std::max(max_rows, 1);
    if (need > NOALLOC_SCRATCH_BYTES)
        return fail(ctx, ICF_E_CAPACITY, "icf_find_closest_face_noalloc: el_all_stride " + std::to_string(es) +
                                             " x " + std::to_string(max_rows) + " adjacent-face rows need " +
                                             std::to_string(need) + " bytes of scratch, more than its " +
                                             std::to_string(NOALLOC_SCRATCH_BYTES) + "; use icf_find_closest_face");
    int *off = (int *)ctx->noalloc;
    void *tmp = ctx->noalloc + tmp_at;
    int *ids = (int *)(ctx->noalloc + ids_at);
    // after every earlier call of the context, on its stream; later calls of either lane wait
    if (int r = lane_barrier(ctx)) return r;
    Timer tm(ctx);
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, ctx->stream, off + es, 1, 0);
    hipLaunchKernelGGL(k_adj_count, dim3(blocks_for(es, 256)), dim3(256), 0, ctx->stream, ie, es, max_rows, off);
    HIPCHK(ctx, hipcub::DeviceScan::ExclusiveSum(tmp, tb, off, off, es + 1, ctx->stream));
    hipLaunchKernelGGL(k_adj_fill, dim3(blocks_for(es, 256)), dim3(256), 0, ctx->stream, ie, es, (const int *)off,
                       ids);
    launch_closest_face(ctx, nPairs, tet_stride, nl2, dn, (const int *)off, (const int *)ids, faces, nd_stride,
                        fc_stride, ctx->stream);
    if (int r = lane_exit(ctx, 0, everything)) return r;
    return tm.finish();
}

int icf_collision_response(icf_ctx *ctx, const int *icr, double *dn, double h, double *A, double *b, int nImpacts,
                           int cr_stride, int nd_stride, double k, double distanceEpsilon)
{
    (void)h;
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nImpacts, cr_stride) || nd_stride < 0 || (nImpacts && (!icr || !dn || !A || !b)))
        return fail(ctx, ICF_E_INVALID, "icf_collision_response: invalid argument");
    if (nImpacts == 0) return 0;
    std::vector<MapReq> req{{TGT_VALS, -1, {{KIND_CONTACT, icr, nImpacts, cr_stride, CR_SLOTS, 16}}},
                            {TGT_RHS, -1, {{KIND_CONTACT, icr, nImpacts, cr_stride, CR_ROWS, 4}}},
                            {TGT_FORCE, -1, {{KIND_CONTACT, icr, nImpacts, cr_stride, CR_NODES, 4}}}};
    if (int r = get_maps(ctx, req)) return r;
    SlotMap *mv = req[0].map, *mr = req[1].map, *mf = req[2].map;
    const bool mixed = ctx->precision == ICF_MIXED;
    if (int r = grow(ctx, ctx->ct, (mixed ? sizeof(float) : sizeof(double)) * CT_TAN_REC * (size_t)nImpacts)) return r;
    if (int r = grow(ctx, ctx->ct_f, sizeof(double) * CT_F_REC * (size_t)nImpacts)) return r;
    Timer tm(ctx);
    const size_t tan_bytes = (mixed ? sizeof(float) : sizeof(double)) * CT_TAN_REC * (size_t)nImpacts;
    const size_t f_bytes = sizeof(double) * CT_F_REC * (size_t)nImpacts;
    // per-impact phase: node positions and the impact records in, impact blocks out
    OnLane l1(ctx, contact_lane(ctx), [&] {
        return Access()
            .rd(icr, (CR_ROWS + 4) * (size_t)cr_stride)
            .rd(dn + (size_t)nd_stride * ND_XC, 3 * (size_t)nd_stride)
            .wr((const char *)ctx->ct.p, tan_bytes)
            .wr((const char *)ctx->ct_f.p, f_bytes);
    });
    if (l1.err) return l1.err;
    const int B = shape_begin(ctx, ICF_SHAPE_IMPACT, nImpacts);
    const dim3 cg(blocks_for(nImpacts, B)), cb(B);
    if (mixed)
        LAUNCH(ctx, "k_contact_impact<mixed>", k_contact_impact<float>, cg, cb, icr, dn, nImpacts, cr_stride, nd_stride,
               k, distanceEpsilon, (float *)ctx->ct.p, (double *)ctx->ct_f.p);
    else
        LAUNCH(ctx, "k_contact_impact<fp64>", k_contact_impact<double>, cg, cb, icr, dn, nImpacts, cr_stride,
               nd_stride, k, distanceEpsilon, (double *)ctx->ct.p, (double *)ctx->ct_f.p);
    shape_end(ctx, ICF_SHAPE_IMPACT);
    if (int r = l1.done()) return r;
    // sums into node forces, BCSR blocks (at slots the call does not bound) and rhs rows
    OnLane l0(ctx, 0, [&] {
        return Access()
            .rd((const char *)ctx->ct.p, tan_bytes)
            .rd((const char *)ctx->ct_f.p, f_bytes)
            .rd(icr, (CR_ROWS + 4) * (size_t)cr_stride)
            .wr(dn + (size_t)nd_stride * ND_F, 3 * (size_t)nd_stride)
            .alloc(A, true)
            .alloc(b, true);
    });
    if (l0.err) return l0.err;
    Stage st = make_stage(ctx, 1.0);
    double *F = dn + (size_t)nd_stride * ND_F;
    if (!(ctx->overlap && contact_sums_fused(ctx, mf, F, nd_stride, mv, A, mr, b, st))) {
        launch_vec3(ctx, mf, F, nd_stride, 1, 1, st);
        launch_vals(ctx, mv, A, 1, st, true);
        launch_vec3(ctx, mr, b, 1, 3, 1, st);
    }
    if (int r = l0.done()) return r;
    return tm.finish();
}

int icf_sum_int(icf_ctx *ctx, const int *d, int n, int *out)
{
    if (int r = check_ctx(ctx)) return r;
    if (n < 0 || !out || (n && !d)) return fail(ctx, ICF_E_INVALID, "icf_sum_int: invalid argument");
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_sum_int returns a host value");
    *out = 0;
    if (n == 0) return 0;
    if (int r = lane_barrier(ctx)) return r;
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, ctx->stream, ctx->small + 4, 1, 0);
    hipLaunchKernelGGL(k_sum_int, dim3(n < 64 * 256 ? blocks_for(n, 256) : 64), dim3(256), 0, ctx->stream, d, n,
                       ctx->small + 4);
    HIPCHK(ctx, hipMemcpyAsync(out, ctx->small + 4, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

// The fused call.
static int assemble_impl(icf_ctx *ctx, const int *ie, int nElems, int el_stride, double *dcz, int *icz, int nCZs,
                         int cz_stride, double *dn, int nd_stride, double h, double *A, int nnzb, double *b, int N,
                         int *nCZDamaged, int *nCZFailed)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nElems, el_stride) || bad_units(nCZs, cz_stride) || nd_stride < 0 || nnzb < 0 || N < 0 ||
        (nElems && !ie) || (nCZs && (!dcz || !icz)) || !dn || (nnzb && !A) || (N && !b) || !(h > 0))
        return fail(ctx, ICF_E_INVALID, "icf_assemble_elems_and_czs: invalid argument");
    ConstUse cu(ctx);
    if (cu.err) return cu.err;
    // node fields read (x0, u, v, a, x) and written (F); CZ records rewritten in place
    const size_t ns = (size_t)nd_stride;
    OnLane ln(ctx, 0, [&] {
        return Access()
            .rd(ie, (EL_ROWS + 4) * (size_t)el_stride)
            .alloc(nCZs ? dcz : nullptr, true)
            .alloc(nCZs ? icz : nullptr, true)
            .rd(dn, ND_F * ns)
            .wr(dn + ND_F * ns, 3 * ns)
            .rd(dn + ND_XC * ns, 3 * ns)
            .wr(A, 9 * (size_t)nnzb)
            .wr(b, 3 * (size_t)N);
    });
    if (ln.err) return ln.err;
    std::vector<SrcKey> sv, sr;
    if (nElems) {
        sv.push_back({KIND_TET, ie, nElems, el_stride, EL_SLOTS, 16});
        sr.push_back({KIND_TET, ie, nElems, el_stride, EL_ROWS, 4});
    }
    if (nCZs) {
        sv.push_back({KIND_CZ, icz, nCZs, cz_stride, CZI_SLOTS, 36});
        sr.push_back({KIND_CZ, icz, nCZs, cz_stride, CZI_ROWS, 6});
    }
    std::vector<MapReq> req{{TGT_VALS, nnzb, sv}, {TGT_RHS, N, sr}};
    if (nElems) req.push_back({TGT_FORCE, -1, {{KIND_TET, ie, nElems, el_stride, EL_NODES, 4}}});
    const MapSrc tet{ie, nElems, el_stride, EL_NODES, 4, KIND_TET};
    if (int r = get_maps(ctx, req, nElems ? &tet : nullptr)) return r;
    SlotMap *mv = req[0].map, *mr = req[1].map, *mf = nElems ? req[2].map : nullptr;
    const bool tsum = mf && mr->tsum_ok;
    if (tsum)
        if (int r = grow(ctx, ctx->tsum, sizeof(double) * 3 * (size_t)mf->nkeys)) return r;
    // buffers grow before any work is issued (growing synchronizes the context's stream)
    if (int r = reserve_stage(ctx, nElems, nCZs)) return r;
    Timer tm(ctx);
    int *counts = ctx->small + 2;   // the two counts of GPU_Functionality.cs:474-475
    const int *dmg = icz ? icz + (size_t)cz_stride * CZI_TDAMAGED : nullptr;
    const int *fld = icz ? icz + (size_t)cz_stride * CZI_TFAILED : nullptr;
    const dim3 cnt_grid(nCZs < 64 * 256 ? blocks_for(std::max(nCZs, 1), 256) : 64);
    const bool fuse = ctx->overlap;
    // phase 1: tets and CZs (the counters are cleared by a kernel, so the call can be captured)
    if (fuse) {
        phase1_fused(ctx, ie, dn, nElems, el_stride, nd_stride, dcz, icz, nCZs, cz_stride, counts);
    } else {
        LAUNCH(ctx, "k_fill_int", k_fill_int, dim3(1), dim3(64), counts, 2, 0);
        stage_tets(ctx, ie, dn, nElems, el_stride, nd_stride);
        stage_czs(ctx, dcz, icz, dn, nCZs, cz_stride, nd_stride);
    }
    Stage st = make_stage(ctx, h);
    double *F = dn + (size_t)nd_stride * ND_F;
    // a blocking call's counters come back with its wait
    const bool tell = (nCZDamaged || nCZFailed || ctx->batch.spec_counts) && ctx->blocking && !ctx->capturing;
    const Report rep = tell ? new_report(ctx) : Report{};
    bool told = false;
    if (tsum && fuse && vals_force_rhs_fused(ctx, mv, A, mf, F, nd_stride, mr, b, dmg, fld, nCZs, counts, st, rep)) {
        told = tell && nCZs > 0;
        // done: node forces with the rhs rows, the counts and the BCSR values in one launch
    } else if (tsum) {
        // BCSR values and node forces (keeping each node's tet sum), then the rhs rows from
        // those sums plus their CZ terms, and the counts
        if (!(fuse && vals_force_fused(ctx, mv, A, mf, F, nd_stride, st))) {
            launch_vals(ctx, mv, A, 0, st);
            LAUNCH(ctx, "k_reduce_vec3<force,acc>", (k_reduce_vec3<true, true>), dim3(blocks_for(mf->nlaunch, 256)),
                   dim3(256), mf->loff, mf->codes, mf->keys, mf->nlaunch, F, nd_stride, 1, st, (double *)ctx->tsum.p);
        }
        if (fuse && (N || nCZs)) {
            const int nbr = N ? (int)(blocks_for(N, 256) + 7) / 8 * 8 : 0;
            LAUNCH(ctx, "k_rhs_counts", k_rhs_counts_fused, dim3(nbr + (nCZs ? cnt_grid.x : 0)), dim3(256), nbr,
                   mr->off, mr->codes, mr->cz_begin, mr->row_node, (const double *)ctx->tsum.p, N, b, st, dmg, fld,
                   nCZs, counts);
        } else {
            if (N)
                LAUNCH(ctx, "k_reduce_rhs_tsum", k_reduce_rhs_tsum, dim3(blocks_for(N, 256)), dim3(256), mr->off,
                       mr->codes, mr->cz_begin, mr->row_node, (const double *)ctx->tsum.p, N, b, st);
            if (nCZs) LAUNCH(ctx, "k_count_flags", k_count_flags, cnt_grid, dim3(256), dmg, fld, nCZs, counts);
        }
    } else {
        launch_vals(ctx, mv, A, 0, st);
        if (mf) launch_vec3(ctx, mf, F, nd_stride, 1, 1, st);
        launch_vec3(ctx, mr, b, 1, 3, 0, st);
        if (nCZs) LAUNCH(ctx, "k_count_flags", k_count_flags, cnt_grid, dim3(256), dmg, fld, nCZs, counts);
    }
    if (int r = ln.done()) return r;
    if (int r = tm.finish()) return r;
    if ((nCZDamaged || nCZFailed) && ctx->blocking && !ctx->capturing) {
        int sums[2] = {0, 0};
        if (told) {
            sums[0] = (int)((volatile unsigned *)rep.host)[CZ_DAMAGED];
            sums[1] = (int)((volatile unsigned *)rep.host)[CZ_FAILED];
        } else if (nCZs) {
            HIPCHK(ctx, hipMemcpyAsync(sums, ctx->small + 2, 2 * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
            HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        }
        if (nCZDamaged) *nCZDamaged = sums[0];
        if (nCZFailed) *nCZFailed = sums[1];
    }
    return 0;
}

int icf_assemble_elems_and_czs(icf_ctx *ctx, const int *ie, int nElems, int el_stride, double *dcz, int *icz, int nCZs,
                               int cz_stride, double *dn, int nd_stride, double h, double *A, int nnzb, double *b,
                               int N, int *nCZDamaged, int *nCZFailed)
{
    return assemble_impl(ctx, ie, nElems, el_stride, dcz, icz, nCZs, cz_stride, dn, nd_stride, h, A, nnzb, b, N,
                         nCZDamaged, nCZFailed);
}

int icf_assemble_batched(icf_ctx *ctx, const icf_worklist *wl, const int *ie, int el_stride, double *dcz, int *icz,
                         int cz_stride, double *dn, int nd_stride, double h, double *A, double *b, int *nCZDamaged,
                         int *nCZFailed)
{
    if (int r = check_ctx(ctx)) return r;
    if (!wl || wl->nSpecimens < 1 || wl->nSpecimens > (1 << 24) || !wl->tet_off || !wl->cz_off || !wl->row_off ||
        !wl->nnzb_off)
        return fail(ctx, ICF_E_INVALID, "icf_assemble_batched: invalid worklist");
    const int n = wl->nSpecimens;
    const int *tabs[4] = {wl->tet_off, wl->cz_off, wl->row_off, wl->nnzb_off};
    std::vector<int> off(4 * ((size_t)n + 1));
    for (int k = 0; k < 4; k++) {
        if (tabs[k][0] != 0) return fail(ctx, ICF_E_INVALID, "icf_assemble_batched: offsets must start at 0");
        for (int s = 0; s <= n; s++) {
            if (s && tabs[k][s] < tabs[k][s - 1])
                return fail(ctx, ICF_E_INVALID, "icf_assemble_batched: offsets must not decrease");
            off[(size_t)k * (n + 1) + s] = tabs[k][s];
        }
    }
    const int nE = wl->tet_off[n], nC = wl->cz_off[n], N = wl->row_off[n], nnzb = wl->nnzb_off[n];
    icf_ctx::Batch &B = ctx->batch;
    if (off != B.off) {
        if (ctx->capturing)
            return fail(ctx, ICF_E_CAPTURE, "icf_assemble_batched: new offsets cannot be uploaded during capture");
        if (int r = lane_barrier(ctx)) return r;
        if (int r = grow(ctx, B.d, sizeof(int) * (off.size() + 2 * (size_t)n))) return r;
        HIPCHK(ctx, hipMemcpyAsync(B.d.p, off.data(), sizeof(int) * off.size(), hipMemcpyHostToDevice, ctx->stream));
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        B.off = off;
        B.n = n;
        B.checked.clear();
        bump(ctx);                 // a captured batch reads the old offsets
    }
    const int *d = (const int *)B.d.p;
    const BatchOff bo{d, d + (n + 1), d + 2 * (n + 1), d + 3 * (n + 1), n};
    int *cnt = (int *)B.d.p + 4 * (n + 1);
    // The block-diagonal layout, checked before anything is written whenever the units or the
    // slot fields may have changed (a library write to them moves the fields' epoch).
    const std::vector<long long> sig{(long long)(uintptr_t)ie, (long long)(uintptr_t)icz, el_stride, cz_stride, nE,
                                     nC, (long long)ctx->fields_epoch};
    if (sig != B.checked) {
        if (ctx->capturing)
            return fail(ctx, ICF_E_CAPTURE, "icf_assemble_batched: run the batch once uncaptured before capture");
        if (int r = lane_barrier(ctx)) return r;
        int *d_err = ctx->small + 1;
        hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, ctx->stream, d_err, 1, 0);
        if (nE + nC)
            hipLaunchKernelGGL(k_batch_check, dim3(blocks_for((long long)nE + nC, 256)), dim3(256), 0, ctx->stream, ie,
                               nE, el_stride, icz, nC, cz_stride, bo, d_err);
        int e = 0;
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipMemcpyAsync(&e, d_err, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        if (e)
            return fail(ctx, ICF_E_INDEX,
                        "icf_assemble_batched: a unit writes a BCSR block or rhs row outside its specimen's ranges");
    }
    B.cz_off = bo.cz;
    B.spec_counts = cnt;
    B.spec_counted = false;
    const int ra = assemble_impl(ctx, ie, nE, el_stride, dcz, icz, nC, cz_stride, dn, nd_stride, h, A, nnzb, b, N,
                                 nullptr, nullptr);
    B.cz_off = nullptr;
    B.spec_counts = nullptr;
    if (ra) return ra;
    if (sig != B.checked) {
        B.checked = sig;
        B.checked.back() = (long long)ctx->fields_epoch;   // map checks inside the call may have moved it
    }
    OnLane ln(ctx, 0, [&] {
        return Access()
            .rd(nE ? ie : nullptr, (EL_ROWS + 4) * (size_t)el_stride)
            .rd(nC ? icz : nullptr, (CZI_ROWS + 6) * (size_t)cz_stride);
    });
    if (ln.err) return ln.err;
    if (nC && B.spec_counted) {
        // written by the fused value launch
    } else if (nC) {
        const int *dmg = icz + (size_t)cz_stride * CZI_TDAMAGED, *fld = icz + (size_t)cz_stride * CZI_TFAILED;
        LAUNCH(ctx, "k_batch_counts", k_batch_counts, dim3(n), dim3(256), dmg, fld, bo.cz, cnt);
    } else {
        LAUNCH(ctx, "k_fill_int", k_fill_int, dim3(blocks_for(2 * (long long)n, 256)), dim3(256), cnt, 2 * n, 0);
    }
    if (int r = ln.done()) return r;
    if ((nCZDamaged || nCZFailed) && ctx->blocking && !ctx->capturing) {
        std::vector<int> c(2 * (size_t)n);
        if (nC && B.spec_counted && n <= REPORT_SPECS) {
            for (size_t k = 0; k < c.size(); k++) c[k] = (int)((volatile unsigned *)ctx->rep_host)[REPORT_WORDS + k];
        } else {
            HIPCHK(ctx, hipMemcpyAsync(c.data(), cnt, sizeof(int) * c.size(), hipMemcpyDeviceToHost, ctx->stream));
            HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        }
        for (int k = 0; k < n; k++) {
            if (nCZDamaged) nCZDamaged[k] = c[2 * (size_t)k];
            if (nCZFailed) nCZFailed[k] = c[2 * (size_t)k + 1];
        }
    }
    return 0;
}

int icf_batch_cz_counts(icf_ctx *ctx, int *nCZDamaged, int *nCZFailed)
{
    if (int r = check_ctx(ctx)) return r;
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_batch_cz_counts during capture");
    const int n = ctx->batch.n;
    if (n == 0) return fail(ctx, ICF_E_INVALID, "icf_batch_cz_counts: no batched call yet");
    if (int r = sync_lanes(ctx)) return r;
    std::vector<int> c(2 * (size_t)n);
    HIPCHK(ctx, hipMemcpyAsync(c.data(), (int *)ctx->batch.d.p + 4 * (n + 1), sizeof(int) * c.size(),
                               hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < n; k++) {
        if (nCZDamaged) nCZDamaged[k] = c[2 * (size_t)k];
        if (nCZFailed) nCZFailed[k] = c[2 * (size_t)k + 1];
    }
    return 0;
}

int icf_nodes_infer(icf_ctx *ctx, const double *st, int st_stride, double *dn, int nd_stride, int nNodes, double h,
                    double beta, double gamma)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nNodes, st_stride) || bad_units(nNodes, nd_stride) || (nNodes && (!st || !dn)) || !(h > 0) ||
        !(beta > 0))
        return fail(ctx, ICF_E_INVALID, "icf_nodes_infer: invalid argument");
    if (nNodes == 0) return 0;
    OnLane ln(ctx, 0, everything);
    if (ln.err) return ln.err;
    Timer tm(ctx);
    LAUNCH(ctx, "k_nodes_infer", k_nodes_infer, dim3(blocks_for(3LL * nNodes, 256)), dim3(256), st, st_stride, dn,
           nd_stride, nNodes, h, beta, gamma);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_nodes_add_dx(icf_ctx *ctx, double *st, int st_stride, const int *altId, int nNodes, const double *dx)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nNodes, st_stride) || (nNodes && (!st || !altId || !dx)))
        return fail(ctx, ICF_E_INVALID, "icf_nodes_add_dx: invalid argument");
    if (nNodes == 0) return 0;
    OnLane ln(ctx, 0, everything);
    if (ln.err) return ln.err;
    Timer tm(ctx);
    LAUNCH(ctx, "k_nodes_add_dx", k_nodes_add_dx, dim3(blocks_for(3LL * nNodes, 256)), dim3(256), st, st_stride,
           altId, nNodes, dx);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_nodes_accept(icf_ctx *ctx, double *st, int st_stride, const double *dn, int nd_stride, int nNodes, double h)
{
    if (int r = check_ctx(ctx)) return r;
    if (bad_units(nNodes, st_stride) || bad_units(nNodes, nd_stride) || (nNodes && (!st || !dn)) || !(h > 0))
        return fail(ctx, ICF_E_INVALID, "icf_nodes_accept: invalid argument");
    if (nNodes == 0) return 0;
    OnLane ln(ctx, 0, everything);
    if (ln.err) return ln.err;
    Timer tm(ctx);
    LAUNCH(ctx, "k_nodes_accept", k_nodes_accept, dim3(blocks_for(3LL * nNodes, 256)), dim3(256), st, st_stride, dn,
           nd_stride, nNodes, h);
    if (int r = ln.done()) return r;
    return tm.finish();
}

int icf_build_pattern(icf_ctx *ctx, const int *altId, int nNodes, const int *ie, int nElems, int el_stride,
                      const int *icz, int nCZs, int cz_stride, const int *icr, int nImpacts, int cr_stride, int N,
                      int *csr_rows, int *csr_cols, int max_nnz, int *nnz)
{
    if (int r = check_ctx(ctx)) return r;
    if (!ctx->capturing)
        if (int r = lane_barrier(ctx)) return r;
    if (!nnz || nNodes < 0 || N < 0 || max_nnz < 0 || bad_units(nElems, el_stride) || bad_units(nCZs, cz_stride) ||
        bad_units(nImpacts, cr_stride) || (nNodes && !altId) || (nElems && !ie) || (nCZs && !icz) ||
        (nImpacts && !icr) || !csr_rows || (max_nnz && !csr_cols))
        return fail(ctx, ICF_E_INVALID, "icf_build_pattern: invalid argument");
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_build_pattern returns a host value");
    *nnz = 0;
    const PatSrc el{ie, nElems, el_stride, EL_NODES, 4, 0}, cz{icz, nCZs, cz_stride, CZI_VRTS, 6, 0},
        im{icr, nImpacts, cr_stride, CR_NODES, 4, 1};
    const long long Ms = (long long)nElems * pat_pairs(4, 0) + (long long)nCZs * pat_pairs(6, 0);
    const long long Mi = (long long)nImpacts * pat_pairs(4, 1);
    if (Ms + Mi >= (1LL << 31) - 1)
        return fail(ctx, ICF_E_CAPACITY, "icf_build_pattern: 2^31 or more candidate pairs");
    int cb = 1;
    while ((1LL << cb) <= (long long)N) cb++;
    const PatFields pf{altId, nNodes, ie, nElems, el_stride, icz, nCZs, cz_stride};
    const long long nsnap = (long long)nNodes + 4LL * nElems + 6LL * nCZs;
    auto &pc = ctx->patc;
    const bool kept = pc.valid && pc.nNodes == nNodes && pc.nElems == nElems && pc.el_stride == el_stride &&
                      pc.nCZs == nCZs && pc.cz_stride == cz_stride && pc.N == N;
    // scratch: keys and their distinct ones, or the impacts' pairs; counts per tile of keys or rows
    const unsigned ktiles = blocks_for(Ms, PAT_TILE), rtiles = blocks_for(N, 256), tiles = std::max(ktiles, rtiles);
    const size_t nr = (size_t)N, mi = (size_t)Mi, nt = (size_t)tiles + Tiles::group_words(tiles);
    const size_t keys = kept ? 0 : (size_t)Ms;
    if (int r = grow(ctx, ctx->pat_a, std::max(sizeof(unsigned long long) * keys, sizeof(int2) * mi) + 1)) return r;
    if (int r = grow(ctx, ctx->pat_b, std::max(sizeof(unsigned long long) * keys, sizeof(int) * 3 * mi) + 1)) return r;
    if (int r = grow(ctx, ctx->bp_l, sizeof(int) * (2 * nr + nt + 2))) return r;
    if (ctx->pat_cnt.bytes < sizeof(int) * nr) {
        if (int r = grow(ctx, ctx->pat_cnt, sizeof(int) * nr)) return r;
        HIPCHK(ctx, hipMemsetAsync(ctx->pat_cnt.p, 0, ctx->pat_cnt.bytes, ctx->stream));
    }
    int *w = (int *)ctx->bp_l.p + 2 * nr, *rank = (int *)ctx->pat_b.p;
    const Tiles tl{(unsigned *)w + 2, (unsigned *)w + 2 + tiles};
    const PatExtra x{(int2 *)ctx->pat_a.p, rank, (int *)ctx->pat_cnt.p, (int *)ctx->bp_l.p, (int *)ctx->bp_l.p + nr,
                     rank + mi, rank + 2 * mi, (unsigned *)w};
    const dim3 b(256);
    // The elements' and CZs' distinct blocks are kept and used while their node ids and the altIds
    // are what they were, which the same launches find out; where they are not, all is built anew.
    bool fresh = !kept;
    Report rep;
    for (;; fresh = true) {
        rep = new_report(ctx);
        if (fresh) {
            pc.valid = false;
            if (int r = grow(ctx, pc.rows, sizeof(int) * (nr + 1))) return r;
            if (int r = grow(ctx, pc.cols, sizeof(int) * (size_t)Ms + 1)) return r;
            if (int r = grow(ctx, pc.snap, sizeof(int) * (size_t)nsnap + 1)) return r;
            if (int r = grow(ctx, ctx->pat_a, sizeof(unsigned long long) * (size_t)Ms + 1)) return r;
            if (int r = grow(ctx, ctx->pat_b, sizeof(unsigned long long) * (size_t)Ms + 1)) return r;
            auto *ka = (unsigned long long *)ctx->pat_a.p, *kb = (unsigned long long *)ctx->pat_b.p;
            int *count = nullptr;
            if (Ms > 0) {
                count = w + 1;
                size_t sb = 0;
                HIPCHK(ctx, hipcub::DeviceRadixSort::SortKeys(nullptr, sb, ka, kb, (int)Ms, 0, 2 * cb, ctx->stream));
                if (int r = grow(ctx, ctx->scan_tmp, sb)) return r;
                hipLaunchKernelGGL(k_pat_emit, dim3(blocks_for(Ms, 256)), b, 0, ctx->stream, el, cz, altId, nNodes, N,
                                   cb, ka, tl, ktiles, rep);
                HIPCHK(ctx, hipcub::DeviceRadixSort::SortKeys(ctx->scan_tmp.p, sb, ka, kb, (int)Ms, 0, 2 * cb,
                                                              ctx->stream));
                hipLaunchKernelGGL(k_pat_count, dim3(ktiles), b, 0, ctx->stream, kb, Ms, cb, tl);
                hipLaunchKernelGGL(k_pat_compact, dim3(ktiles), b, 0, ctx->stream, kb, Ms, cb, tl, ka, (int *)pc.cols.p,
                                   count);
            }
            hipLaunchKernelGGL(k_pat_rows, dim3(blocks_for((long long)N + 1, 256)), b, 0, ctx->stream, ka, count, N, cb,
                               (int *)pc.rows.p);
            if (nsnap > 0)
                hipLaunchKernelGGL(k_pat_snap, dim3(blocks_for(nsnap, 256)), b, 0, ctx->stream, pf, nsnap,
                                   (int *)pc.snap.p);
        }
        const int *srow = (const int *)pc.rows.p, *scol = (const int *)pc.cols.p;
        PatExtra xe = x;           // the buffers may have moved for the keys
        xe.item = (int2 *)ctx->pat_a.p;
        xe.rank = (int *)ctx->pat_b.p;
        xe.raw = xe.rank + mi;
        xe.cols = xe.raw + mi;
        const unsigned cmp = fresh ? 0u : blocks_for(nsnap, 256), pairs = blocks_for(Mi, 256);
        if (cmp + pairs)
            hipLaunchKernelGGL(k_pat_extra, dim3(cmp + pairs), b, 0, ctx->stream, pf, nsnap, (const int *)pc.snap.p, cmp,
                               im, nNodes, N, srow, scol, xe, tl, rtiles, rep);
        if (Mi > 0 && N > 0) {
            hipLaunchKernelGGL(k_pat_reserve, dim3(rtiles), b, 0, ctx->stream, N, xe);
            hipLaunchKernelGGL(k_pat_fill, dim3(pairs), b, 0, ctx->stream, Mi, xe);
            hipLaunchKernelGGL(k_pat_distinct, dim3(rtiles), b, 0, ctx->stream, N, xe, tl);
        }
        hipLaunchKernelGGL(k_pat_write, dim3(blocks_for((long long)N + 1, 256)), b, 0, ctx->stream, srow, scol, N,
                           Mi > 0 && N > 0, xe, tl, rtiles, max_nnz, csr_rows, csr_cols, rep);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        if (fresh || !reported(rep, PAT_DIFF)) break;
    }
    if (fresh && !reported(rep, PAT_ERR_STATIC)) {
        pc.nNodes = nNodes, pc.nElems = nElems, pc.el_stride = el_stride, pc.nCZs = nCZs;
        pc.cz_stride = cz_stride, pc.N = N;
        pc.valid = true;
    }
    if (reported(rep, PAT_ERR_STATIC) || reported(rep, PAT_ERR_IMPACT))
        return fail(ctx, ICF_E_INDEX, "icf_build_pattern: a node id or altId is out of range");
    *nnz = (int)((volatile unsigned *)rep.host)[PAT_NNZ];
    if (*nnz > max_nnz) return fail(ctx, ICF_E_CAPACITY, "icf_build_pattern: more blocks than max_nnz");
    return 0;
}

int icf_pack_pcsr(icf_ctx *ctx, const int *altId, int nNodes, const int *csr_rows, const int *csr_cols, int N,
                  int *ie, int nElems, int el_stride, int *icz, int nCZs, int cz_stride, int *icr, int nImpacts,
                  int cr_stride)
{
    if (int r = check_ctx(ctx)) return r;
    if (!ctx->capturing)
        if (int r = lane_barrier(ctx)) return r;
    if (nNodes < 0 || N < 0 || bad_units(nElems, el_stride) || bad_units(nCZs, cz_stride) ||
        bad_units(nImpacts, cr_stride) || (nNodes && !altId) || !csr_rows || (nElems && !ie) || (nCZs && !icz) ||
        (nImpacts && !icr))
        return fail(ctx, ICF_E_INVALID, "icf_pack_pcsr: invalid argument");
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_pack_pcsr reports index errors to the host");
    PackAll ps{{{ie, nElems, el_stride}, {icz, nCZs, cz_stride}, {icr, nImpacts, cr_stride}}, {}};
    const SlotMap *held[3][2] = {};
    for (int k = 0; k < 3; k++) {
        PackPart &p = ps.part[k];
        const int slot0 = k == 1 ? CZI_SLOTS : EL_SLOTS, row0 = k == 1 ? CZI_ROWS : EL_ROWS, K = k == 1 ? 6 : 4;
        if (!p.n) continue;
        held[k][0] = map_over(ctx, p.base, p.n, p.stride, slot0, K * K, &p.slots);
        held[k][1] = map_over(ctx, p.base, p.n, p.stride, row0, K, &p.rows);
    }
    ps.wave1[0] = pack_waves(nElems, 4);
    ps.wave1[1] = ps.wave1[0] + pack_waves(nCZs, 6);
    ps.wave1[2] = ps.wave1[1] + pack_waves(nImpacts, 4);
    if (ps.wave1[2] == 0) return 0;
    const Report rep = new_report(ctx);
    hipLaunchKernelGGL(k_pack_pcsr, dim3(blocks_for(ps.wave1[2], 4)), dim3(256), 0, ctx->stream, ps, altId, nNodes,
                       csr_rows, csr_cols, N, rep);
    const hipError_t launched = hipGetLastError();
    const hipError_t waited = hipStreamSynchronize(ctx->stream);
    const bool err = launched != hipSuccess || waited != hipSuccess || reported(rep, PACK_ERR);
    for (int k = 0; k < 3; k++) {
        const PackPart &p = ps.part[k];
        if (!p.n) continue;
        const int slot0 = k == 1 ? CZI_SLOTS : EL_SLOTS, row0 = k == 1 ? CZI_ROWS : EL_ROWS, K = k == 1 ? 6 : 4;
        const uintptr_t lo = (uintptr_t)(p.base + (size_t)p.stride * slot0),
                        mid = (uintptr_t)(p.base + (size_t)p.stride * row0),
                        hi = (uintptr_t)(p.base + (size_t)p.stride * (row0 + K));
        for (int f = 0; f < 2; f++) {
            const uintptr_t a = f ? mid : lo, b = f ? hi : mid;
            const bool differ = err || reported(rep, PACK_CHANGED + 2 * k + f);
            packed_range(ctx, a, b, held[k][f], !differ, differ && !err);
        }
    }
    HIPCHK(ctx, launched);
    HIPCHK(ctx, waited);
    if (err) return fail(ctx, ICF_E_INDEX, "icf_pack_pcsr: a node id is out of range or a pair is not in the pattern");
    return 0;
}

int icf_broad_phase(icf_ctx *ctx, const double *dn, int nd_stride, const int *ie, int el_all_stride, int nTets,
                    int exclude_shared, int *pairs, long long max_pairs, long long *nOut)
{
    if (int r = check_ctx(ctx)) return r;
    if (!ctx->capturing)
        if (int r = lane_barrier(ctx)) return r;
    if (!nOut || bad_units(nTets, el_all_stride) || nd_stride < 0 || max_pairs < 0 || (nTets && (!dn || !ie)) ||
        (max_pairs && !pairs))
        return fail(ctx, ICF_E_INVALID, "icf_broad_phase: invalid argument");
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_broad_phase returns a host value");
    *nOut = 0;
    if (nTets == 0) return 0;
    const int nT = nTets;
    if (nT > (1 << 23)) return fail(ctx, ICF_E_CAPACITY, "icf_broad_phase: more than 2^23 surface tets");
    // scratch: in cell order the records (8 nT doubles' worth), k-DOPs in FP64 (24 nT) and FP32 (12 nT); minimum
    // corners (3 nT), bounds, grid
    const int nb = std::min<int>(blocks_for(nT, 256), BP_BLOCKS);
    const size_t nbounds = (size_t)BP_BLOCKS * BP_NBOUNDS, ngrid = (sizeof(BpGrid) + 7) / 8;
    if (int r = grow(ctx, ctx->bp_f, sizeof(double) * ((size_t)47 * nT + nbounds + ngrid))) return r;
    if (int r = grow(ctx, ctx->bp_i, sizeof(int) * 3 * (size_t)nT)) return r;
    BpTet *srec = (BpTet *)ctx->bp_f.p;
    double2 *skd = (double2 *)(srec + nT);                         // 12 double2 = 24 doubles per tet
    float4 *sk32 = (float4 *)(skd + (size_t)BP_DIRS * nT);         // 6 float4 = 12 doubles per tet
    double *lo = (double *)ctx->bp_f.p + (size_t)44 * nT, *bounds = lo + (size_t)3 * nT;
    BpGrid *grid = (BpGrid *)(bounds + nbounds);
    auto *key = (unsigned *)ctx->bp_i.p;
    int *rank = (int *)(key + nT), *sidx = rank + nT;
    // Every launch takes the grid from device memory and what it counts from there too, so one wait at
    // the end serves all (with two, library scans, copies of the counts and the slower search a call took
    // 219 us on 3,300 tets and 546 on 353,000, now 75 and 345); the launches and buffers are as large as the last search's grid and candidates ask
    // for, and a search whose do not fit is repeated with what it found.
    const long long cells = ctx->bp_cells ? ctx->bp_cells : 8192, inner = ctx->bp_inner ? ctx->bp_inner : 4096;
    long long capG = cells + cells / 4 + 64, capC = inner + inner / 4 + 64;
    // at least 64 places per region, so that every region's grid row has a workgroup
    long long cap = std::max<long long>({ctx->bp_cap, 4LL * nT, 64LL * BP_PARTS});
    const unsigned atiles = blocks_for(nT, BP_TILE);
    long long ncand = 0;
    bool grown = false, fine = false;
    for (;;) {
        if (cap >= (1LL << 31)) return fail(ctx, ICF_E_CAPACITY, "icf_broad_phase: more than 2^31 candidate pairs");
        const unsigned ctiles = blocks_for(capG, BP_TILE);
        const size_t ntotal = (size_t)BP_PARTS * BP_PART_STRIDE, nct = ctiles + Tiles::group_words(ctiles);
        const size_t nw = nct + atiles + Tiles::group_words(atiles);
        if (int r = grow(ctx, ctx->bp_l, sizeof(long long) * ntotal + sizeof(unsigned) * nw)) return r;
        if (int r = grow(ctx, ctx->bp_c, sizeof(int) * 2 * ((size_t)capG + 1))) return r;
        if (int r = grow(ctx, ctx->pat_a, sizeof(unsigned long long) * (size_t)cap)) return r;
        if (int r = grow(ctx, ctx->pat_b, sizeof(unsigned long long) * (size_t)cap)) return r;
        if (int r = grow(ctx, ctx->bp_g, sizeof(int) * (2 * ((size_t)nT + 1) + (size_t)cap))) return r;
        auto *tot = (unsigned long long *)ctx->bp_l.p;
        auto *w = (unsigned *)(tot + ntotal);
        const Tiles ct{w, w + ctiles}, at{w + nct, w + nct + atiles};
        int *count = (int *)ctx->bp_c.p, *first = count + capG + 1;   // per cell, and their exclusive scan
        int *acount = (int *)ctx->bp_g.p, *start = acount + nT + 1, *rnk = start + nT + 1;
        auto *pa = (unsigned long long *)ctx->pat_a.p, *grp = (unsigned long long *)ctx->pat_b.p;
        const Report rep = new_report(ctx);
        const dim3 b(256), tets(blocks_for(nT, 256));
        hipLaunchKernelGGL(k_bp_clear, dim3(blocks_for(std::max<long long>({capG + 1, nT + 1LL, (long long)ntotal}), 256)),
                           b, 0, ctx->stream, count, (int)(capG + 1), acount, nT + 1, tot, (int)ntotal, ct, ctiles, at,
                           atiles);
        hipLaunchKernelGGL(k_bp_kdop, dim3(nb), b, 0, ctx->stream, dn, nd_stride, ie, el_all_stride, nT, lo, bounds, rep);
        hipLaunchKernelGGL(k_bp_cell, tets, b, 0, ctx->stream, lo, nT, bounds, nb, (int)capG, (int)capC, grid, key, rank,
                           count, rep);
        hipLaunchKernelGGL(k_bp_tiles, dim3(ctiles), b, 0, ctx->stream, count, -1, grid, ct);
        hipLaunchKernelGGL(k_bp_scan, dim3(ctiles), b, 0, ctx->stream, count, -1, grid, ct, first, -1, rep);
        hipLaunchKernelGGL(k_bp_sorted, tets, b, 0, ctx->stream, dn, nd_stride, nT, key, rank, first, ie, el_all_stride,
                           grid, sidx, srec, skd, sk32);
        // candidate pairs per cell (16-bit steps), collected in LDS and appended in batches; the
        // exact test; the passing pairs grouped by a (a counting sort) and placed by their rank of b
        // within the group: the pairs in (a, b) order.  The launches after the search take the
        // candidate count from device memory (their grids cover the buffer).  Where the
        // launch has room for 10,240 cells at most (the last search's, about 8,100, and a quarter) several
        // waves share one: 166 us a call against 180 with 25 tets in each of 4,096 cells, 117 against 128
        // in 1,728; from 8,000 cells on the shared ones are slower (244 against 235, 292 against 277 in
        // 10,648).  With 6 tets a cell sharing costs 1 us of 71 to 5 of 95 over these sizes.
        int slices = (int)std::min<long long>(16, std::max(1LL, 20480 / capC));
        if (slices > 1) slices -= slices % BPW_WAVES;      // a workgroup's waves share a cell
        hipLaunchKernelGGL(fine ? k_bp_cellwave<true> : k_bp_cellwave<false>,
                           dim3(blocks_for(capC * slices, 512 * BPW_WAVES) * 512), dim3(64 * BPW_WAVES), 0, ctx->stream,
                           srec, sk32, exclude_shared, grid, slices, slices > 1 ? 4 : BPW_OWN, first, tot, pa, cap);
        const dim3 gparts(blocks_for(cap / BP_PARTS, 256), BP_PARTS);   // a grid row per region
        hipLaunchKernelGGL(k_bp_exact, gparts, b, 0, ctx->stream, skd, sk32, sidx, tot, cap, pa, rnk, acount);
        hipLaunchKernelGGL(k_bp_tiles, dim3(atiles), b, 0, ctx->stream, acount, nT, grid, at);
        hipLaunchKernelGGL(k_bp_scan, dim3(atiles), b, 0, ctx->stream, acount, nT, grid, at, start, BP_NV, rep);
        hipLaunchKernelGGL(k_bp_scatter, gparts, b, 0, ctx->stream, pa, rnk, tot, cap, start, grp, rep);
        if (max_pairs > 0)
            hipLaunchKernelGGL(k_bp_place, dim3(blocks_for(cap, 256)), b, 0, ctx->stream, grp, start, nT, grid, max_pairs,
                               pairs);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        const volatile unsigned *got = rep.host;
        if (reported(rep, BP_BAD)) return fail(ctx, ICF_E_INDEX, "icf_broad_phase: bad node id");
        if (reported(rep, BP_NONFINITE))
            return fail(ctx, ICF_E_INVALID, "icf_broad_phase: non-finite node positions");
        ctx->bp_cells = got[BP_G];
        ctx->bp_inner = got[BP_NCELL];
        if (reported(rep, BP_BIG)) {
            capG = std::max(capG, ctx->bp_cells + ctx->bp_cells / 4);
            capC = std::max(capC, ctx->bp_inner + ctx->bp_inner / 4);
            continue;
        }
        ncand = got[BP_CAND];
        if (ncand <= cap / BP_PARTS) {
            *nOut = got[BP_NV];
            break;
        }
        if (!fine && BP_PARTS * ncand > BP_DENSE * nT) {
            fine = true;
            continue;
        }
        if (grown) return fail(ctx, ICF_E_CAPACITY, "icf_broad_phase: pair count changed between two searches");
        grown = true;
        cap = BP_PARTS * (ncand + ncand / 4);
    }
    ctx->bp_cap = std::max(ctx->bp_cap, BP_PARTS * (ncand + ncand / 4));
    if (*nOut > max_pairs) return fail(ctx, ICF_E_CAPACITY, "icf_broad_phase: more pairs than max_pairs");
    return 0;
}

int icf_nl2set(icf_ctx *ctx, const int *masks, const int *pairs, int nPairs, const int *ie, int el_all_stride,
               int *nl2, int tet_stride, int *nOut)
{
    if (int r = check_ctx(ctx)) return r;
    if (!ctx->capturing)
        if (int r = lane_barrier(ctx)) return r;
    if (!nOut || nPairs < 0 || el_all_stride < 0 || tet_stride < 0 || (nPairs && (!masks || !pairs || !ie)) ||
        (tet_stride && !nl2))
        return fail(ctx, ICF_E_INVALID, "icf_nl2set: invalid argument");
    if (ctx->capturing) return fail(ctx, ICF_E_CAPTURE, "icf_nl2set returns a host value");
    *nOut = 0;
    if (nPairs == 0) return 0;
    if (int r = note_write(ctx, nl2, sizeof(int) * 2 * (size_t)tet_stride, "icf_nl2set")) return r;
    const unsigned nb = blocks_for(nPairs, 256);
    const size_t ng = Tiles::group_words(nb);
    if (int r = grow(ctx, ctx->bp_i, (size_t)nPairs)) return r;
    if (int r = grow(ctx, ctx->bp_l, sizeof(unsigned) * ((size_t)nb + 2 * ng))) return r;
    auto *w = (unsigned *)ctx->bp_l.p;
    const Tiles tl{w, w + nb};
    auto *kept = (unsigned char *)ctx->bp_i.p;
    // the table: a power of two at least twice the last call's distinct tuples (a quarter more) or one
    // for 16 pairs; a tuple without a slot in 16 buckets asks for another round with room for all
    unsigned long long need = std::max({2048LL, ctx->nl2_last + ctx->nl2_last / 4, (long long)nPairs / 16});
    for (int round = 0;; round++) {
        unsigned long long H = 1;
        while (H < 2ULL * need) H <<= 1;
        if (int r = grow(ctx, ctx->pat_a, sizeof(Nl2Bucket) * (H / 4))) return r;
        const Nl2Table t{(Nl2Bucket *)ctx->pat_a.p, H / 4 - 1, w + nb + ng};
        const Report rep = new_report(ctx);
        hipLaunchKernelGGL(k_nl2_clear, dim3(blocks_for((long long)H, 256)), dim3(256), 0, ctx->stream, t, tl, nb);
        hipLaunchKernelGGL(k_nl2_emit, dim3(nb), dim3(256), 0, ctx->stream, masks, pairs, nPairs, ie, el_all_stride, t,
                           round ? H / 4 : 16ULL, kept, rep);
        hipLaunchKernelGGL(k_nl2_keep, dim3(nb), dim3(256), 0, ctx->stream, pairs, nPairs, ie, el_all_stride, t, kept,
                           tl, rep);
        hipLaunchKernelGGL(k_nl2_write, dim3(nb), dim3(256), 0, ctx->stream, kept, pairs, nPairs, ie, el_all_stride, t, tl,
                           nl2, tet_stride, rep);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
        const volatile unsigned *got = rep.host;
        need = got[NL2_TOTAL];
        if (need > NL2_MAX) return fail(ctx, ICF_E_CAPACITY, "icf_nl2set: more than 2^28 tuples");
        if (reported(rep, NL2_FULL)) continue;
        *nOut = (int)got[NL2_NUM];
        ctx->nl2_last = *nOut;
        break;
    }
    if (*nOut > tet_stride) return fail(ctx, ICF_E_CAPACITY, "icf_nl2set: more tuples than tet_stride");
    return 0;
}

}  // extern "C"
