// icf_device.h -- device-side constants, layouts and math helpers shared by every kernel of
// libicflow_hip.so.  Included once, by icf_lib.hip (single translation unit, so one
// __constant__ block serves all kernels).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace icf {

// ---- SoA field offsets of the reference buffers -------------------------------------------
// node array (double, 18 x nd_stride): GPU_Functionality.cs:55-61
constexpr int ND_X0 = 0, ND_UN = 3, ND_VN = 6, ND_AN = 9, ND_F = 12, ND_XC = 15;
// elastic tet (int, 28 x el_stride): elem_kernels9/element_kernels2.h:2-5
constexpr int EL_NODES = 0, EL_SLOTS = 4, EL_ROWS = 20;
// CZ int (58 x cz_stride) / double (16 x cz_stride): cz_kernels9/cz_kernels.h:13-32
constexpr int CZI_FAILED = 0, CZI_TCONTACT = 1, CZI_TDAMAGED = 2, CZI_TFAILED = 3, CZI_VRTS = 4,
              CZI_SLOTS = 10, CZI_ROWS = 46;
constexpr int CZD_PMAX = 0, CZD_TMAX = 3, CZD_TPMAX = 6, CZD_TTMAX = 9, CZD_DN = 12, CZD_DT = 13,
              CZD_TN = 14, CZD_TT = 15;
// impact (int, 28 x cr_stride): collision_response.h:48-50, GPU_Functionality.cs:643-663
constexpr int CR_NODES = 0, CR_SLOTS = 4, CR_ROWS = 20;

// ---- kinds of contributing units (top bits of a slot-map code) ----------------------------
constexpr uint32_t KIND_TET = 0, KIND_CZ = 1, KIND_CONTACT = 2;
constexpr int CODE_UNIT_BITS = 24;
constexpr uint32_t CODE_UNIT_MAX = (1u << CODE_UNIT_BITS) - 1;
__host__ __device__ inline uint32_t make_code(uint32_t kind, uint32_t unit, uint32_t q)
{
    return (kind << 30) | (unit << 6) | q;
}
constexpr uint32_t CODE_NONE = 0xffffffffu;      // no contribution (kind 3 does not exist)
__host__ __device__ inline uint32_t code_kind(uint32_t c) { return c >> 30; }
// The unit is hidden from the optimizer after the mask: knowing it to be 24 bits, the compiler
// (ROCm 7.2) takes a record's address for a 24-bit product, drops the mask that such a product
// would not need, and then emits the full-width v_mad_u64_u32 -- an address kind << 24 records off.
__device__ inline uint32_t code_unit(uint32_t c)
{
    uint32_t u = (c >> 6) & CODE_UNIT_MAX;
    asm("" : "+v"(u));
    return u;
}
__host__ __device__ inline uint32_t code_q(uint32_t c) { return c & 63u; }

// In the lists of BCSR blocks the local index of a CZ's block (a, b) = (q / 6, q % 6) is kept as
// what its value needs: the pair of midplane nodes and whether the block is negated (top with
// bottom nodes).
__host__ __device__ inline int cz_pair(int ia, int ib)
{
    const int lo = ia < ib ? ia : ib, hi = ia < ib ? ib : ia;
    return lo * 3 - lo * (lo - 1) / 2 + (hi - lo);   // 00 01 02 11 12 22
}
__device__ inline uint32_t czv_code(uint32_t q)
{
    const int a = (int)(q / 6), b = (int)(q % 6);
    return (uint32_t)cz_pair(a % 3, b % 3) | ((a < 3) != (b < 3) ? 8u : 0u);
}
__device__ inline uint32_t czv_pair(uint32_t c) { return c & 7u; }
__device__ inline bool czv_neg(uint32_t c) { return (c & 8u) != 0; }

// ---- staged per-unit records (AoS, one record per unit) -----------------------------------
// tet tangent, isotropic E: corotated gradients g~ = R g (12), rest volume V, 3 pad.
constexpr int TET_ISO_REC = 16;
// tet tangent, general E: R (9, row-major), rest gradients g (12), V, 2 pad.
constexpr int TET_GEN_REC = 24;
// tet residual: 12 doubles.
constexpr int TET_RHS_REC = 12;
// CZ tangent: per pair (ia, ib), ia <= ib, of midplane nodes the symmetric 3x3 block
// sum_gp s_ia s_ib Q_gp, Q = (w a_J) R^T T_d R, as xx,xy,xz,yy,yz,zz.
constexpr int CZ_PAIRS = 6, CZ_TAN_REC = 6 * CZ_PAIRS;
// CZ residual: the three top nodes' parts; the bottom nodes' are their negatives.
constexpr int CZ_RHS_REC = 9;
// contact: 78 packed upper-triangle entries of (k/2) Hess d^2, then 12 forces, 6 pad.
// impact records: the 10 upper 3x3 blocks of the 12x12 tangent, block (a, b) a <= b at
// ct_block(a, b), each whole and row-major (90 values, FP32 in mixed mode), and the 12 node
// forces (FP64) in a separate array
constexpr int CT_TAN_REC = 90, CT_F_REC = 12;
__host__ __device__ inline int ct_block(int a, int b) { return a * 4 - (a * (a - 1)) / 2 + (b - a); }

// ---- model constants -----------------------------------------------------------------------
struct DevConsts {
    double E[36];
    double M[144];
    double nbeta, ngamma, dampM, dampK, rho, grav;
    double G_fn, G_ft, f_tn, f_tt, alpha, beta, rn, rt;
    double p_m, p_n, deln, delt, pMtn, pMnt, gam_n, gam_t;
    double sf[9];           // sf[node*3 + gp]
    double lam, mu;         // isotropic split of E (valid when iso != 0)
    double m4[16];          // M[(3i)*12 + 3j]: the mass block (i,j) is m4[4i+j] I3 when iso != 0
    double m_ii, m_ij;      // its two values, where it has only two: on and off the diagonal
    float m_iif, m_ijf;
    int m_two;              // whether it has
    int iso;
    int alpha_n, beta_n;    // alpha, beta where they are integers from 2 to 16, else 0
    // constant factors of the PPR expressions, formed on the host with the same operations
    // and order as in PPR_math.h / cz_kernels.h, so they are the same doubles
    double k_tn, k_tt;              // gam_n / deln, gam_t / delt
    double k_dnn, k_dtt, k_dnt;     // gam_n / (deln deln), gam_t / (delt delt), gam_n gam_t / (deln delt)
    double pm_alpha, pn_beta;       // p_m / alpha, p_n / beta
    double thr_n, thr_t;            // f_tn * 0.05, f_tt * 0.05
    double lim_n, lim_t;            // deln * rn / 5, delt * rt / 5
    // powers at zero opening: (1 - 0)^e = 1 and (p/a + 0)^e, used by Dnn_(0, .) etc.
    double bn0[3], bt0[3];  // (p_m/alpha)^{p_m, p_m-1, p_m-2}, (p_n/beta)^{p_n, p_n-1, p_n-2}
    float Ef[36];
    float Mf[144];
    float lamf, muf;
    float m4f[16];
};

// 16 bytes at an 8-byte aligned place
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(8), may_alias));
typedef double f64x2 __attribute__((ext_vector_type(2), aligned(8), may_alias));

// ---- small vector helpers --------------------------------------------------------------------
template <typename T>
__device__ inline T dot3(const T *a, const T *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// What a call's kernels tell the host: words in pinned host memory, read after the wait that the
// call makes anyway, so that no copy and no clearing launch is needed.  A word is set when it holds
// the call's sequence number; the device copy of the words keeps all but the first few threads
// that set one off the bus.
constexpr int REPORT_WORDS = 32;
constexpr int CZ_DAMAGED = 23, CZ_FAILED = 24;      // values: the CZ counts of an assembly
constexpr int REPORT_SPECS = 1024;                  // behind the words, two counts of as many specimens
struct Report {
    unsigned *dev, *host;
    unsigned seq;
    __device__ inline void set(int k) const
    {
        if (is(k)) return;
        __hip_atomic_store(dev + k, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(host + k, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // whether an earlier launch of the call set word k; any launch
    __device__ inline bool was(int k) const { return dev[k] == seq; }
    __device__ inline bool is(int k) const
    {
        return __hip_atomic_load(dev + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == seq;
    }
    // a value, from one thread
    __device__ inline void put(int k, unsigned v) const
    {
        __hip_atomic_store(host + k, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
};

// Sum over the 256 threads of the workgroup, in every thread.
__device__ inline unsigned sum256(unsigned x, unsigned *part)
{
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = x;
    __syncthreads();
    const unsigned t = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    return t;
}

// Exclusive scan over the 256 threads of the workgroup; total in every thread.
template <typename T>
__device__ inline T scan256(T v, T *part, T &total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const T y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) part[wave] = x;
    __syncthreads();
    T before = 0;
    total = 0;
    for (int w = 0; w < 4; w++) {
        if (w < wave) before += part[w];
        total += part[w];
    }
    __syncthreads();
    return before + x - v;
}

// Where each workgroup's part of an ordered list starts, without a scan launch in between: a launch
// leaves one count per workgroup and per GROUP workgroups (`groups`, zero before it), and in the
// next one every workgroup adds up what lies before its own.  A library scan is two or three
// launches of 4 to 7 us each for lists of any size that occurs here.  The groups' counts lie a cache
// line apart: side by side, the atomics of 6,458 workgroups took 44 us, one after the other.
struct Tiles {
    static constexpr unsigned GROUP = 256, STRIDE = 32;
    unsigned *sums, *groups;
    __host__ __device__ static unsigned ngroups(unsigned n) { return (n + GROUP - 1) / GROUP; }
    // words of the groups' counts
    __host__ __device__ static size_t group_words(unsigned n) { return (size_t)ngroups(n) * STRIDE; }
    __device__ static inline void add(unsigned *groups, unsigned w, unsigned v)
    {
        if (v) atomicAdd(groups + (size_t)(w / GROUP) * STRIDE, v);
    }
    // from one thread of workgroup w
    __device__ inline void put(unsigned w, unsigned v) const
    {
        sums[w] = v;
        add(groups, w, v);
    }
    // all 256 threads: the sum of the workgroups before w; of all n
    __device__ inline unsigned before(unsigned w, unsigned *part) const
    {
        const unsigned g = w / GROUP, t = g * GROUP + threadIdx.x;
        unsigned x = t < w ? sums[t] : 0u;
        for (unsigned i = threadIdx.x; i < g; i += 256) x += groups[(size_t)i * STRIDE];
        return sum256(x, part);
    }
    __device__ inline unsigned total(unsigned n, unsigned *part) const
    {
        unsigned x = 0;
        for (unsigned i = threadIdx.x; i < ngroups(n); i += 256) x += groups[(size_t)i * STRIDE];
        return sum256(x, part);
    }
    // all threads of one workgroup, in a launch before
    __device__ static inline void clear(unsigned *groups, unsigned n)
    {
        for (unsigned i = threadIdx.x; i < ngroups(n); i += blockDim.x) groups[(size_t)i * STRIDE] = 0u;
    }
};

// Index of entry (r, c), r <= c, in a packed upper triangle of a 12x12 matrix.
__host__ __device__ inline int upper12(int r, int c) { return r * 12 - (r * (r - 1)) / 2 + (c - r); }

}  // namespace icf
