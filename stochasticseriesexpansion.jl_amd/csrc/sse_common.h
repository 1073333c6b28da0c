// sse_common.h -- device-side data layout and helpers of the SSE sweep.
//
// Layout in HBM (one allocation per batch unless noted):
//   DevModel[n_models]      model graph + per-bond-type VertexData tables
//   DevWalker[n_walkers]    per-walker scalars and slab pointers
//   slab pool               per walker one slab: ops[cap] (u32), then a record
//                           region used as dense links[legs*cap] (i32, legs =
//                           2 * sites per bond) by the lane kernels; the wave
//                           kernels keep there, per slot p and bond site k,
//                             idx[sites*cap]  how many earlier operators act on
//                                             the operator's k-th site (u32)
//                           and behind it the worm update's entry words of the
//                           slots, or its records when they do not fit LDS
//                           (sse_worm.h); carved from a device bump allocator,
//                           so the cutoff L grows inside the kernels
//   spins/first/last        [n_walkers][n_sites] u8 / i32 / i32 (wave kernels: last
//                           holds the site's operator count, first its first entry)
//
// Operator code (u32): 0 = identity, else 1 | vcode<<1 | bond<<11,
// vcode = diag | vidx<<1 (vidx 0-based).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define SSE_WAVE 64

struct DevVD {
    int32_t dims0, dims1, nv, max_worm, n_exits, nsites;
    int32_t dims[4];           // local dimension of each of the nsites bond sites
    double energy_offset;
    const double *weights;     // [nv]
    const int8_t *signs;       // [nv]
    const uint8_t *leg_states; // [nv][2*nsites]
    const int32_t *diag_vertex;// [prod(dims)]
    const int32_t *toff;       // [nv][max_worm][2*nsites]
    const int32_t *tcnt;       // [nv][max_worm][2*nsites]
    const double *cum;         // [n_exits]
    const int32_t *tgt;        // [n_exits]
    const uint8_t *eleg;       // [n_exits]
    const uint8_t *ewrm;       // [n_exits]
};

struct DevModel {
    int32_t n_sites, n_bonds, n_types, n_est, est_max_dim, max_dim;
    int32_t nsb, pad_nsb;      // sites per bond (all bonds alike), leg count 2*nsb
    double energy_offset, norm;
    const uint8_t *site_dims;  // [n_sites]
    const int32_t *bond_type;  // [n_bonds]
    const int32_t *bond_sites; // [n_bonds][nsb]
    const DevVD *types;        // [n_types]
    const double *est_coef;    // [n_est][n_sites]
    const double *est_mval;    // [n_est][n_sites][est_max_dim]
    // packed per-bond record for the kernels: sites and type in one int2
    const int2 *bond_rec;      // [n_bonds] (site0 | type<<20, site1)
    // worm tables (sse_worm.h).  Bond types with equal vertices and transitions
    // share one range of vertex codes, code = range base + vertex index; an
    // operator's entry on its k-th site carries c = code << w_lg | k.
    const uint4 *wbond;        // [n_bonds] sites two per word (u16), code base, 0
    const uint2 *wcode;        // [w_ncode] lower leg states, one byte per site; vcode | type << 10
    // distinct exit thresholds, ascending, ended by ~0 and padded to a multiple of
    // 8; then (above 8, with one of the next two) u16[256], thresholds <= bucket << 45
    const uint64_t *wthr;
    const uint32_t *wrow;      // exit rows (null: too large, or some word has no exit)
    const uint4 *wexit;        // 16-byte exit entries (null: too many codes or thresholds)
    const uint32_t *wwide;     // wide exit entries, of any table; 64-byte aligned
    int32_t w_ncode, w_lg, w_nthr, w_mw;
    int32_t w_nent;            // exit entries: ((w_ncode << w_lg) + 1) * 2 * w_mw
    int32_t w_dim;             // local dimension of every site, 0 when they differ
    int32_t w_rank, pad_w;     // bytes of the threshold search image, 0 for up to 8 thresholds
    // diagonal-update table, copied to LDS by K1: per group of bond types with
    // equal tables a 16-byte header {diagonal off, weights off, upper-state off,
    // nv | dims0 << 16}, then per group {f64 weight, i32 vertex code or -1, 0}
    // [dims0*dims1], f64 weights[nv], u16 upper leg states [nv]; from k1tab_boff the
    // bonds' sites (u16 each) and, with more than one group, the header's offset
    // (u32); offsets from the table start
    const uint8_t *k1tab;
    int32_t k1tab_bytes, k1tab_boff, k1tab_one, pad_k1;
    // lookups of the generic diagonal-update kernel, copied to LDS when they
    // fit (any bond size): per type a 32-byte header {weights off, diagonal-
    // vertex off, upper-states off, nv, dims packed one byte each}, then per
    // bond {type, sites[nsb]} (i32 each, from k1n_bond_off), then per type f64
    // weights[nv], i32 diagonal vertex codes [prod dims] (or -1) and u32 upper
    // leg states [nv] (one byte per bond position); offsets from the start
    const uint8_t *k1ntab;
    int32_t k1ntab_bytes, k1n_bond_off;
    // measurement tables (null when too large): per
    // (bond, vertex) at bond * est_dnv + vertex, the change of each estimator
    // across the vertex, f64 [n_est] (the measurement adds it for off-diagonal
    // vertices), and the vertex's sign, i8
    const double *est_dtab;
    const int8_t *est_dsgn;
    int32_t est_dnv, any_neg;  // vertex stride; some vertex has a negative sign
};

// Exit j of a scatter is the first j with r < cum[j], r = (word >> 11) * 2^-53.
// With m = word >> 11 (an integer < 2^53) and K = ceil(cum * 2^53) this is
// exactly m < K.  A model of few bond types has few distinct K (the Heisenberg
// magnet 2), so a word is reduced once to q = the number of K of the model that are
// <= m, and m < K becomes q < r with r = 1 + the index of K: exact, and independent
// of where the worm is.  The tables in LDS use q, the wide table the words.
//
// Exit entry (c, worm-1, side the worm enters by: 0 lower, 1 upper) has index
// c * 2 * w_mw + 2 * (worm - 1) + side.  Its exit word names the leg relative
// to the entering site, the port 2 * (worm - 1) + side with which the worm
// enters the next operator, and the new vertex code.
//
// Wide entry (words): thresholds r0 r1 r2, exits o0 o1 o2 o3, r3, o4 (r3 and o4 with
// four sites to a bond).  Exit j is the first with the word's top 32 bits below r_j
// (ascending; ~0: always), else the last.  Equal top bits are looked up exactly.
// An exit: selector << 4 in bits 0..6, port in 7..19, new vertex - old one in 20..30
// (two's complement); bit 31 alone: no exit here (worm_exact).
__host__ __device__ constexpr int worm_wide_words(int ns) { return ns == 4 ? 16 : 8; }
__host__ __device__ inline uint32_t worm_entry_word(uint32_t leg, uint32_t port, int step)
{
    return leg << 4 | port << 7 | ((uint32_t)step & 0x7FFu) << 20;
}
__host__ __device__ inline uint32_t worm_entry_port(uint32_t o) { return (o >> 7) & 0x1FFFu; }
__host__ __device__ inline int32_t worm_entry_step(uint32_t o) { return (int32_t)(o << 1) >> 21; }
#define kWormSpecial (1ull << 63)
// words (of 53 bits) from here on are looked up exactly
constexpr uint64_t kWormTail = (1ull << 53) - 4096u;

// Leg selector of an exit: for one and two sites per bond other | upper << 1
// (other: not the entering site), else (position - entering position) mod sites
// | upper << 2.  16 * selector is the shift that picks the next entry.
__host__ __device__ inline uint32_t worm_leg(int ns, uint32_t pos_in, uint32_t leg_out)
{
    const uint32_t n = (uint32_t)ns, up = leg_out >= n, pos = up ? leg_out - n : leg_out;
    const uint32_t rel = (pos + n - pos_in) % n;
    return n <= 2 ? rel | up << 1 : rel | up << 2;
}
// Wide exit word: selector << 4 in bits 0..6, port in 8..31, code << lg in 32..62.
__host__ __device__ inline uint64_t worm_word(uint32_t leg, uint32_t port, uint32_t code_lg)
{
    return (uint64_t)(leg << 4 | port << 8) | (uint64_t)code_lg << 32;
}

// Pointers known to address global memory.  Loads and stores through them are
// global (not flat) instructions, which count only against the vector-memory
// counter: an LDS or scalar-load wait then does not also wait for them.
template <class T>
using gmem = __attribute__((address_space(1))) T;
template <class T>
__device__ __forceinline__ gmem<T> *as_global(T *p)
{
    return (gmem<T> *)p;
}
template <class T>
__device__ __forceinline__ const gmem<T> *as_global(const T *p)
{
    return (const gmem<T> *)p;
}

struct DevWalker {
    // parameters
    int32_t model, warmup;
    double T, target_wlf, atten;
    uint64_t key;
    int64_t thermalization, init_cutoff;
    // chain state
    double avg_worm_length, num_worms;
    int64_t L, n, cap;
    uint64_t ctr;
    int64_t sweeps, measured;
    // diagnostics of the last sweep
    int64_t last_scatter;
    double last_total, last_wlf;
    int32_t error, n_sites;
    // buffers
    uint32_t *ops;    // [cap]
    int32_t *links;   // record region (lane: dense links [legs*cap]; wave: idx, records)
    uint8_t *spins;   // [n_sites]
    int32_t *first;   // [n_sites] lane: first leg; wave: first entry (global records)
    int32_t *last;    // [n_sites] lane: last leg; wave: operators on the site
    // work counters (sum over sweeps since reset)
    int64_t acc_L, acc_n, acc_W, acc_sweeps;
    int32_t meas_offset, meas_width;
    // serving slots: active walkers are swept; a finite budget of sweeps
    // (remaining >= 0) retires the walker after its last sweep + measure
    int32_t active, pending;
    int64_t remaining;
    int32_t retire;
    int32_t acc_slot;  // accumulator row (count index) of the walker's temperature slot
};

struct DevPool {
    unsigned long long next;  // bytes used
    unsigned long long size;
    char *base;
    int32_t overflow;
    int32_t status;           // bit (1 << code) per walker error code seen
    int32_t max_sites, pad;   // sites of the batch's largest lattice (slab_bytes)
    // largest LDS size the worm update could use for a walker (worm_lds_need),
    // per walker group (stream group; slot 7: every other launch)
    unsigned long long max_need[8];
};

// What the host reads after a call, in pinned host memory: the pool's error words
// and maxima, then (doubles) the measurement of a call that returns one.
constexpr size_t kReportOut = 8192;
struct PoolReport {
    int32_t overflow, status;
    unsigned long long max_need[8];
    double out[kReportOut];
};

__device__ __forceinline__ void flag_error(DevPool *pool, int code)
{
    atomicOr(&pool->status, 1 << code);
}

#define SSE_OP_BOND_SHIFT_D 11
__device__ __forceinline__ uint32_t op_bond(uint32_t op) { return op >> SSE_OP_BOND_SHIFT_D; }
__device__ __forceinline__ uint32_t op_vcode(uint32_t op) { return (op >> 1) & 1023u; }
__device__ __forceinline__ uint32_t op_make(uint32_t bond, uint32_t vcode)
{
    return 1u | (vcode << 1) | (bond << SSE_OP_BOND_SHIFT_D);
}

// ---------------------------------------------------------------- Philox4x32-10
// Counter-based generator of Salmon et al. (SC'11).  64-bit word i of a
// walker's stream with key k: block b = i/2 with counter (lo32 b, hi32 b, 0, 0)
// and key (lo32 k, hi32 k); word = out0|out1<<32 for even i, out2|out3<<32 odd.
__device__ __forceinline__ void philox_block(uint64_t b, uint64_t key, uint32_t &o0, uint32_t &o1,
                                             uint32_t &o2, uint32_t &o3)
{
    uint32_t c0 = (uint32_t)b, c1 = (uint32_t)(b >> 32), c2 = 0u, c3 = 0u;
    uint32_t k0 = (uint32_t)key, k1 = (uint32_t)(key >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    o0 = c0; o1 = c1; o2 = c2; o3 = c3;
}

__device__ __forceinline__ double word_to_float(uint64_t w) { return (double)(w >> 11) * 0x1.0p-53; }

// Per-lane sequential stream with a one-block cache.
struct LaneRng {
    uint64_t key, ctr, blk;
    uint32_t o0, o1, o2, o3;
    __device__ void init(uint64_t k, uint64_t c)
    {
        key = k;
        ctr = c;
        blk = ~0ull;
    }
    __device__ __forceinline__ uint64_t next()
    {
        uint64_t b = ctr >> 1;
        if (b != blk) {
            philox_block(b, key, o0, o1, o2, o3);
            blk = b;
        }
        uint64_t w = (ctr & 1) ? ((uint64_t)o2 | ((uint64_t)o3 << 32))
                               : ((uint64_t)o0 | ((uint64_t)o1 << 32));
        ++ctr;
        return w;
    }
    __device__ __forceinline__ double next_float() { return word_to_float(next()); }
    // rand(1:s) - 1, Lemire's nearly divisionless method on 64-bit words
    __device__ __forceinline__ uint64_t range(uint64_t s)
    {
        uint64_t x = next();
        uint64_t l = x * s;
        uint64_t h = __umul64hi(x, s);
        if (l < s) {
            uint64_t t = (0ull - s) % s;
            while (l < t) {
                x = next();
                l = x * s;
                h = __umul64hi(x, s);
            }
        }
        return h;
    }
};

// ---------------------------------------------------------------- tanh
// Worm-number controller tanh.  Evaluated by exactly this sequence of IEEE
// operations (no contraction): Cody-Waite reduction x = k ln2 + r and the
// degree-16 Taylor polynomial of expm1(r); tanh(x) = e/(e+2), e = expm1(2|x|).
__device__ __forceinline__ double sse_expm1(double x)
{
    const double C[16] = {
        0x1.0000000000000p+0, 0x1.0000000000000p-1, 0x1.5555555555555p-3, 0x1.5555555555555p-5,
        0x1.1111111111111p-7, 0x1.6c16c16c16c17p-10, 0x1.a01a01a01a01ap-13, 0x1.a01a01a01a01ap-16,
        0x1.71de3a556c734p-19, 0x1.27e4fb7789f5cp-22, 0x1.ae64567f544e4p-26, 0x1.1eed8eff8d898p-29,
        0x1.6124613a86d09p-33, 0x1.93974a8c07c9dp-37, 0x1.ae7f3e733b81fp-41, 0x1.ae7f3e733b81fp-45};
    if (x == 0.0)
        return x;
    double kf = rint(x * 0x1.71547652b82fep+0);
    double r = (x - kf * 0x1.62e42fee00000p-1) - kf * 0x1.a39ef35793c76p-33;
    double p = C[15];
#pragma unroll
    for (int j = 14; j >= 0; --j)
        p = p * r + C[j];
    double em1 = p * r;
    int k = (int)kf;
    if (k == 0)
        return em1;
    double two_k = ldexp(1.0, k);
    return two_k * em1 + (two_k - 1.0);
}

__device__ __forceinline__ double sse_tanh(double x)
{
    double ax = fabs(x);
    if (!(ax < 22.0))
        return copysign(1.0, x);
    if (ax < 0x1p-28)
        return x;
    double e = sse_expm1(2.0 * ax);
    double t = e / (e + 2.0);
    return copysign(t, x);
}

// Natural logarithm of the parallel-tempering exchange test: x = m 2^e with
// m in (sqrt(1/2), sqrt(2)], log(m) = 2 atanh(s) = 2 sum_j s^(2j+1)/(2j+1),
// s = (m-1)/(m+1), twelve terms (|s| <= 0.1716).  Exactly this sequence of
// IEEE operations, so the host-side checker decides every exchange the same
// way.  x positive, finite, normal.
__device__ __forceinline__ double sse_log(double x)
{
    const uint64_t bits = (uint64_t)__double_as_longlong(x);
    int e = (int)((bits >> 52) & 0x7ff) - 1023;
    double m = __longlong_as_double((long long)((bits & 0x000fffffffffffffull) | 0x3ff0000000000000ull));
    if (m > 0x1.6a09e667f3bcdp+0) {
        m = m * 0.5;
        e += 1;
    }
    const double s = (m - 1.0) / (m + 1.0);
    const double z = s * s;
    double p = 1.0 / 23.0;
#pragma unroll
    for (int k = 21; k >= 1; k -= 2)
        p = p * z + 1.0 / (double)k;
    const double lm = 2.0 * s * p;
    const double ef = (double)e;
    return ef * 0x1.62e42fee00000p-1 + (lm + ef * 0x1.a39ef35793c76p-33);
}

// Philox4x32-10 of a full 128-bit counter block.
__device__ __forceinline__ void philox_block4(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                              uint64_t key, uint32_t &o0, uint32_t &o1)
{
    uint32_t k0 = (uint32_t)key, k1 = (uint32_t)(key >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    o0 = c0;
    o1 = c1;
}

// Worm-number controller and WormLengthFraction (sse.jl:200-217).
__device__ __forceinline__ void worm_controller(DevWalker &w, double total, bool thermalized)
{
    w.last_total = total;
    w.last_wlf = __longlong_as_double(0x7ff8000000000000ll);
    if (thermalized && w.n != 0)
        w.last_wlf = total / (double)w.n;
    double avg = total / ceil(w.num_worms);
    if (!thermalized) {
        w.avg_worm_length += w.atten * (avg - w.avg_worm_length);
        double target = w.target_wlf * (double)w.n / w.avg_worm_length;
        w.num_worms += w.atten * (target - w.num_worms + 100.0 * sse_tanh(target - w.num_worms));
        if (w.atten != 0.0) {
            double hi = 1.0 + (double)w.n / 2.0;
            double x = w.num_worms;
            w.num_worms = x > hi ? hi : (x < 1.0 ? 1.0 : x);
        }
    }
}

// WormLengthFraction (sse.jl:200-202) of the last sweep into the slot's
// accumulator {sum, sum of squares, count}: the reference measures it in
// every thermalized sweep with n != 0 (last_wlf is NaN otherwise).  The slot
// follows the temperature under parallel tempering, like the other sums.
__device__ __forceinline__ void worm_fraction_accumulate(const DevWalker &w, double *wlf)
{
    const double v = w.last_wlf;
    if (v == v) {
        double *q = wlf + 3 * (size_t)w.acc_slot;
        q[0] += v;
        q[1] += v * v;
        q[2] += 1.0;
    }
}

// Growth rule of the cutoff (sse.jl:138-145): n >= L/2 -> L = floor(1.5 L + 100).
__device__ __forceinline__ int64_t grown_cutoff(int64_t L) { return (3 * L) / 2 + 100; }

// Capacity of a fresh slab for cutoff L: two further growth steps of headroom.
__device__ __host__ __forceinline__ int64_t slab_capacity(int64_t L)
{
    int64_t c = L < 64 ? 64 : L;
    c = (3 * c) / 2 + 100;
    c = (3 * c) / 2 + 100;
    return (c + 63) & ~(int64_t)63;
}

// Bytes of a worm code in global records: 2, or 4 when the codes need them.
__device__ __host__ __forceinline__ int worm_code_bytes(const DevModel &m)
{
    return ((int64_t)m.w_ncode << m.w_lg) <= 65535 ? 2 : 4;
}

// Slab of a walker: ops[cap], then the record region.  Lane kernels: dense
// links.  Wave kernels: idx (4 bytes per slot and bond site), then the global
// worm records (a 4-byte partner and a worm code per entry, one entry per slot
// and bond site and two more per lattice site of the batch's largest lattice, so
// that a slot's slab serves every model of its shape); the entry words of the
// LDS layouts, 4 or 8 bytes per slot, take the same place.
__device__ __host__ __forceinline__ uint64_t slab_bytes(int64_t cap, const DevModel &m, int sites, bool wave)
{
    const uint64_t ns = (uint64_t)m.nsb, c = (uint64_t)cap, cb = (uint64_t)worm_code_bytes(m);
    const uint64_t rec = wave ? 4u * ns * c + (4u + cb) * (ns * c + 2u * (uint64_t)sites) : 8u * ns * c;
    return (c * 4u + rec + 255u) & ~(uint64_t)255u;
}

// Bump allocation from the batch's slab pool; returns nullptr on exhaustion.
__device__ __forceinline__ char *pool_alloc(DevPool *pool, uint64_t bytes)
{
    unsigned long long off = atomicAdd(&pool->next, (unsigned long long)bytes);
    if (off + bytes > pool->size) {
        atomicExch(&pool->overflow, 1);
        return nullptr;
    }
    return pool->base + off;
}
