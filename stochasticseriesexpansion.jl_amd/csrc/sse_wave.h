// sse_wave.h -- one wavefront (64 lanes) per walker.
//
// K1 wave_diag_vlist_kernel: diagonal update (sse.jl:137-191) and vertex-list
//   construction (vertex_list.jl:15-54) fused into one streaming pass over the
//   operator string, 64 slots per step:
//   * draw offsets: slot types (identity 2 draws, diagonal 1, off-diagonal 0)
//     are fixed before the update, so every lane's Philox words follow from a
//     ballot prefix count; the words come from a 256-word LDS buffer that all
//     lanes refill cooperatively.
//   * spins at identity slots and places along the sites: every lane ORs its
//     bit into per-site LDS lane masks (one for bond position 0, one for 1);
//     "latest earlier operator on site s" is the highest lower bit of the mask
//     filtered by the off-diagonal (spins) or final non-identity (places) set.
//   * the acceptance tests depend on the running operator count n, but each
//     is monotone in n and n moves by at most one per slot: a lane's decision
//     is fixed if it agrees at both ends of its window [n0-lane, n0+lane];
//     the rare ambiguous lanes are resolved in slot order with the exact n.
//   * a Lemire rejection of the bond draw (probability Nb/2^64) would shift
//     later draw offsets; that chunk is then processed slot by slot.
// K2 wave_worm_kernel: worm_update (sse.jl:193-303), sse_worm.h.
// K3 wave_measure_kernel: measure (sse.jl:70-87,305-376) with the estimator
//   running sums as wave prefix sums.
#pragma once
#include <type_traits>
#include <vector>

#include "sse_common.h"
#include "sse_lane.h"

struct WaveConfig {
    int max_sites = 0;
    int max_warmup = 0;
    size_t lds_k1 = 0, lds_k2 = 0, lds_k3 = 0;
    size_t lds_limit = 65536;  // device limit on dynamic LDS per workgroup
    int rec_mode = 0;          // SSE_OPT_WORM_RECORDS (worm_walker's mode)
    size_t lds_k2_fixed = 0;   // worm-kernel LDS per walker set by the caller (0 = sized here)
    size_t lds_k2_group[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // per stream group (0 = lds_k2)
    int fuse_measure = 0;      // measuring sweeps: worm update + measurement in one kernel
    int generic = 0;           // some model has bonds of other than two sites: sse_wave_n.h kernels
    size_t lds_k1n = 0;        // LDS of the generic diagonal-update kernel
};

__device__ __forceinline__ uint64_t below_mask(int lane) { return lane ? (~0ull >> (64 - lane)) : 0ull; }
__device__ __forceinline__ uint64_t above_mask(int lane) { return lane >= 63 ? 0ull : (~0ull << (lane + 1)); }
__device__ __forceinline__ int hi_bit(uint64_t x) { return 63 - __clzll((long long)x); }
__device__ __forceinline__ int popc(uint64_t x) { return __popcll(x); }

// Orders the LDS accesses of the lanes of a one-wave workgroup.  The LDS runs
// a wave's instructions in order, so only code motion must be prevented; unlike
// __syncthreads this does not wait for global loads still in flight.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Philox words of one walker staged in LDS: buf holds words
// [bbase, bbase+256) and the next word to draw is bbase+off.  All members are
// wave-uniform; every call must be made by the whole wave.
template <int NW>
__device__ __noinline__ void wave_refill(uint64_t *buf, uint64_t key, uint64_t base)
{
    const int l = threadIdx.x;
    wave_lds_sync();
#pragma unroll
    for (int j = l; j < NW / 2; j += 64) {
        uint32_t o0, o1, o2, o3;
        philox_block((base >> 1) + (uint64_t)j, key, o0, o1, o2, o3);
        buf[2 * j] = (uint64_t)o0 | ((uint64_t)o1 << 32);
        buf[2 * j + 1] = (uint64_t)o2 | ((uint64_t)o3 << 32);
    }
    wave_lds_sync();
}

template <int NW>
struct WaveStreamT {
    uint64_t *buf;
    uint64_t key, bbase;
    uint32_t off;  // next word is bbase + off; off > 256 marks an empty buffer
    __device__ void init(uint64_t *b, uint64_t k, uint64_t c)
    {
        buf = b;
        key = k;
        bbase = c;
        off = 1024;  // empty: the first ensure() refills at c
    }
    __device__ __forceinline__ uint64_t ctr() const { return bbase + off - (off >= 1024 ? 1024 : 0); }
    // make words [ctr, ctr+need) resident (need <= 255)
    __device__ __forceinline__ void ensure(uint32_t need)
    {
        if (off >= 1024) {  // empty: start at the pending counter bbase
            const uint64_t c = bbase;
            bbase = c & ~1ull;
            off = (uint32_t)(c - bbase);
            wave_refill<NW>(buf, key, bbase);
        } else if (off + need > NW) {
            const uint64_t c = bbase + off;
            bbase = c & ~1ull;
            off = (uint32_t)(c - bbase);
            wave_refill<NW>(buf, key, bbase);
        }
    }
    // word k positions after the next one (after ensure)
    __device__ __forceinline__ uint64_t peek(uint32_t k) const { return buf[off + k]; }
    __device__ __forceinline__ void advance(uint32_t k) { off += k; }
    __device__ __forceinline__ uint64_t next()
    {
        ensure(1);
        uint64_t w = buf[off];
        ++off;
        return w;
    }
    __device__ __forceinline__ double next_float() { return word_to_float(next()); }
    __device__ __forceinline__ uint64_t range(uint64_t s)
    {
        uint64_t x = next();
        uint64_t lo = x * s, hi = __umul64hi(x, s);
        if (lo < s) {
            uint64_t t = (0ull - s) % s;
            while (lo < t) {
                x = next();
                lo = x * s;
                hi = __umul64hi(x, s);
            }
        }
        return hi;
    }
};

typedef WaveStreamT<256> WaveStream;
// The state refresh's Philox words in registers: lane l holds word bbase + l of
// the walker's stream (bbase even).  A wave-uniform draw is two v_readlane with a
// scalar index; lanes that draw different words read them with ds_bpermute.  No
// LDS and no barrier; all members except the two per-lane words are wave-uniform
// and every call is made by the whole wave.
struct K2RegStream {
    static constexpr uint32_t kNW = 64;
    uint32_t wlo, whi;
    uint64_t key, bbase;
    uint32_t off;  // next word is bbase + off; off >= 1024 marks an empty buffer
    __device__ void init(uint64_t k, uint64_t c)
    {
        key = k;
        bbase = c;
        off = 1024;
    }
    __device__ __forceinline__ void fill()
    {
        const uint32_t lane = threadIdx.x;
        uint32_t o0, o1, o2, o3;
        philox_block((bbase >> 1) + (lane >> 1), key, o0, o1, o2, o3);
        wlo = (lane & 1u) ? o2 : o0;
        whi = (lane & 1u) ? o3 : o1;
    }
    __device__ __forceinline__ uint64_t ctr() const { return bbase + off - (off >= 1024 ? 1024 : 0); }
    // make words [ctr, ctr+need) resident (need <= 63)
    __device__ __forceinline__ void ensure(uint32_t need)
    {
        if (off >= 1024) {
            const uint64_t c = bbase;
            bbase = c & ~1ull;
            off = (uint32_t)(c - bbase);
            fill();
        } else if (off + need > kNW) {
            const uint64_t c = bbase + off;
            bbase = c & ~1ull;
            off = (uint32_t)(c - bbase);
            fill();
        }
    }
    // word k (wave-uniform, < kNW) of the buffer
    __device__ __forceinline__ uint64_t word_at(uint32_t k) const
    {
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)wlo, (int)k);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)whi, (int)k);
        return ((uint64_t)hi << 32) | lo;
    }
    // word k positions after the next one, k per lane (after ensure)
    __device__ __forceinline__ uint64_t peek(uint32_t k) const
    {
        const int a = (int)((off + k) << 2);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(a, (int)wlo);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(a, (int)whi);
        return ((uint64_t)hi << 32) | lo;
    }
    __device__ __forceinline__ void advance(uint32_t k) { off += k; }
    __device__ __forceinline__ uint64_t next()
    {
        ensure(1);
        const uint64_t x = word_at(off);
        ++off;
        return x;
    }
    __device__ __forceinline__ uint64_t range(uint64_t s)
    {
        uint64_t x = next();
        uint64_t lo = x * s, hi = __umul64hi(x, s);
        if (lo < s) {
            uint64_t t = (0ull - s) % s;
            while (lo < t) {
                x = next();
                lo = x * s;
                hi = __umul64hi(x, s);
            }
        }
        return hi;
    }
};
__device__ __forceinline__ uint32_t uni(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uni64(uint64_t x)
{
    return (uint64_t)uni((uint32_t)x) | ((uint64_t)uni((uint32_t)(x >> 32)) << 32);
}

#include "sse_worm.h"

// LDS layout of K1 (per workgroup = one walker):
//   rbuf  u64[256]        Philox words
//   tm    {u64, u64}[N]   per-site lane masks, bond positions 0 and 1
//   cnt   u32[N]          operators on the site so far
//   sp    u8[N]           spins at the current slot
__host__ __device__ inline size_t k1_lds_bytes(int N)
{
    size_t b = 2048 + 16 * (size_t)N + 4 * (size_t)N + (size_t)N;
    return (b + 15) & ~(size_t)15;
}

constexpr int K1_BLOCK = 16;  // 64-slot chunks per block of operator-string loads

// Model lookups of the diagonal update / vertex list: from the LDS copy of
// DevModel::k1tab (K1Staged), or from the model's global arrays (K1Global).  A
// type token comes with a bond: K1Staged's is the byte offset of the type's
// header; with one table for all bonds (kOne: bond types with equal weights,
// diagonal vertices and upper states share one) the header is in registers.
struct K1Bond {
    uint32_t s0, s1, t;
};
struct K1Weight {
    double w;   // weight of the diagonal vertex, 0 without one
    int32_t dv; // its vertex code, -1 without one
};
struct K1Global {
    static constexpr bool kChecked = true;  // lookups need indexes in range
    const DevModel *m;
    __device__ __forceinline__ void stage(const DevModel &) {}
    __device__ __forceinline__ K1Bond bond(uint32_t b) const
    {
        const int2 r = m->bond_rec[b];
        return K1Bond{(uint32_t)r.x & 0xFFFFFu, (uint32_t)r.y, (uint32_t)r.x >> 20};
    }
    __device__ __forceinline__ uint32_t nv(uint32_t t) const { return (uint32_t)m->types[t].nv; }
    __device__ __forceinline__ K1Weight diag(uint32_t t, uint32_t v0, uint32_t v1) const
    {
        const DevVD &vd = m->types[t];
        const int32_t dv = vd.diag_vertex[(v0 - 1u) + (uint32_t)vd.dims0 * (v1 - 1u)];
        return K1Weight{dv < 0 ? 0.0 : vd.weights[dv >> 1], dv};
    }
    __device__ __forceinline__ double weight(uint32_t t, uint32_t v) const { return m->types[t].weights[v]; }
    __device__ __forceinline__ uint32_t upper(uint32_t t, uint32_t v) const
    {
        const uint8_t *ls = m->types[t].leg_states + 4 * v;
        return ls[2] | ((uint32_t)ls[3] << 8);
    }
};
template <bool kOne>
struct K1Staged {
    static constexpr bool kChecked = false;  // an index out of range reads another LDS word
    uint32_t kt;                             // LDS byte address of the k1tab copy
    uint32_t boff;                           // bond records in it
    uint32_t h0, h1, h2, h3;                 // the only type's header (kOne)
    // copy the model's k1tab into LDS (whole wave)
    __device__ __forceinline__ void stage(const DevModel &m)
    {
        worm_copy_table(kt, m.k1tab, (size_t)m.k1tab_bytes);
        boff = (uint32_t)m.k1tab_boff;
        const uint32_t *g = (const uint32_t *)m.k1tab;
        h0 = uni(g[0]);
        h1 = uni(g[1]);
        h2 = uni(g[2]);
        h3 = uni(g[3]);
    }
    __device__ __forceinline__ K1Bond bond(uint32_t b) const
    {
        if constexpr (kOne) {
            const uint32_t s = *lds_at<lds_u32>(kt + boff + 4u * b);
            return K1Bond{s & 0xFFFFu, s >> 16, 0u};
        } else {
            const uint64_t s = *lds_at<lds_u64>(kt + boff + 8u * b);
            return K1Bond{(uint32_t)s & 0xFFFFu, (uint32_t)s >> 16, (uint32_t)(s >> 32)};
        }
    }
    __device__ __forceinline__ u32x4 hdr(uint32_t t) const
    {
        if constexpr (kOne)
            return u32x4{h0, h1, h2, h3};
        else
            return *lds_at<lds_u32x4>(kt + t);
    }
    __device__ __forceinline__ uint32_t nv(uint32_t t) const { return hdr(t).w & 0xFFFFu; }
    __device__ __forceinline__ K1Weight diag(uint32_t t, uint32_t v0, uint32_t v1) const
    {
        const u32x4 h = hdr(t);
        const uint32_t i = (v0 - 1u) + __umul24(h.w >> 16, v1 - 1u);
        const u32x4 x = *lds_at<lds_u32x4>(kt + h.x + 16u * i);
        return K1Weight{__hiloint2double((int)x.y, (int)x.x), (int32_t)x.z};
    }
    __device__ __forceinline__ double weight(uint32_t t, uint32_t v) const
    {
        const uint64_t x = *lds_at<lds_u64>(kt + hdr(t).y + 8u * v);
        return __longlong_as_double((long long)x);
    }
    __device__ __forceinline__ uint32_t upper(uint32_t t, uint32_t v) const
    {
        return *lds_at<lds_u16>(kt + hdr(t).z + 2u * v);
    }
};

// LDS bytes of K1 with the model's lookups staged behind the base layout
__host__ __device__ inline size_t k1_lds_staged(int N, int k1tab_bytes)
{
    return k1_lds_bytes(N) + (size_t)k1tab_bytes;
}

// Slot-by-slot processing of one chunk (reference order).  Used when a bond
// draw of the chunk hits a Lemire rejection, and when forced for validation.
// Emits the same idx words as the parallel path.
__device__ void k1_serial_chunk(DevWalker &w, const DevModel &m, WaveStream &rs, int64_t base,
                                int64_t &n, double pm_raw, double pr_raw, bool do_diag, bool do_vl,
                                uint8_t *sp, uint32_t *cnt)
{
    const int lane = threadIdx.x;
    const int64_t L = w.L;
    uint32_t *gidx = (uint32_t *)w.links;
    for (int i = 0; i < 64 && base + i < L; ++i) {
        const int64_t p = base + i;
        uint32_t op = w.ops[p];
        uint32_t nop = op;
        if (do_diag) {
            if (op == 0u) {
                uint32_t b = (uint32_t)rs.range((uint64_t)m.n_bonds);
                int2 br = m.bond_rec[b];
                const DevVD &vd = m.types[br.x >> 20];
                int s0 = br.x & 0xFFFFF, s1 = br.y;
                int idx = (sp[s0] - 1) + vd.dims0 * (sp[s1] - 1);
                int32_t dv = vd.diag_vertex[idx];
                double wgt = dv < 0 ? 0.0 : vd.weights[dv >> 1];
                double p_make = pm_raw / (double)(L - n);
                if (rs.next_float() < p_make * wgt) {
                    nop = op_make(b, (uint32_t)dv);
                    n += 1;
                }
            } else {
                uint32_t vc = op_vcode(op);
                int2 br = m.bond_rec[op_bond(op)];
                const DevVD &vd = m.types[br.x >> 20];
                if (vc & 1u) {
                    double wgt = vd.weights[vc >> 1];
                    double p_remove = (double)(L - n + 1) * pr_raw;
                    if (rs.next_float() * wgt < p_remove) {
                        nop = 0u;
                        n -= 1;
                    }
                } else {
                    const uint8_t *ls = vd.leg_states + 4 * (vc >> 1);
                    __syncthreads();
                    if (lane == 0) {
                        sp[br.x & 0xFFFFF] = ls[2];
                        sp[br.y] = ls[3];
                    }
                    __syncthreads();
                }
            }
        }
        if (do_vl && nop != 0u) {
            int2 br = m.bond_rec[op_bond(nop)];
            const int sites[2] = {br.x & 0xFFFFF, br.y};
            __syncthreads();
            if (lane == 0)
                for (int k = 0; k < 2; ++k) {
                    gidx[2 * p + k] = cnt[sites[k]];
                    cnt[sites[k]] += 1u;
                }
            __syncthreads();
        }
        if (lane == 0 && nop != op)
            w.ops[p] = nop;
    }
    __syncthreads();
}

// k1_serial_chunk out of line, everything by value (the caller's walker copy
// and stream stay in registers; the rare path gets a call instead of inlined
// code in the chunk loop).  Returns the counts and the stream position.
struct K1SerialOut {
    int64_t n;
    uint64_t bbase;
    uint32_t off;
};
__device__ __noinline__ K1SerialOut k1_serial_chunk_ool(DevWalker w, const DevModel *m, WaveStream rs,
                                                        int64_t base, int64_t n, double pm_raw,
                                                        double pr_raw, bool do_diag, bool do_vl,
                                                        uint8_t *sp, uint32_t *cnt)
{
    k1_serial_chunk(w, *m, rs, base, n, pm_raw, pr_raw, do_diag, do_vl, sp, cnt);
    return K1SerialOut{n, rs.bbase, rs.off};
}

// bits of a per-lane mask below this lane
__device__ __forceinline__ uint32_t bits_below(uint64_t x)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(x >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)x, 0u));
}
// value of lane q's x (all lanes active)
__device__ __forceinline__ uint32_t from_lane(uint32_t x, uint32_t q)
{
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(q << 2), (int)x);
}

// phases: 1 diagonal update, 2 vertex list, 8 force the slot-by-slot path.
// warm >= 0: init warm-up round (diagonal only; walkers with fewer warm-up
// sweeps are skipped).
//
// A chunk of 64 slots is a chain of LDS lookups (words -> bond -> lane masks ->
// states -> weight), a decision and the stores; with few walkers its latency
// bounds the kernel, with many the instructions it issues.  So every lane runs
// one path, whatever its slot holds, states of earlier operators come straight
// from their lanes' registers, and the make test multiplies where the
// reference divides: u < (pm / d) w is decided by u d against pm w unless the
// two are within 2^-40 of each other, and then exactly, in slot order.
// Measured on 16x16 Heisenberg at beta = 8 (137 chunks), one wave to a SIMD:
// 300 -> 199 us per sweep against divides, branches by slot kind and a table
// per lookup; 383 -> 265 us with 1536 walkers.  Blocks of 8 chunks at three waves
// per SIMD (168 registers) against 16 at two (193): 194 and 268 us, no gain.
template <class Tab>
__device__ __forceinline__ void k1_walker_t(DevWalker *W, const DevModel *models, DevPool *pool, int wi,
                                            int phases, int warm, char *lds, Tab tab, int grp)
{
    const int lane = threadIdx.x;
    DevWalker w = W[wi];
    if (w.error)
        return;
    // warm-up rounds touch pending walkers only; a sweep skips inactive
    // walkers and slots whose sweep budget ran out (retire set)
    if (warm >= 0 ? (warm >= w.warmup || !w.pending) : (!w.active || w.retire))
        return;
    const DevModel &m = models[w.model];
    tab.stage(m);
    const int N = m.n_sites;
    uint64_t *rbuf = (uint64_t *)lds;
    uint32_t *cnt = (uint32_t *)(lds + 2048 + 16 * (size_t)N);
    uint8_t *sp = (uint8_t *)(cnt + N);
    const uint32_t lbase = (uint32_t)(uintptr_t)(lds_u8 *)lds;
    const uint32_t tmb = lbase + 2048u, cntb = tmb + 16u * (uint32_t)N, spb = cntb + 4u * (uint32_t)N;

    const bool do_diag = phases & 1;
    const bool do_vl = (phases & 2) && warm < 0;
    const bool force_serial = phases & 8;

    for (int i = lane; i < N; i += 64) {
        *lds_at<lds_u32x4>(tmb + 16u * i) = u32x4{0u, 0u, 0u, 0u};
        cnt[i] = 0u;
        sp[i] = w.spins[i];
    }
    // growth check, no draws (sse.jl:138-145)
    if (do_diag && (double)w.n >= (double)w.L * 0.5) {
        int64_t nl = grown_cutoff(w.L);
        if (nl > w.cap) {
            int64_t cap = slab_capacity(nl);
            unsigned long long sp_addr = 0;
            if (lane == 0)
                sp_addr = (unsigned long long)pool_alloc(pool, slab_bytes(cap, m, pool->max_sites, true));
            uint32_t lo = __shfl((uint32_t)sp_addr, 0), hi = __shfl((uint32_t)(sp_addr >> 32), 0);
            char *s = (char *)(((unsigned long long)hi << 32) | lo);
            if (!s) {
                if (lane == 0) {
                    W[wi].error = SSE_ERR_OOM;
                    flag_error(pool, SSE_ERR_OOM);
                }
                return;
            }
            uint32_t *nops = (uint32_t *)s;
            for (int64_t p = lane; p < w.L; p += 64)
                nops[p] = w.ops[p];
            w.ops = nops;
            w.links = (int32_t *)(s + (size_t)cap * 4);
            w.cap = cap;
        }
        for (int64_t p = w.L + lane; p < nl; p += 64)
            w.ops[p] = 0u;
        w.L = nl;
    }
    __syncthreads();

    WaveStream rs;
    rs.init(rbuf, w.key, w.ctr);
    const double pm_raw = (double)m.n_bonds / w.T;
    const double pr_raw = w.T / (double)m.n_bonds;
    const uint32_t L = (uint32_t)w.L;
    uint32_t n0 = uni((uint32_t)w.n);
    gmem<uint64_t> *gidx = as_global((uint64_t *)w.links);  // both sites' idx words of a slot
    gmem<uint32_t> *ops = as_global(w.ops);

    // The operator string reaches the chunks in blocks of K1_BLOCK chunks held
    // in registers (lane l: slot l of each chunk): a block's loads are issued a
    // whole block ahead and moved into place when the block starts, so the loop
    // waits on global memory once per block.  (A load consumed in the next
    // chunk would be waited on together with the chunk's global stores: the
    // memory counter does not order loads against stores.)  K1 writes only the
    // current chunk's slots, so the loaded values of later chunks stay current.
    // The chunk index within the block is wave-uniform, so cur[slot] is a
    // register-indexed move.  Model scalars are read once, before the loop,
    // for the same reason (a read inside it would wait for the stores).
    const uint32_t nbonds = uni((uint32_t)m.n_bonds);
    uint32_t cur[K1_BLOCK], pf[K1_BLOCK];
#pragma unroll
    for (int u = 0; u < K1_BLOCK; ++u) {
        const uint32_t q = 64u * u + lane;
        cur[u] = q < L ? ops[q] : 0u;
    }
#pragma unroll
    for (int u = 0; u < K1_BLOCK; ++u) {
        const uint32_t q = 64u * (K1_BLOCK + u) + lane;
        pf[u] = q < L ? ops[q] : 0u;
    }
    bool bad = false;
    for (uint32_t base = 0; base < L; base += 64) {
        const uint32_t p = base + lane;
        const bool valid = p < L;
        const uint32_t chunk = base >> 6;
        const int slot = (int)uni(chunk % K1_BLOCK);
        if (slot == 0 && chunk > 0) {
#pragma unroll
            for (int u = 0; u < K1_BLOCK; ++u)
                cur[u] = pf[u];
#pragma unroll
            for (int u = 0; u < K1_BLOCK; ++u) {
                const uint32_t q = base + 64u * (K1_BLOCK + u) + lane;
                pf[u] = q < L ? ops[q] : 0u;
            }
        }
        const uint32_t op = cur[slot];
        const uint32_t vc = op_vcode(op), vx = vc >> 1;
        const bool ident = valid && op == 0u;
        const bool dia = op != 0u && (vc & 1u);
        const bool offd = op != 0u && !(vc & 1u);
        const uint64_t identm = __ballot(ident), diam = __ballot(dia), offm = __ballot(offd);
        uint32_t b = op_bond(op);
        // an operator outside the model (a corrupted string): reported when the
        // walker ends, its bond replaced by one that exists
        bad |= b >= nbonds;
        b = b < nbonds ? b : 0u;
        double u = 0.0;
        if (do_diag) {
            // draws of the slots before this one: two per identity, one per
            // diagonal operator
            const uint32_t D = 2u * (uint32_t)popc(identm) + (uint32_t)popc(diam);
            const uint32_t off = 2u * bits_below(identm) + bits_below(diam);
            // two words more, which the lanes behind the last draw read
            rs.ensure(D + 2u);
            // identity: bond, then the test's number; diagonal: the number
            const uint64_t x0 = rs.peek(off), x1 = rs.peek(off + 1u);
            // rand(1:n_bonds): high half of word * n_bonds, rejected where the low
            // half could be below 2^64 mod n_bonds
            const uint64_t pl = (uint64_t)(uint32_t)x0 * nbonds;
            const uint64_t ph = (uint64_t)(uint32_t)(x0 >> 32) * nbonds + (pl >> 32);
            const bool maybe = ident && (uint32_t)ph == 0u && (uint32_t)pl < nbonds;
            if (__builtin_expect(force_serial || wave_any(maybe), 0)) {
                bad |= op != 0u && vx >= tab.nv(tab.bond(b).t);
                if (wave_any(bad))  // its lookups take indexes as they are
                    break;
                const K1SerialOut so = k1_serial_chunk_ool(w, &m, rs, base, n0, pm_raw, pr_raw, do_diag,
                                                           do_vl, sp, cnt);
                n0 = uni((uint32_t)so.n);
                rs.bbase = so.bbase;
                rs.off = so.off;
                continue;
            }
            b = ident ? (uint32_t)(ph >> 32) : b;
            u = word_to_float(ident ? x1 : x0);
            rs.advance(D);
        } else if (force_serial) {
            bad |= op != 0u && vx >= tab.nv(tab.bond(b).t);
            if (wave_any(bad))
                break;
            const K1SerialOut so = k1_serial_chunk_ool(w, &m, rs, base, n0, pm_raw, pr_raw, do_diag,
                                                       do_vl, sp, cnt);
            n0 = uni((uint32_t)so.n);
            rs.bbase = so.bbase;
            rs.off = so.off;
            continue;
        }

        const K1Bond br = tab.bond(b);
        const uint32_t s0 = br.s0, s1 = br.s1;
        uint32_t vi = vx;
        if (Tab::kChecked) {
            const uint32_t nv = tab.nv(br.t);
            bad |= op != 0u && vx >= nv;
            vi = vx < nv ? vx : 0u;
        } else {
            bad |= op != 0u && vx >= tab.nv(br.t);
        }
        // per-site lane masks of the slots that hold or may get an operator
        const bool has = op != 0u || (ident && do_diag);
        const uint32_t t0 = tmb + 16u * s0, t1 = tmb + 16u * s1;
        if (has) {
            const uint32_t half = (lane >> 5) * 4u, bit = 1u << (lane & 31);
            atomicOr((uint32_t *)(lds + (t0 - lbase) + half), bit);
            atomicOr((uint32_t *)(lds + (t1 - lbase) + 8u + half), bit);
        }
        const uint32_t up = tab.upper(br.t, vi);      // an off-diagonal operator's states after it
        double wgt = tab.weight(br.t, vi);            // a diagonal operator's weight
        const uint32_t sp0 = *lds_at<lds_u8>(spb + s0), sp1 = *lds_at<lds_u8>(spb + s1);
        const uint32_t c0 = *lds_at<lds_u32>(cntb + 4u * s0), c1 = *lds_at<lds_u32>(cntb + 4u * s1);
        wave_lds_sync();
        const u32x4 ma = *lds_at<lds_u32x4>(t0), mc = *lds_at<lds_u32x4>(t1);
        const uint64_t a0 = (uint64_t)ma.x | (uint64_t)ma.y << 32, a1 = (uint64_t)ma.z | (uint64_t)ma.w << 32;
        const uint64_t e0 = (uint64_t)mc.x | (uint64_t)mc.y << 32, e1 = (uint64_t)mc.z | (uint64_t)mc.w << 32;
        const uint64_t A = a0 | a1, C = e0 | e1;  // lanes on site 0, on site 1
        const uint64_t below = below_mask(lane), above = above_mask(lane);

        uint64_t plus = 0, minus = 0;
        uint32_t fop = op;
        if (do_diag) {
            // states at the slot: of the latest off-diagonal operator on the
            // site earlier in the chunk, else at the chunk's start
            const uint64_t oa = A & offm & below, oc = C & offm & below;
            const uint32_t qa = oa ? (uint32_t)hi_bit(oa) : 0u, qc = oc ? (uint32_t)hi_bit(oc) : 0u;
            const uint32_t ua = from_lane(up, qa), uc = from_lane(up, qc);
            const uint32_t v0 = oa ? (((a0 >> qa) & 1ull) ? ua & 255u : ua >> 8) : sp0;
            const uint32_t v1 = oc ? (((e0 >> qc) & 1ull) ? uc & 255u : uc >> 8) : sp1;
            const K1Weight dw = tab.diag(br.t, v0, v1);
            wgt = ident ? dw.w : wgt;
            // the window of n that earlier slots of the chunk leave open; each
            // test is monotone in n, so a decision at both ends holds between
            const uint32_t room = L - n0 + (ident ? 0u : 1u);
            const uint32_t dl = room + (uint32_t)lane < L ? room + (uint32_t)lane : L;
            const uint32_t dh = room > (uint32_t)lane ? room - (uint32_t)lane : 1u;
            const double fl = (double)dl, fh = (double)dh;
            const double pmw = pm_raw * wgt, uw = u * wgt;
            const bool yes = ident ? (u * fl) * (1.0 + 0x1p-40) < pmw : uw < fh * pr_raw;
            const bool no = ident ? (u * fh) * (1.0 - 0x1p-40) > pmw : !(uw < fl * pr_raw);
            plus = __ballot(ident && yes);
            minus = __ballot(dia && yes);
            uint64_t ambm = __ballot((ident || dia) && !yes && !no);
            while (ambm) {
                const int a = __ffsll((long long)ambm) - 1;
                const uint64_t ba = below_mask(a);
                const int64_t na = (int64_t)n0 + popc(plus & ba) - popc(minus & ba);
                bool d = false;
                if (lane == a) {
                    if (ident)
                        d = u < (pm_raw / (double)((int64_t)L - na)) * wgt;
                    else
                        d = u * wgt < (double)((int64_t)L - na + 1) * pr_raw;
                }
                const uint64_t dm = __ballot(d);
                if ((identm >> a) & 1ull)
                    plus |= dm;
                else
                    minus |= dm;
                ambm &= ambm - 1;
            }
            n0 += (uint32_t)popc(plus) - (uint32_t)popc(minus);
            if (ident && ((plus >> lane) & 1ull))
                fop = op_make(b, (uint32_t)dw.dv);
            if (dia && ((minus >> lane) & 1ull))
                fop = 0u;
            if (fop != op)
                ops[p] = fop;
        }

        // vertex list over the chunk's final non-identity operators: how many
        // earlier operators act on each of the operator's sites
        const uint64_t NI = do_diag ? ((identm & plus) | (diam & ~minus) | offm) : (diam | offm);
        if (do_vl && ((NI >> lane) & 1ull)) {
            const uint32_t i0 = c0 + bits_below(A & NI), i1 = c1 + bits_below(C & NI);
            gidx[p] = (uint64_t)i0 | (uint64_t)i1 << 32;
            atomicAdd(cnt + s0, 1u);
            atomicAdd(cnt + s1, 1u);
        }
        // spins after the chunk: the last off-diagonal operator on a site wins
        if (do_diag && offd) {
            if (((A & offm) & above) == 0ull)
                *lds_at<lds_u8>(spb + s0) = (uint8_t)(up & 255u);
            if (((C & offm) & above) == 0ull)
                *lds_at<lds_u8>(spb + s1) = (uint8_t)(up >> 8);
        }
        if (has) {
            *lds_at<lds_u64>(t0) = 0ull;
            *lds_at<lds_u64>(t1 + 8u) = 0ull;
        }
        wave_lds_sync();
    }
    if (wave_any(bad)) {
        if (lane == 0) {
            W[wi].error = SSE_ERR_STATE;
            flag_error(pool, SSE_ERR_STATE);
        }
        return;
    }

    if (do_vl) {
        for (int s = lane; s < N; s += 64)
            w.last[s] = (int32_t)cnt[s];
    }
    if (do_diag) {
        for (int s = lane; s < N; s += 64)
            w.spins[s] = sp[s];
    }
    if (lane == 0) {
        DevWalker &o = W[wi];
        o.n = n0;
        o.L = L;
        o.cap = w.cap;
        o.ops = w.ops;
        o.links = w.links;
        o.ctr = rs.ctr();
        if (do_vl)
            atomicMax(&pool->max_need[grp & 7], (unsigned long long)worm_lds_need(m, n0));
    }
}

// K1 of walker wi; the model's lookups come from LDS when the launch's LDS
// (lds_bytes) holds them
__device__ __forceinline__ void k1_walker(DevWalker *W, const DevModel *models, DevPool *pool, int wi,
                                          int phases, int warm, char *lds, int lds_bytes, int grp)
{
    const DevModel &m = models[W[wi].model];
    const size_t base = k1_lds_bytes(m.n_sites);
    if (k1_lds_staged(m.n_sites, m.k1tab_bytes) <= (size_t)lds_bytes) {
        const uint32_t kt = (uint32_t)(uintptr_t)(lds_u8 *)lds + (uint32_t)base;
        if (m.k1tab_one)
            k1_walker_t(W, models, pool, wi, phases, warm, lds, K1Staged<true>{kt, 0, 0, 0, 0, 0}, grp);
        else
            k1_walker_t(W, models, pool, wi, phases, warm, lds, K1Staged<false>{kt, 0, 0, 0, 0, 0}, grp);
    } else {
        k1_walker_t(W, models, pool, wi, phases, warm, lds, K1Global{&m}, grp);
    }
}

// kernels of the per-sweep path take a walker range [w_begin, w_end), one
// workgroup (one wave) per walker
// Walker of workgroup b of a launch over positions [w_begin, w_end): with a
// schedule (order: walker indices, largest expected operator count first) the
// position indexes it, else it is the walker index itself.
__device__ __forceinline__ int walker_at(const int32_t *order, int pos)
{
    return order ? order[pos] : pos;
}

__global__ __launch_bounds__(64) void wave_diag_vlist_kernel(DevWalker *W, const DevModel *models,
                                                             DevPool *pool, int w_begin, int w_end,
                                                             int phases, int warm, int lds_bytes,
                                                             const int32_t *order, int grp)
{
    extern __shared__ __align__(16) char lds[];
    const int pos = w_begin + (int)blockIdx.x;
    if (pos < w_end)
        k1_walker(W, models, pool, walker_at(order, pos), phases, warm, lds, lds_bytes, grp);
}

// ------------------------------------------------------------------ K2
// LDS holds the walker's worm records and exit table when they fit lds_bytes;
// rec_mode as worm_walker's mode.
__global__ __launch_bounds__(64) void wave_worm_kernel(DevWalker *W, const DevModel *models,
                                                       DevPool *pool, int w_begin, int w_end,
                                                       int full_sweep, int lds_bytes, int rec_mode,
                                                       const int32_t *order)
{
    extern __shared__ __align__(16) char lds[];
    const int pos = w_begin + (int)blockIdx.x;
    if (pos < w_end)
        worm_walker<2>(W, models, pool, walker_at(order, pos), full_sweep, lds_bytes, rec_mode, lds);
}

// ------------------------------------------------------------------ init
__global__ __launch_bounds__(64) void wave_init_kernel(DevWalker *W, const DevModel *models, int n_walkers)
{
    __shared__ uint64_t rbuf[256];
    const int wi = blockIdx.x;
    if (wi >= n_walkers)
        return;
    const int lane = threadIdx.x;
    DevWalker w = W[wi];
    if (!w.pending)
        return;
    const DevModel &m = models[w.model];
    WaveStream rs;
    rs.init(rbuf, w.key, 0);
    // random state per site (sse.jl:48), one int draw each in site order
    for (int i = 0; i < m.n_sites; ++i) {
        uint8_t v = (uint8_t)(1 + rs.range((uint64_t)m.site_dims[i]));
        if (lane == 0)
            w.spins[i] = v;
    }
    for (int64_t p = lane; p < w.L; p += 64)
        w.ops[p] = 0u;
    if (lane == 0) {
        W[wi].n = 0;
        W[wi].ctr = rs.ctr();
    }
}

// ------------------------------------------------------------------ K3
__device__ __forceinline__ double wave_sum(double x)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        x += __shfl_xor(x, o);
    return x;
}

__device__ __forceinline__ int wave_sum_int(int x)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        x += __shfl_xor(x, o);
    return x;
}
// lane q's x, wave-uniform
__device__ __forceinline__ double lane_f64(double x, int q)
{
    const long long b = __double_as_longlong(x);
    return __hiloint2double(__builtin_amdgcn_readlane((int)(b >> 32), q), __builtin_amdgcn_readlane((int)b, q));
}

// x moved across lanes by one DPP pattern, both 32-bit halves; lanes without
// a source (or outside the row mask) read 0
template <int kCtrl, int kRowMask>
__device__ __forceinline__ double dpp_f64(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, kCtrl, kRowMask, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kCtrl, kRowMask, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Inclusive prefix sum over the wave on the VALU's cross-lane (DPP) paths:
// shifts by 1, 2, 4 and 8 within each row of 16 lanes, then lane 15 of rows
// 0 and 2 added to rows 1 and 3, then lane 31 added to rows 2 and 3.
__device__ __forceinline__ double wave_incl_scan(double x)
{
    x += dpp_f64<0x111, 0xf>(x);  // row_shr:1
    x += dpp_f64<0x112, 0xf>(x);  // row_shr:2
    x += dpp_f64<0x114, 0xf>(x);  // row_shr:4
    x += dpp_f64<0x118, 0xf>(x);  // row_shr:8
    x += dpp_f64<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
    x += dpp_f64<0x143, 0xc>(x);  // row_bcast:31 into rows 2 and 3
    return x;
}

// One pass over the operator string: the sign (sse.jl:305-314) when want_sign,
// and estimators e0 .. e0+ne-1 of the MagnetizationEstimator family
// (magnetization_estimator.jl:96-230), whose running sums over the operator
// positions are wave prefix sums.  Writes the five outputs of each of its
// estimators.  Estimators per pass: with the tables, whose pass holds eight
// values of each at a time, and without.
constexpr int K3_TABLE_E = 2, K3_MAXE = 4;
template <int E>
__device__ __forceinline__ void k3_finish(const DevWalker &w, const DevModel &m, int e0, int ne,
                                          bool want_sign, int neg, int64_t cnt, const double *tmp0,
                                          const double *mag, const double *absmag, const double *mag2,
                                          const double *mag4, double &sign, double *o);
// The estimators' values before the first operator.
template <int E>
__device__ __forceinline__ void k3_start(const DevWalker &w, const DevModel &m, int e0, int ne, double *tmp0)
{
    const int N = m.n_sites, D = m.est_max_dim;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        double t0 = 0.0;
        if (k < ne) {
            const double *cf = m.est_coef + (size_t)(e0 + k) * N, *mk = m.est_mval + (size_t)(e0 + k) * N * D;
            for (int i = threadIdx.x; i < N; i += 64)
                t0 += cf[i] * mk[i * D + w.spins[i] - 1];
        }
        tmp0[k] = k < ne ? wave_sum(t0) : 0.0;
    }
}

// From per-(bond, vertex) tables: an operator's estimator changes and sign are
// one gather each.  A lane takes four slots in a row, so one prefix sum over the
// wave, which was most of a chunk's work, serves 256 slots instead of 64; the
// operators are loaded two chunks ahead, their table values one ahead.  Measured
// on 16x16 Heisenberg at beta = 8 (8711 slots, two estimators): 88 -> 52 us of a
// lone wave, 125 -> 77 us with 1536 walkers.  Four estimators in a pass (173
// registers) gave half of that back in the work-queue kernel.
__device__ __forceinline__ void k3_table_pass(const DevWalker &w, const DevModel &m, int e0, int ne,
                                              bool want_sign, double &sign, double *o)
{
    constexpr int E = K3_TABLE_E;
    const int lane = threadIdx.x;
    const int64_t L = w.L;
    double tmp0[E], run[E], mag[E] = {}, absmag[E] = {}, mag2[E] = {}, mag4[E] = {};
    k3_start<E>(w, m, e0, ne, tmp0);
#pragma unroll
    for (int k = 0; k < E; ++k)
        run[k] = tmp0[k];
    const gmem<uint32_t> *ops = as_global((const uint32_t *)w.ops);
    constexpr int K = 4;
    const gmem<double> *DT = as_global(m.est_dtab);
    const gmem<int8_t> *SG = as_global(m.est_dsgn);
    const uint32_t dnv = (uint32_t)m.est_dnv, NE = (uint32_t)m.n_est;
    const bool sgn = want_sign && m.any_neg;
    // slots past L (the vector may hold up to three) read as identities
    auto ops_at = [&](int64_t q, uint32_t (&op)[K]) {
        u32x4 x = {0u, 0u, 0u, 0u};
        if (q < L)
            x = *(const gmem<u32x4> *)(ops + q);
        op[0] = x.x;
        op[1] = q + 1 < L ? x.y : 0u;
        op[2] = q + 2 < L ? x.z : 0u;
        op[3] = q + 3 < L ? x.w : 0u;
    };
    auto vals_of = [&](const uint32_t (&op)[K], double (&d)[E][K], int &ng) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const uint32_t ix = op_bond(op[j]) * dnv + (op_vcode(op[j]) >> 1);
            const bool offd = op[j] != 0u && !(op_vcode(op[j]) & 1u);
#pragma unroll
            for (int k = 0; k < E; ++k)
                d[k][j] = k < ne && offd ? DT[(size_t)ix * NE + e0 + k] : 0.0;
            if (sgn && op[j] != 0u)
                ng += SG[ix] < 0;
        }
    };
    int ngl = 0, cntl = 0;
    uint32_t op0[K], op1[K];
    ops_at(K * lane, op0);
    ops_at(64 * K + K * lane, op1);
    double d0[E][K];
    vals_of(op0, d0, ngl);
    for (int64_t base = 0; base < L; base += 64 * K) {
        uint32_t op2[K];
        ops_at(base + 128 * K + K * lane, op2);
        double d1[E][K];
        vals_of(op1, d1, ngl);
#pragma unroll
        for (int j = 0; j < K; ++j)
            cntl += op0[j] != 0u;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            if (k < ne) {
                const double own = (d0[k][0] + d0[k][1]) + (d0[k][2] + d0[k][3]);
                const double inc = wave_incl_scan(own);
                double t = run[k] + (inc - own);
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    t += d0[k][j];
                    const double u = op0[j] != 0u ? t : 0.0;
                    const double u2 = u * u;
                    mag[k] += u;
                    absmag[k] += fabs(u);
                    mag2[k] += u2;
                    mag4[k] += u2 * u2;
                }
                run[k] += lane_f64(inc, 63);
            }
        }
#pragma unroll
        for (int j = 0; j < K; ++j) {
            op0[j] = op1[j];
            op1[j] = op2[j];
#pragma unroll
            for (int k = 0; k < E; ++k)
                d0[k][j] = d1[k][j];
        }
    }
    k3_finish<E>(w, m, e0, ne, want_sign, wave_sum_int(ngl), wave_sum_int(cntl), tmp0, mag, absmag, mag2,
                 mag4, sign, o);
}

// The same from the bonds' and vertices' own tables, for models without the
// per-(bond, vertex) ones.
__device__ __forceinline__ void k3_gather_pass(const DevWalker &w, const DevModel &m, int e0, int ne,
                                               bool want_sign, double &sign, double *o)
{
    const int lane = threadIdx.x;
    const int64_t L = w.L;
    const int N = m.n_sites, D = m.est_max_dim;
    const double *coef[K3_MAXE], *mv[K3_MAXE];
    double tmp0[K3_MAXE], run[K3_MAXE], mag[K3_MAXE] = {}, absmag[K3_MAXE] = {}, mag2[K3_MAXE] = {},
                                        mag4[K3_MAXE] = {};
    k3_start<K3_MAXE>(w, m, e0, ne, tmp0);
#pragma unroll
    for (int k = 0; k < K3_MAXE; ++k) {
        coef[k] = m.est_coef + (size_t)(e0 + k) * N;
        mv[k] = m.est_mval + (size_t)(e0 + k) * N * D;
        run[k] = tmp0[k];
    }
    int neg = 0;
    int64_t cnt = 0;
    const gmem<uint32_t> *ops = as_global((const uint32_t *)w.ops);
    const gmem<uint64_t> *brec = as_global((const uint64_t *)m.bond_rec);  // int2 pairs
    // Software pipeline over the 64-slot chunks: the operator is loaded three
    // chunks ahead, its bond record two ahead, the vertex's sign and leg states
    // one ahead, so a chunk waits only for its estimator table values.  The
    // vertex tables of up to four bond types are addressed from registers.
    const int nt = m.n_types;
    const int8_t *sgt[4];
    const uint8_t *lst[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        sgt[t] = t < nt ? m.types[t].signs : nullptr;
        lst[t] = t < nt ? m.types[t].leg_states : nullptr;
    }
    auto op_at = [&](int64_t q) -> uint32_t { return q < L ? ops[q] : 0u; };
    auto bond_of = [&](uint32_t op) -> uint64_t { return op != 0u ? brec[op_bond(op)] : 0ull; };
    // sign of a vertex and, for an off-diagonal one, its four leg states (one u32)
    auto vertex_of = [&](uint32_t op, uint64_t bv, int8_t &sg, uint32_t &legs) {
        sg = 0;
        legs = 0u;
        if (op != 0u) {
            const int type = (int)((uint32_t)bv >> 20);
            const uint32_t v = op_vcode(op) >> 1;
            const int8_t *sp = nt <= 4 ? (type == 0 ? sgt[0] : type == 1 ? sgt[1] : type == 2 ? sgt[2] : sgt[3])
                                       : m.types[type].signs;
            const uint8_t *lp = nt <= 4 ? (type == 0 ? lst[0] : type == 1 ? lst[1] : type == 2 ? lst[2] : lst[3])
                                        : m.types[type].leg_states;
            sg = as_global(sp)[v];
            if (!(op_vcode(op) & 1u))  // off-diagonal: the leg states matter
                legs = *(const gmem<uint32_t> *)as_global((const uint32_t *)(lp + 4 * v));
        }
    };
    // prime the pipeline
    uint32_t op0 = op_at(lane), op1 = op_at(64 + lane), op2 = op_at(128 + lane);
    uint64_t bv0 = bond_of(op0), bv1 = bond_of(op1);
    int8_t sg0;
    uint32_t lg0;
    vertex_of(op0, bv0, sg0, lg0);
    for (int64_t base = 0; base < L; base += 64) {
        // issue the later stages' loads for the chunks ahead
        const uint32_t op3 = op_at(base + 192 + lane);
        const uint64_t bv2 = bond_of(op2);
        int8_t sg1;
        uint32_t lg1;
        vertex_of(op1, bv1, sg1, lg1);
        // this chunk
        const uint32_t op = op0;
        const uint32_t vc = op_vcode(op);
        if (want_sign)
            neg += popc(__ballot(op != 0u && sg0 < 0));
        cnt += popc(__ballot(op != 0u));
        const bool offd = op != 0u && !(vc & 1u);
        const uint32_t l0 = lg0 & 255u, l1 = (lg0 >> 8) & 255u, l2 = (lg0 >> 16) & 255u, l3 = lg0 >> 24;
        const int sa = (int)((uint32_t)bv0 & 0xFFFFFu), sb = (int)(uint32_t)(bv0 >> 32);
#pragma unroll
        for (int k = 0; k < K3_MAXE; ++k) {
            if (k < ne) {
                double delta = 0.0;
                if (offd) {
                    const gmem<double> *cf = as_global(coef[k]), *mk = as_global(mv[k]);
                    delta = cf[sa] * (mk[sa * D + l2 - 1] - mk[sa * D + l0 - 1]);
                    delta += cf[sb] * (mk[sb * D + l3 - 1] - mk[sb * D + l1 - 1]);
                }
                const double inc = wave_incl_scan(delta);
                if (op != 0u) {
                    const double t = run[k] + inc;
                    const double t2 = t * t;
                    mag[k] += t;
                    absmag[k] += fabs(t);
                    mag2[k] += t2;
                    mag4[k] += t2 * t2;
                }
                run[k] += __shfl(inc, 63);
            }
        }
        // rotate the pipeline
        op0 = op1;
        op1 = op2;
        op2 = op3;
        bv0 = bv1;
        bv1 = bv2;
        sg0 = sg1;
        lg0 = lg1;
    }
    k3_finish<K3_MAXE>(w, m, e0, ne, want_sign, neg, cnt, tmp0, mag, absmag, mag2, mag4, sign, o);
}

// The five outputs of each estimator of a pass (and the sign of the first).
template <int E>
__device__ __forceinline__ void k3_finish(const DevWalker &w, const DevModel &m, int e0, int ne,
                                          bool want_sign, int neg, int64_t cnt, const double *tmp0,
                                          const double *mag, const double *absmag, const double *mag2,
                                          const double *mag4, double &sign, double *o)
{
    const int lane = threadIdx.x;
    if (want_sign)
        sign = (neg & 1) ? -1.0 : 1.0;
    const double Nn = m.norm;
    const double en = 1.0 + (double)cnt;
    const double norm = 1.0 / Nn;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        if (k < ne) {
            double smag = tmp0[k] + wave_sum(mag[k]);
            double sabs = fabs(tmp0[k]) + wave_sum(absmag[k]);
            double s2 = tmp0[k] * tmp0[k];
            double smag2 = s2 + wave_sum(mag2[k]);
            double smag4 = s2 * s2 + wave_sum(mag4[k]);
            smag *= norm;
            sabs *= norm;
            smag2 *= norm * norm;
            smag4 *= (norm * norm) * (norm * norm);
            if (lane == 0) {
                double *oe = o + 5 + 5 * (e0 + k);
                oe[0] = sign * smag / en;
                oe[1] = sign * sabs / en;
                oe[2] = sign * smag2 / en;
                oe[3] = sign * smag4 / en;
                const double chi = 1.0 / w.T / (en + 1.0) / en * (smag * smag + smag2) * Nn;
                oe[4] = sign * chi;
            }
        }
    }
}

// measure (sse.jl:70-87, 305-376) of walker wi.  mode 0: explicit measure;
// mode 1: thermalized walkers only, accumulated into the per-walker sums
// (fused sweep+measure loop).  Estimators are taken a few per pass over the
// operator string; the first pass also computes the sign.
__device__ __forceinline__ void k3_walker(DevWalker *W, const DevModel *models, double *out, double *sum,
                                          double *sumsq, int64_t *count, double *wlf, int wi, int mode,
                                          int32_t *done)
{
    const int lane = threadIdx.x;
    const DevWalker w = W[wi];
    // a pending slot's opstring and spins are not initialised yet
    if (w.error || w.pending || (mode == 1 && !w.active))
        return;
    if (mode == 1 && !(w.sweeps > w.thermalization)) {
        if (w.retire && lane == 0) {
            W[wi].retire = 0;
            W[wi].active = 0;
            done[wi] = 1;
        }
        return;
    }
    const DevModel &m = models[w.model];
    double *o = out + w.meas_offset;
    double sign = 1.0;
    int e0 = 0;
    do {
        const int E = m.est_dtab ? K3_TABLE_E : K3_MAXE;
        const int ne = m.n_est - e0 < E ? m.n_est - e0 : E;
        if (m.est_dtab)
            k3_table_pass(w, m, e0, ne, e0 == 0, sign, o);
        else
            k3_gather_pass(w, m, e0, ne, e0 == 0, sign, o);
        e0 += E;
    } while (e0 < m.n_est);
    const double nn = (double)w.n;
    if (lane == 0) {
        o[0] = sign;
        o[1] = nn;
        o[2] = sign * nn;
        o[3] = sign * (nn * nn);
        o[4] = ((-sign) * (nn * w.T + m.energy_offset)) / m.norm;
    }
    if (mode == 1) {
        __syncthreads();
        for (int j = lane; j < w.meas_width; j += 64) {
            const double x = o[j];
            sum[w.meas_offset + j] += x;
            sumsq[w.meas_offset + j] += x * x;
        }
        if (lane == 0) {
            count[w.acc_slot] += 1;
            worm_fraction_accumulate(w, wlf);
            if (w.retire) {
                W[wi].retire = 0;
                W[wi].active = 0;
                done[wi] = 1;
            }
        }
    }
}

__global__ __launch_bounds__(64) void wave_measure_kernel(DevWalker *W, const DevModel *models,
                                                          double *out, double *sum, double *sumsq,
                                                          int64_t *count, double *wlf, int w_begin,
                                                          int w_end, int mode, int32_t *done,
                                                          const int32_t *order)
{
    const int pos = w_begin + (int)blockIdx.x;
    if (pos < w_end)
        k3_walker(W, models, out, sum, sumsq, count, wlf, walker_at(order, pos), mode, done);
}

// K2 and the accumulated measurement of the same sweep in one kernel: each
// walker's wave measures as soon as its own worm update is written back, so the
// measurement runs inside the launch's worm tail instead of after it.  The
// measurement reads the operator string, spins and DevWalker that the worm
// phase of the same wave has just stored, through vector loads after the
// barrier (nothing of it goes through the scalar cache).
__global__ __launch_bounds__(64) void wave_worm_measure_kernel(
    DevWalker *W, const DevModel *models, DevPool *pool, int w_begin, int w_end, int lds_bytes,
    int rec_mode, const int32_t *order, double *out, double *sum, double *sumsq, int64_t *count,
    double *wlf, int32_t *done)
{
    extern __shared__ __align__(16) char lds[];
    const int pos = w_begin + (int)blockIdx.x;
    if (pos < w_end) {
        const int wi = walker_at(order, pos);
        worm_walker<2>(W, models, pool, wi, 1, lds_bytes, rec_mode, lds);
        __syncthreads();
        k3_walker(W, models, out, sum, sumsq, count, wlf, wi, 1, done);
    }
}

// pending walkers become active once initialised
__global__ void activate_pending_kernel(DevWalker *W, int n_walkers)
{
    int wi = blockIdx.x * blockDim.x + threadIdx.x;
    if (wi >= n_walkers)
        return;
    if (W[wi].pending) {
        W[wi].pending = 0;
        W[wi].active = 1;
    }
}

// ------------------------------------------------------------------ host side
#include "sse_wave_n.h"

// LDS of the generic diagonal-update kernel: the base layout for the largest
// site count and bond size, raised to stage a model's lookups in LDS where that
// keeps it within 32 KiB (other models read them from global memory)
static inline size_t k1n_lds_for(const std::vector<DevModel> &models, int max_sites, int max_ns)
{
    size_t b = k1n_lds_bytes(max_sites, max_ns);
    for (const DevModel &m : models) {
        const size_t st = k1n_lds_staged(m.n_sites, m.nsb, m.k1ntab_bytes);
        if (st <= 32768 && st > b)
            b = st;
    }
    return b;
}

static inline int wave_configure(WaveConfig &c, const std::vector<DevModel> &models, int max_sites)
{
    c.max_sites = max_sites;
    c.lds_k1 = k1_lds_bytes(max_sites);
    int max_ns = 2;
    c.generic = 0;
    for (const DevModel &m : models) {
        max_ns = std::max(max_ns, (int)m.nsb);
        if (m.nsb != 2)
            c.generic = 1;
    }
    c.lds_k1n = k1n_lds_for(models, max_sites, max_ns);
    if (c.generic && c.lds_k1n > 65536)
        (void)hipFuncSetAttribute((const void *)waven_diag_vlist_kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds_k1n);
    // stage each model's lookups in LDS if that keeps K1 within 32 KiB (high
    // occupancy matters more than the lookups of larger models)
    for (const DevModel &m : models) {
        const size_t st = (k1_lds_staged(m.n_sites, m.k1tab_bytes) + 15) & ~(size_t)15;
        if (st <= 32768 && st > c.lds_k1)
            c.lds_k1 = st;
    }
    int dev = 0, lim = 65536;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
        lim > 0)
        c.lds_limit = (size_t)lim;
    if (c.lds_k1 > c.lds_limit || (c.generic && c.lds_k1n > c.lds_limit))
        return SSE_ERR_INVALID;
    c.lds_k2 = 4096;
    if (c.lds_limit > 65536) {
        (void)hipFuncSetAttribute((const void *)waven_worm_kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds_limit);
        (void)hipFuncSetAttribute((const void *)wave_worm_measure_kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds_limit);
        (void)hipFuncSetAttribute((const void *)wave_worm_kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds_limit);
        (void)hipFuncSetAttribute((const void *)wave_diag_vlist_kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds_limit);
    }
    return SSE_OK;
}

// LDS per walker the worm kernel is sized for at most: beyond it a walker keeps
// its records in global memory instead of lowering every walker's residency
constexpr size_t K2_LDS_CAP = 65536;

// Residency measured on MI355X: a workgroup takes round512(bytes + 256) of the CU's
// LDS and 162816 bytes are usable per CU (26880 B run 6 walkers per CU, 32000 B run 5,
// 32256 B and up only 4, whatever the occupancy query says); registers allow 8.
constexpr size_t kLdsPerCu = 162816;
static inline size_t lds_walkers(size_t bytes)
{
    return std::min((size_t)8, std::max((size_t)1, kLdsPerCu / ((bytes + 256 + 511) & ~(size_t)511)));
}
// the largest size that k walkers per CU can have
static inline size_t lds_for_walkers(size_t k) { return ((kLdsPerCu / k) & ~(size_t)511) - 256; }

// Worm-kernel LDS per walker for the largest need (worm_lds_need) among the
// last call's walkers, with a little headroom; walkers that do not fit keep
// their records in global memory for that sweep.  The allocation is then
// widened to the largest size that keeps the same number of walkers per CU
// (more headroom at no cost in residency).
static inline size_t wave_k2_lds_for(const WaveConfig &c, unsigned long long max_need)
{
    if (c.lds_k2_fixed)
        return c.lds_k2_fixed;
    size_t need = (size_t)max_need + (size_t)max_need / 64 + 256;
    if (need > K2_LDS_CAP)
        need = K2_LDS_CAP;
    need = (need + 255) & ~(size_t)255;
    if (need > c.lds_limit)
        need = c.lds_limit;
    // walkers per CU: as many as fit, at most the 8 that the registers allow.  So
    // batches of small walkers keep one size, and a captured launch stays valid.
    return std::max(need, std::min(c.lds_limit, lds_for_walkers(lds_walkers(need))));
}

static inline void wave_resize_lds(WaveConfig &c, unsigned long long max_need)
{
    c.lds_k2 = wave_k2_lds_for(c, max_need);
}

static inline int wave_launch_init(WaveConfig &c, hipStream_t s, DevWalker *W, const DevModel *M,
                                   DevPool *pool, int n, int max_warmup)
{
    hipLaunchKernelGGL(wave_init_kernel, dim3(n), dim3(64), 0, s, W, M, n);
    for (int r = 0; r < max_warmup; ++r) {
        if (c.generic)
            hipLaunchKernelGGL(waven_diag_vlist_kernel, dim3(n), dim3(64), c.lds_k1n, s, W, M, pool, 0,
                               n, 1, r, (const int32_t *)nullptr, 0, (const int32_t *)nullptr, 0,
                               (int)c.lds_k1n);
        else
            hipLaunchKernelGGL(wave_diag_vlist_kernel, dim3(n), dim3(64), c.lds_k1, s, W, M, pool, 0, n,
                               1, r, (int)c.lds_k1, (const int32_t *)nullptr, 0);
    }
    hipLaunchKernelGGL(activate_pending_kernel, dim3((n + 63) / 64), dim3(64), 0, s, W, n);
    return hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP;
}

// one sweep (phase mask) of the walkers at schedule positions [w0, w1) on
// stream s; grp is their stream group (0..6: its own worm-kernel LDS size
// once sized; -1: one stream for all walkers)
static inline int wave_launch_sweep(WaveConfig &c, hipStream_t s, DevWalker *W, const DevModel *M,
                                    DevPool *pool, int w0, int w1, int phases, hipEvent_t *ev,
                                    const int32_t *order = nullptr, int grp = -1)
{
    const int n = w1 - w0;
    const int k1 = phases & (1 | 2 | 8);
    const int g = grp >= 0 && grp < 7 ? grp : 7;  // slot 7 collects the rest
    const size_t lds2 = g < 7 && c.lds_k2_group[g] ? c.lds_k2_group[g] : c.lds_k2;
    if (c.generic) {
        if (k1 & 3)
            hipLaunchKernelGGL(waven_diag_vlist_kernel, dim3(n), dim3(64), c.lds_k1n, s, W, M, pool, w0,
                               w1, k1, -1, order, g, (const int32_t *)nullptr, 0, (int)c.lds_k1n);
        if (ev)
            (void)hipEventRecord(ev[1], s);
        if (phases & 4)
            hipLaunchKernelGGL(waven_worm_kernel, dim3(n), dim3(64), lds2, s, W, M, pool, w0, w1,
                               (phases & 7) == 7 ? 1 : 0, order, (const int32_t *)nullptr, 0,
                               (int)lds2, c.rec_mode);
        if (ev)
            (void)hipEventRecord(ev[2], s);
        return hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP;
    }
    if (k1 & 3) {
        hipLaunchKernelGGL(wave_diag_vlist_kernel, dim3(n), dim3(64), c.lds_k1, s, W, M, pool, w0, w1, k1,
                           -1, (int)c.lds_k1, order, g);
    }
    if (ev)
        (void)hipEventRecord(ev[1], s);
    if (phases & 4)
        hipLaunchKernelGGL(wave_worm_kernel, dim3(n), dim3(64), lds2, s, W, M, pool, w0, w1,
                           (phases & 7) == 7 ? 1 : 0, (int)lds2, c.rec_mode, order);
    if (ev)
        (void)hipEventRecord(ev[2], s);
    return hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP;
}

// one measuring sweep of the walkers at schedule positions [w0, w1): K1, then
// the worm update and measurement in one kernel (ev[1] after K1, ev[2] after
// the fused kernel)
static inline int wave_launch_sweep_measure(WaveConfig &c, hipStream_t s, DevWalker *W,
                                            const DevModel *M, DevPool *pool, int w0, int w1,
                                            hipEvent_t *ev, const int32_t *order, int grp,
                                            double *out, double *sum, double *sumsq,
                                            int64_t *count, double *wlf, int32_t *done)
{
    const int n = w1 - w0;
    const int g = grp >= 0 && grp < 7 ? grp : 7;
    if (c.generic) {  // no fused form: sweep, then measure
        int rc = wave_launch_sweep(c, s, W, M, pool, w0, w1, 7, ev, order, grp);
        if (!rc)
            hipLaunchKernelGGL(waven_measure_kernel, dim3(n), dim3(64), 0, s, W, M, out, sum, sumsq,
                               count, wlf, w0, w1, 1, done, order, (const int32_t *)nullptr, 0);
        return rc ? rc : (hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP);
    }
    const size_t lds2 = g < 7 && c.lds_k2_group[g] ? c.lds_k2_group[g] : c.lds_k2;
    hipLaunchKernelGGL(wave_diag_vlist_kernel, dim3(n), dim3(64), c.lds_k1, s, W, M, pool, w0, w1, 3,
                       -1, (int)c.lds_k1, order, g);
    if (ev)
        (void)hipEventRecord(ev[1], s);
    hipLaunchKernelGGL(wave_worm_measure_kernel, dim3(n), dim3(64), lds2, s, W, M, pool, w0, w1,
                       (int)lds2, c.rec_mode, order, out, sum, sumsq, count, wlf, done);
    if (ev)
        (void)hipEventRecord(ev[2], s);
    return hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP;
}

static inline int wave_launch_measure(WaveConfig &c, hipStream_t s, DevWalker *W, const DevModel *M,
                                      double *out, double *sum, double *sumsq, int64_t *count,
                                      double *wlf, int w0, int w1, int mode, int32_t *done,
                                      const int32_t *order = nullptr)
{
    if (c.generic)
        hipLaunchKernelGGL(waven_measure_kernel, dim3(w1 - w0), dim3(64), 0, s, W, M, out, sum, sumsq,
                           count, wlf, w0, w1, mode, done, order, (const int32_t *)nullptr, 0);
    else
        hipLaunchKernelGGL(wave_measure_kernel, dim3(w1 - w0), dim3(64), 0, s, W, M, out, sum, sumsq,
                           count, wlf, w0, w1, mode, done, order);
    return hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP;
}

