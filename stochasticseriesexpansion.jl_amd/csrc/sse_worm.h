// sse_worm.h -- the worm update (sse.jl:193-303), one wavefront per walker, for
// bonds of any site count NS = 1..4.
//
// The traversal is a sequential pointer chase, so its speed is the latency of
// one step.  Measured on MI355X (cycles): LDS load 60, the same made
// wave-uniform for the scalar unit 88, L1 load 120, scalar load of a 64-byte
// entry 77, v_readlane feeding a v_readlane 29, a dependent vector instruction
// about 6.  So the step stays on the vector unit: every lane holds the same
// position, codes and exits, and nothing crosses to the scalar unit except
// branches, which resolve while a load is in flight.  A step is two dependent
// LDS loads and a handful of vector instructions:
//
//   c, partner = records[e]        the entry the worm is at
//   word       = exits[q_t, c, port]    q_t: the step's random word as a rank
//   e'         = (e - 1, partner - 1, e + 1, partner + 1)[word]
//
// Records by site: the operators of a lattice site lie one after another, so
// the neighbour along the site is the next or previous entry and no link is
// stored; an entry keeps the entry of its operator on the bond's next site
// (cyclically) and the operator's vertex code.  A guard entry at either end of a
// site's range closes it periodically.  That is 3 bytes per entry (u16 partner,
// u8 code), 6 bytes per operator of a two-site bond against 8 for four links
// and a code, and it holds up to 32768 entries.  An entry's partner carries a flag bit in
// guards, in the entry the current worm started from and in the entry behind the
// leg it started from: one test per step covers closure, periodic closure and
// the worm's end, and its branch waits for nothing.
//
// LDS of a walker: exit table | codes | partners | first entry per site.  Entry
// ids are the code's byte address (8-bit codes) or half of it (16-bit codes).
// Walkers that do not fit keep the records in global memory; with three and four
// sites to a bond the codes stay in LDS where they fit it without the partners.
//
// Measured (64 walkers, one to a CU; the worm kernel, us, against records of four
// links and 64-bit threshold compares on the scalar unit): 16x16 Heisenberg at
// beta = 8 (n = 2920) 2088 -> 1502, a step 288 -> 200 cycles; spin-1 honeycomb
// 1355 -> 946; dimer ladder 736 -> 635; against links read from L2: ring of
// three-site bonds 3660 -> 1920, of four-site bonds 1034 -> 607.
#pragma once
#include "sse_common.h"

typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) int16_t lds_i16;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint64_t lds_u64;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef const __attribute__((address_space(4))) uint64_t const_u64;
typedef const __attribute__((address_space(4))) uint8_t const_u8;

// LDS by byte address: entry ids and table rows are addresses, so that the step
// adds no base
template <class T>
__device__ __forceinline__ T *lds_at(uint32_t a)
{
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wint-to-pointer-cast"
    return (T *)a;
#pragma clang diagnostic pop
}

constexpr uint32_t kWormIds = 32768;  // entry ids of the LDS layouts stay below (flag bit)

template <int NS>
struct WormNS {
    static constexpr int LG = NS == 1 ? 0 : NS == 2 ? 1 : 2;   // log2 of the code stride
    static constexpr int LCB = NS <= 2 ? 2 : 3;                // bits of a leg selector
};

__device__ __forceinline__ uint32_t rdlane(uint32_t v, uint32_t l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ bool wave_any(bool x) { return __builtin_amdgcn_ballot_w64(x) != 0ull; }

// ------------------------------------------------------------------ ranks
// q = number of the model's thresholds that are <= m, for the tables in LDS.  Up to
// 8: compared one by one against scalar operands.  More: a 256-bucket start by the
// mantissa's top bits, then the bucket's own thresholds, few as a rule; from the LDS
// copy of DevModel::wthr behind the exit table.  The 64 ranks of a buffer of words
// take some 300 cycles for 25-35 thresholds, by comparing all 1500-3000.
struct WormRank {
    const uint64_t *thr;
    int n;
    uint32_t lds;  // byte address of the LDS copy (n > 8)
    __device__ __forceinline__ uint32_t of(uint64_t m) const
    {
        uint32_t q = 0;
        if (n <= 8) {
            const_u64 *t = (const_u64 *)(const void *)uni64((uint64_t)(const void *)thr);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                q += t[u] <= m ? 1u : 0u;
            return q;
        }
        const uint32_t pad = ((uint32_t)n + 8u) & ~7u;  // entries ahead of the buckets
        q = *lds_at<lds_u16>(lds + 8u * pad + 2u * (uint32_t)(m >> 45));
        for (;;) {
            const bool up = *lds_at<lds_u64>(lds + 8u * q) <= m;  // ~0 ends the list
            if (!wave_any(up))
                return q;
            q += up ? 1u : 0u;
        }
    }
};

// ------------------------------------------------------------------ exit tables
// A word from kWormTail on is marked in its row's top bit and looked up exactly, so
// that a table whose last cumulative probability misses 1 by rounding still has an
// exit for every other word.  Exit rows mark nothing: they are built only where no
// threshold but 1 lies in the tail.
__device__ __forceinline__ uint32_t worm_tail_bit(uint64_t m) { return m >= kWormTail ? 0x80000000u : 0u; }

// A table gives for an entry's word and the step's row, in two parts so that the
// next entry's loads leave before the rest is worked out: pick(), with sh() =
// 16 * leg selector (TabRows: its low six bits); then the port of the next entry
// and the operator's new codes at entry e and its cyclic successors.
template <int NS>
struct WormExit {
    uint32_t port, c[NS];
    uint32_t none;  // bit 31: the entry has no exit for the word
};

// Exit rows in LDS, one word per (q, entry): selector << 4 in the low six bits,
// port in byte 1, the new codes of e and its partner in bytes 2 and 3.  For
// small tables (NS <= 2, codes of 8 bits) whose every word has an exit: no
// compare at all is left in the step.
template <int NS>
struct TabRows {
    static constexpr bool kNone = false, kScalar = false;
    WormRank rank;
    uint32_t base, rowbytes, ports;  // ports: 2 * worm types
    typedef uint32_t Word;
    __device__ __forceinline__ uint32_t row_of(uint64_t m) const { return base + rank.of(m) * rowbytes; }
    // all but the code is known before the code's load returns.  Volatile, so that the load stays ahead of the flag
    // test whose branch resolves under it.
    __device__ __forceinline__ Word load(uint32_t row, uint32_t c, uint32_t port) const
    {
        uint32_t pre = row + port * 4u;
        asm("" : "+v"(pre));
        return *lds_at<volatile lds_u32>(__umul24(c, ports * 4u) + pre);
    }
    typedef uint32_t Pick;
    __device__ __forceinline__ Pick pick(Word w, uint32_t) const { return w; }
    __device__ __forceinline__ static uint32_t sh(Pick w) { return w; }
    __device__ __forceinline__ WormExit<NS> exit(Pick w, uint32_t) const
    {
        WormExit<NS> x;
        x.port = (w >> 8) & 255u;
        x.c[0] = (w >> 16) & 255u;
        if constexpr (NS > 1)
            x.c[1] = w >> 24;
        x.none = 0u;
        return x;
    }
};

// One 16-byte entry in LDS: four 16-bit exits (selector, port, code; bit 15 where
// there is none), then three ranks in 10-bit fields (and, for four sites per
// bond, a fourth rank and a fifth exit).  With the row word Q = q in three fields, each with a
// guard bit above, the guards left standing in Q - ranks count the ranks
// <= q, which is the exit's index.
template <int NS>
struct TabExits {
    static constexpr bool kNone = true, kScalar = false;
    static constexpr uint32_t kGuards = 1u << 9 | 1u << 19 | 1u << 29;
    WormRank rank;
    uint32_t base, ports;  // ports: 2 * worm types
    typedef u32x4 Word;
    __device__ __forceinline__ uint32_t row_of(uint64_t m) const
    {
        return rank.of(m) * (1u | 1u << 10 | 1u << 20) | kGuards | worm_tail_bit(m);
    }
    __device__ __forceinline__ Word load(uint32_t, uint32_t c, uint32_t port) const
    {
        uint32_t pre = base + port * 16u;
        asm("" : "+v"(pre));
        return *lds_at<volatile lds_u32x4>(__umul24(c, ports * 16u) + pre);
    }
    typedef uint32_t Pick;
    __device__ __forceinline__ Pick pick(Word w, uint32_t row) const
    {
        const uint32_t j = (uint32_t)__popc((row - w.z) & kGuards);
        const uint64_t outs = (uint64_t)w.x | (uint64_t)w.y << 32;
        uint32_t o = (uint32_t)(outs >> (16u * j));
        if constexpr (NS == 4)  // a fifth exit behind a fourth rank
            o = (row & 511u) >= (w.w & 0xFFFFu) ? w.w >> 16 : o;
        return o;
    }
    __device__ __forceinline__ static uint32_t sh(Pick o) { return o << 4; }
    __device__ __forceinline__ WormExit<NS> exit(Pick o, uint32_t c) const
    {
        constexpr int LG = WormNS<NS>::LG, LCB = WormNS<NS>::LCB;
        WormExit<NS> x;
        x.port = (o >> LCB) & ((1u << (8 - LCB)) - 1u);
        x.none = o << 16;
        const uint32_t nc = ((o >> 8) & 255u) << LG;
        uint32_t pos = c & ((1u << LG) - 1u);
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            x.c[k] = nc | pos;
            pos = NS == 2 ? pos ^ 1u : pos + 1u == NS ? 0u : pos + 1u;
        }
        return x;
    }
};

// Wide entries in global memory: any number of codes, worm types and thresholds.  The
// table is constant, and one load to the scalar unit brings a whole entry; a word is
// compared by its top 32 bits against the entry's own thresholds, so that no rank is
// needed, however many bond types a model has.  Where they are equal (2^-32 a
// compare) and in the tail the exact search decides.  Against ranks searched in global
// memory and entries of 64 bytes selected through scratch, a step of an XXZ square in
// a field took, by number of different bonds: 32 320 -> 170 ns, 512 401 -> 181 ns.
template <int NS>
struct TabWide {
    static constexpr bool kNone = true, kScalar = true;
    uint32_t ports;
    const uint32_t *t;
    typedef uint32_t Word __attribute__((ext_vector_type(worm_wide_words(NS))));
    typedef const __attribute__((address_space(4))) Word const_word;
    __device__ __forceinline__ uint32_t row_of(uint64_t m) const { return (uint32_t)(m >> 21); }
    __device__ __forceinline__ Word load(uint32_t, uint32_t c, uint32_t port) const
    {
        // below 4 GB: a 32-bit offset goes into the load instruction
        const uint32_t at = (uni(c) * ports + uni(port)) * (uint32_t)sizeof(Word);
        return *(const_word *)((const_u8 *)(const void *)t + at);
    }
    __device__ __forceinline__ static uint32_t unsure(Word w, uint32_t row)
    {
        bool u = row == w[0] || row == w[1] || row == w[2] || row == ~0u;
        if constexpr (NS == 4)
            u = u || row == w[7];
        return u ? 0x80000000u : 0u;
    }
    typedef uint32_t Pick;
    __device__ __forceinline__ Pick pick(Word w, uint32_t row) const
    {
        uint32_t o = w[6];
        if constexpr (NS == 4)
            o = row < w[7] ? o : w[8];
        o = row < w[2] ? w[5] : o;
        o = row < w[1] ? w[4] : o;
        return row < w[0] ? w[3] : o;
    }
    __device__ __forceinline__ static uint32_t sh(Pick o) { return o; }
    __device__ __forceinline__ WormExit<NS> exit(Pick o, uint32_t c) const
    {
        constexpr int LG = WormNS<NS>::LG;
        WormExit<NS> x;
        x.port = worm_entry_port(o);
        x.none = o;
        uint32_t pos = c & ((1u << LG) - 1u);
        const uint32_t nc = c - pos + ((uint32_t)worm_entry_step(o) << LG);
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            x.c[k] = nc | pos;
            pos = NS == 2 ? pos ^ 1u : pos + 1u == NS ? 0u : pos + 1u;
        }
        return x;
    }
};

// ------------------------------------------------------------------ records
// Entry ids start at id0.  An entry's partners are a Part: the entry of its operator on
// the bond's next site, whose own gives the one after that, and the flag.
template <uint32_t kFlag>
struct RecNext {
    typedef int32_t Part;
    // bit 31: flagged
    __device__ __forceinline__ static uint32_t top(Part p) { return (uint32_t)p; }
    __device__ __forceinline__ static Part plain(Part p) { return (Part)((uint32_t)p & (kFlag - 1u)); }
    __device__ __forceinline__ static Part flagged(Part p) { return (Part)((uint32_t)p | kFlag); }
    // of a guard, the entry at the other end of the site's range
    __device__ __forceinline__ static uint32_t other_end(Part p) { return (uint32_t)plain(p); }
    __device__ __forceinline__ static Part guard(uint32_t to) { return (Part)(to | kFlag); }
    // partners of entry e[k]
    template <int NS>
    __device__ __forceinline__ static Part link(const uint32_t *e, int k)
    {
        return NS == 1 ? 0 : (Part)e[(k + 1) % NS];
    }
};
struct RecL8 : RecNext<0x8000u> {  // LDS, 8-bit codes: id = byte address of the code
    static constexpr bool kGlobal = false;
    uint32_t id0, poff;  // partner of id at poff + 2 * id
    __device__ __forceinline__ RecL8(uint32_t i, uint32_t p) : id0(i), poff(p) {}
    __device__ __forceinline__ uint32_t code(uint32_t id) const { return *lds_at<lds_u8>(id); }
    __device__ __forceinline__ Part part(uint32_t id) const { return *lds_at<lds_i16>(poff + 2u * id); }
    __device__ __forceinline__ void set_code(uint32_t id, uint32_t c) const
    {
        *lds_at<lds_u8>(id) = (uint8_t)c;
    }
    __device__ __forceinline__ void set_part(uint32_t id, Part p) const
    {
        *lds_at<lds_u16>(poff + 2u * id) = (uint16_t)p;
    }
};
struct RecL16 : RecNext<0x8000u> {  // LDS, 16-bit codes: id = half the byte address of the code
    static constexpr bool kGlobal = false;
    uint32_t id0, poff;  // partner of id at poff + 2 * id
    __device__ __forceinline__ RecL16(uint32_t i, uint32_t p) : id0(i), poff(p) {}
    __device__ __forceinline__ uint32_t code(uint32_t id) const { return *lds_at<lds_u16>(2u * id); }
    __device__ __forceinline__ Part part(uint32_t id) const { return *lds_at<lds_i16>(poff + 2u * id); }
    __device__ __forceinline__ void set_code(uint32_t id, uint32_t c) const
    {
        *lds_at<lds_u16>(2u * id) = (uint16_t)c;
    }
    __device__ __forceinline__ void set_part(uint32_t id, Part p) const
    {
        *lds_at<lds_u16>(poff + 2u * id) = (uint16_t)p;
    }
};
template <class C>
struct RecG : RecNext<0x80000000u> {  // global memory; every lane stores, so each lane's own later load is ordered after it
    static constexpr bool kGlobal = true;
    gmem<uint32_t> *p;
    gmem<C> *c;
    uint32_t n;  // entries
    static constexpr uint32_t id0 = 0;
    __device__ __forceinline__ RecG(gmem<uint32_t> *p_, gmem<C> *c_, uint32_t n_) : p(p_), c(c_), n(n_) {}
    __device__ __forceinline__ uint32_t code(uint32_t id) const { return c[id]; }
    __device__ __forceinline__ Part part(uint32_t id) const { return (Part)p[id]; }
    __device__ __forceinline__ void set_code(uint32_t id, uint32_t x) const { c[id] = (C)x; }
    __device__ __forceinline__ void set_part(uint32_t id, Part x) const { p[id] = (uint32_t)x; }
};
// Global memory, bonds of three and four sites: all partners of an entry in one
// 8-byte load, where a chain of partners costs one more trip to L2 per site and step.
// Ids have 31 bits with three sites, 21 with four.
template <int NS>
struct RecGAll {
    static constexpr bool kGlobal = true;
    static constexpr uint32_t kBits = NS == 3 ? 32 : 21;
    static constexpr uint32_t kMaxIds = NS == 3 ? 1u << 31 : 1u << 21;
    typedef uint64_t Part;
    gmem<uint64_t> *p;
    gmem<uint16_t> *c;
    uint32_t n;  // entries
    static constexpr uint32_t id0 = 0;
    __device__ __forceinline__ static uint32_t id(Part p, int k)
    {
        return (uint32_t)((p >> (kBits * k)) & (kMaxIds - 1u));
    }
    __device__ __forceinline__ static uint32_t top(Part p) { return (uint32_t)(p >> 32); }
    __device__ __forceinline__ static Part plain(Part p) { return p & ~(1ull << 63); }
    __device__ __forceinline__ static Part flagged(Part p) { return p | 1ull << 63; }
    __device__ __forceinline__ static uint32_t other_end(Part p) { return id(p, 0); }
    __device__ __forceinline__ static Part guard(uint32_t to) { return (Part)to | 1ull << 63; }
    template <int>
    __device__ __forceinline__ static Part link(const uint32_t *e, int k)
    {
        Part x = 0;
#pragma unroll
        for (int j = 1; j < NS; ++j)
            x |= (Part)e[(k + j) % NS] << (kBits * (j - 1));
        return x;
    }
    __device__ __forceinline__ RecGAll(gmem<uint64_t> *p_, gmem<uint16_t> *c_, uint32_t n_) : p(p_), c(c_), n(n_) {}
    __device__ __forceinline__ uint32_t code(uint32_t id) const { return c[id]; }
    __device__ __forceinline__ Part part(uint32_t id) const { return p[id]; }
    __device__ __forceinline__ void set_code(uint32_t id, uint32_t x) const { c[id] = (uint16_t)x; }
    __device__ __forceinline__ void set_part(uint32_t id, Part x) const { p[id] = x; }
};
// The same with the codes in LDS, byte address base on: a step then stores nothing to
// global memory.  Ring of 1000 three-site bonds at beta = 12 (n = 16400), 64 walkers:
// 45 ms per sweep with a chain of partners and codes in global memory, 31.6 without the
// chain, 28.0 with the codes in LDS, 22.2 now (WormHop out of scratch memory).
template <int NS, class C>
struct RecHAll : RecGAll<NS> {
    typedef __attribute__((address_space(3))) C lds_c;
    uint32_t base;
    __device__ __forceinline__ RecHAll(gmem<uint64_t> *p_, uint32_t b, uint32_t n_)
        : RecGAll<NS>(p_, nullptr, n_), base(b)
    {
    }
    __device__ __forceinline__ lds_c *at(uint32_t id) const { return lds_at<lds_c>(base + (uint32_t)sizeof(C) * id); }
    __device__ __forceinline__ uint32_t code(uint32_t id) const { return *at(id); }
    __device__ __forceinline__ void set_code(uint32_t id, uint32_t x) const { *at(id) = (C)x; }
};
// entries of an operator behind q[0], whose partners are pt (not flagged)
template <int NS, class R>
__device__ __forceinline__ void rec_others(const R &rec, int32_t pt, uint32_t *q)
{
    if constexpr (NS > 1)
        q[1] = (uint32_t)pt;
#pragma unroll
    for (int j = 2; j < NS; ++j)
        q[j] = (uint32_t)R::plain(rec.part(q[j - 1]));
}
template <int NS, class R>
__device__ __forceinline__ void rec_others(const R &, uint64_t pt, uint32_t *q)
{
#pragma unroll
    for (int j = 1; j < NS; ++j)
        q[j] = R::id(pt, j - 1);
}
__device__ __forceinline__ int32_t uni_part(int32_t p) { return (int32_t)uni((uint32_t)p); }
__device__ __forceinline__ uint64_t uni_part(uint64_t p) { return uni64(p); }

// ------------------------------------------------------------------ stream
// The walker's Philox words in registers: lane l holds word bbase + l (bbase
// even) and the word's row in the exit table.  All members but the three
// per-lane words are wave-uniform; every call is made by the whole wave.
struct WormStream {
    uint32_t wlo, whi, row;
    uint64_t key, bbase;
    uint32_t off;  // next word is bbase + off, off <= 64
    // entry words of the slots that the lanes' words would start a worm at,
    // loaded with the words where worms are short (ahead): the lookup then
    // passes under the steps, where it would be waited for at each start
    const uint32_t *ent;
    uint32_t L, legs, ahead;
    uint32_t slot, e0, e1;  // per lane: the slot drawn by the word, its entry word(s)
    uint64_t reject;        // lanes whose word may be rejected as a slot or leg draw
    __device__ __forceinline__ void slots()
    {
        const uint64_t a = (uint64_t)wlo * L, b = (uint64_t)whi * L + (a >> 32);
        slot = (uint32_t)(b >> 32);
        bool rej = (uint32_t)b == 0u && (uint32_t)a < L;  // low half of word * L below L
        if (legs == 6u)
            rej |= word() * 6ull < 6ull;
        reject = __builtin_amdgcn_ballot_w64(rej);
    }
    __device__ __forceinline__ void entries()
    {
        slots();
        const gmem<uint32_t> *g = as_global(ent) + (size_t)(legs > 4u ? 2u : 1u) * slot;
        e0 = g[0];
        e1 = legs > 4u ? g[1] : 0u;
    }
    template <class T>
    __device__ __forceinline__ void fill(const T &tab)
    {
        const uint32_t lane = threadIdx.x;
        uint32_t o0, o1, o2, o3;
        philox_block((bbase >> 1) + (lane >> 1), key, o0, o1, o2, o3);
        wlo = (lane & 1u) ? o2 : o0;
        whi = (lane & 1u) ? o3 : o1;
        row = tab.row_of((((uint64_t)whi << 32) | wlo) >> 11);
        if (ahead)
            entries();
    }
    template <class T>
    __device__ __forceinline__ void start(uint64_t k, uint64_t ctr, const T &tab)
    {
        slot = e0 = e1 = 0u;
        reject = 0ull;
        key = k;
        bbase = ctr & ~1ull;
        off = (uint32_t)(ctr & 1u);
        fill(tab);
    }
    __device__ __forceinline__ uint64_t ctr() const { return bbase + off; }
    // reload so that the next word is at lane 0 or 1
    template <class T>
    __device__ __forceinline__ void reload(const T &tab)
    {
        const uint64_t c = bbase + off;
        bbase = c & ~1ull;
        off = (uint32_t)(c & 1u);
        fill(tab);
    }
    __device__ __forceinline__ uint64_t word() const { return ((uint64_t)whi << 32) | wlo; }
    __device__ __forceinline__ uint64_t word_at(uint32_t k) const
    {
        return ((uint64_t)rdlane(whi, k) << 32) | rdlane(wlo, k);
    }
    template <class T>
    __device__ __forceinline__ uint64_t next(const T &tab)
    {
        if (off >= 64u)
            reload(tab);
        const uint64_t x = word_at(off);
        off += 1u;
        return x;
    }
    template <class T>
    __device__ __forceinline__ uint64_t range(uint64_t s, const T &tab)
    {
        uint64_t x = next(tab);
        uint64_t lo = x * s, hi = __umul64hi(x, s);
        if (lo < s) {
            const uint64_t t = (0ull - s) % s;
            while (lo < t) {
                x = next(tab);
                lo = x * s;
                hi = __umul64hi(x, s);
            }
        }
        return hi;
    }
};

// Where the worm update of one walker finds things (uniform, by value).
struct WormCtx {
    const uint32_t *ops;
    const uint32_t *idx;   // [slot][NS]
    uint32_t *ent;         // entry words of the slots (LDS layouts)
    int32_t *first;        // [site] first entry (global records)
    const int32_t *last;   // [site] operators on the site
    const uint4 *wbond;
    const uint2 *wcode;
    const uint8_t *site_dims;
    lds_u16 *sb;           // [site] first entry (LDS layouts)
    uint32_t L, n, N, n_bonds, guard;
};

template <int NS>
__device__ __forceinline__ uint32_t wbond_site(const uint4 &b, int k)
{
    const uint32_t w = k < 2 ? b.x : b.y;
    return (k & 1) ? w >> 16 : w & 0xFFFFu;
}

// inclusive prefix sum over the wave (as wave_incl_scan)
template <int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kCtrl, kRowMask, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t x)
{
    x += dpp_u32<0x111, 0xf>(x);
    x += dpp_u32<0x112, 0xf>(x);
    x += dpp_u32<0x114, 0xf>(x);
    x += dpp_u32<0x118, 0xf>(x);
    x += dpp_u32<0x142, 0xa>(x);
    x += dpp_u32<0x143, 0xc>(x);
    return x;
}

// Build the records of a walker: the entry ranges of the sites from their operator
// counts, then every operator's entries from its slot's idx words (8 chunks of
// 64 slots per pass, their loads in flight together).  Returns false when the
// counts do not belong to the operator string; all ids written are in range.
// A function of its own so that its registers stay out of the chase's.
template <int NS, class R>
__device__ __noinline__ bool worm_stage(R rec, WormCtx x)
{
    constexpr int LG = WormNS<NS>::LG, K = 8;
    const uint32_t lane = threadIdx.x;
    uint32_t run = rec.id0;
    uint32_t ops_on_sites = 0;
    for (uint32_t s0 = 0; s0 < x.N; s0 += 64) {
        const uint32_t s = s0 + lane;
        const bool in = s < x.N;
        const uint32_t cnt = in ? (uint32_t)as_global(x.last)[s] : 0u;
        // more operators on a site than in the string: not this string's counts
        if (wave_any(cnt > x.n))
            return false;
        const uint32_t incl = wave_incl_scan_u32(in ? cnt + 2u : 0u);
        const uint32_t total = rdlane(incl, 63);
        ops_on_sites += total - 2u * (x.N - s0 < 64u ? x.N - s0 : 64u);
        if (ops_on_sites > NS * x.n)
            return false;
        const uint32_t g = run + incl - (cnt + 2u);
        if (in) {
            if constexpr (R::kGlobal)
                as_global(x.first)[s] = (int32_t)(g + 1u);
            else
                x.sb[s] = (uint16_t)(g + 1u);
            rec.set_code(g, x.guard);
            rec.set_code(g + cnt + 1u, x.guard);
            rec.set_part(g, R::guard(g + cnt));
            rec.set_part(g + cnt + 1u, R::guard(g + 1u));
        }
        run += total;
    }
    if (ops_on_sites != NS * x.n)
        return false;
    __syncthreads();
    bool bad = false;
    uint32_t found = 0;
    const gmem<uint32_t> *gops = as_global(x.ops), *gidx = as_global(x.idx);
    const gmem<uint4> *gb = as_global(x.wbond);
    for (uint32_t b0 = 0; b0 < x.L; b0 += 64 * K) {
        uint32_t op[K], ix[K][NS];
        uint4 wb[K];
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const uint32_t p = b0 + 64u * u + lane;
            op[u] = p < x.L ? gops[p] : 0u;
#pragma unroll
            for (int k = 0; k < NS; ++k)
                ix[u][k] = p < x.L ? gidx[(size_t)NS * p + k] : 0u;
        }
#pragma unroll
        for (int u = 0; u < K; ++u) {
            uint32_t bd = op_bond(op[u]);
            if (bd >= x.n_bonds) {
                bad = true;
                bd = 0u;
            }
            const gmem<uint4> &q = gb[bd];
            wb[u] = make_uint4(q.x, q.y, q.z, 0u);
        }
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const uint32_t p = b0 + 64u * u + lane;
            uint32_t e[NS];
            bool ok = op[u] != 0u;
            found += ok ? 1u : 0u;
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                e[k] = rec.id0;
                if (ok) {
                    const uint32_t s = wbond_site<NS>(wb[u], k);
                    uint32_t f, c;
                    if constexpr (R::kGlobal) {
                        f = (uint32_t)as_global(x.first)[s];
                        c = (uint32_t)as_global(x.last)[s];
                    } else {
                        f = x.sb[s];
                        c = (s + 1u < x.N ? (uint32_t)x.sb[s + 1u] : run + 1u) - f - 2u;
                    }
                    if (ix[u][k] >= c) {
                        bad = true;
                        ok = false;
                    }
                    e[k] = f + ix[u][k];
                }
            }
            if (ok) {
                const uint32_t c = (wb[u].z + (op_vcode(op[u]) >> 1)) << LG;
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    rec.set_code(e[k], c | (uint32_t)k);
                    rec.set_part(e[k], R::template link<NS>(e, k));
                }
            }
            if constexpr (!R::kGlobal) {
                if (p < x.L) {
                    if constexpr (NS <= 2) {
                        as_global(x.ent)[p] = !ok ? ~0u : e[0] | (NS == 2 ? e[NS - 1] << 16 : 0u);
                    } else {
                        gmem<uint2> *g2 = (gmem<uint2> *)as_global(x.ent);
                        gmem<uint2> &d = g2[p];
                        d.x = !ok ? ~0u : e[0] | e[1] << 16;
                        d.y = !ok ? ~0u : e[2] | (NS == 4 ? e[NS - 1] << 16 : 0u);
                    }
                }
            }
        }
    }
    const uint32_t all = rdlane(wave_incl_scan_u32(found), 63);
    return !wave_any(bad) && all == x.n;
}

// Entries of slot p's operator: false for an identity slot.
template <int NS, class R>
__device__ __forceinline__ bool worm_entry(const WormCtx &x, const R &, uint32_t p, uint32_t pos,
                                           uint32_t &e)
{
    if constexpr (R::kGlobal) {
        const uint32_t op = as_global(x.ops)[p];
        if (op == 0u)
            return false;
        const uint4 b = x.wbond[op_bond(op)];
        const uint32_t w = pos < 2u ? b.x : b.y;
        const uint32_t s = (pos & 1u) ? w >> 16 : w & 0xFFFFu;
        e = (uint32_t)as_global(x.first)[s] + as_global(x.idx)[(size_t)NS * p + pos];
        return true;
    } else if constexpr (NS <= 2) {
        const uint32_t w = as_global(x.ent)[p];
        e = pos ? w >> 16 : w & 0xFFFFu;
        return w != ~0u;
    } else {
        const uint32_t w = as_global(x.ent)[2u * (size_t)p + (pos >> 1)];
        e = (pos & 1u) ? w >> 16 : w & 0xFFFFu;
        return (w & 0xFFFFu) != 0xFFFFu;
    }
}

// A worm's start: slot, leg and entry, and the stream behind the draws.
struct WormBegin {
    WormStream rs;
    uint32_t p, leg;
};

// The draws of a worm start one by one (a Lemire rejection shifts them).
template <int NS, class R, class T>
__device__ __noinline__ WormBegin worm_start_exact(WormCtx x, R rec, WormStream rs, T tab)
{
    for (;;) {
        const uint32_t p = (uint32_t)uni64(rs.range((uint64_t)x.L, tab));
        const uint32_t leg = uni((uint32_t)rs.range(2ull * NS, tab));
        uint32_t e = 0;
        if (uni((uint32_t)worm_entry<NS>(x, rec, p, 0u, e)))
            return WormBegin{rs, p, leg};
    }
}

// Worm start (sse.jl:241-247): (slot, leg) pairs are drawn until the slot
// holds an operator.  All attempts that the buffered words allow are looked up
// at once, one per lane, and the first that finds an operator counts; the words
// before it are used up.  Returns the entry that the leg belongs to; p receives
// the slot, leg the leg.
template <int NS, class R, class T>
__device__ __forceinline__ uint32_t worm_start(const WormCtx &x, const R &rec, WormStream &rs,
                                               const T &tab, uint32_t &p, uint32_t &leg)
{
    for (;;) {
        if (rs.off + 2u > 64u)
            rs.reload(tab);
        const uint32_t off = rs.off;
        if constexpr (R::kGlobal)
            rs.slots();
        else if (!rs.ahead)
            rs.entries();
        uint32_t e = 0;
        if (__builtin_expect((rs.reject >> off) != 0ull, 0)) {
            const WormBegin g = worm_start_exact<NS, R, T>(x, rec, rs, tab);
            rs.wlo = g.rs.wlo;
            rs.whi = g.rs.whi;
            rs.row = g.rs.row;
            rs.slot = g.rs.slot;
            rs.e0 = g.rs.e0;
            rs.e1 = g.rs.e1;
            rs.off = uni(g.rs.off);
            rs.bbase = uni64(g.rs.bbase);
            rs.reject = uni64(g.rs.reject);
            leg = uni(g.leg);
            p = uni(g.p);
            worm_entry<NS>(x, rec, p, NS == 1 ? 0u : leg % NS, e);
            return uni(e);
        }
        // attempts start at words off, off + 2, ... with their leg's word in the buffer
        const uint64_t cand = (0x5555555555555555ull << (off & 1u)) & (~0ull << off) & (~0ull >> 1);
        bool hit;
        if constexpr (R::kGlobal)
            hit = ((cand >> threadIdx.x) & 1ull) && worm_entry<NS>(x, rec, rs.slot, 0u, e);
        else
            hit = rs.e0 != ~0u;
        const uint64_t hits = __builtin_amdgcn_ballot_w64(hit) & cand;
        if (hits) {
            const uint32_t j = (uint32_t)__builtin_ctzll(hits);
            // rand(1:legs): the high half of word * legs
            const uint32_t wh = rdlane(rs.whi, j + 1u), wl = rdlane(rs.wlo, j + 1u);
            leg = (uint32_t)(((uint64_t)wh * (2u * NS) + (((uint64_t)wl * (2u * NS)) >> 32)) >> 32);
            rs.off = j + 2u;
            p = rdlane(rs.slot, j);
            const uint32_t pos = NS == 1 ? 0u : leg % NS;
            if constexpr (R::kGlobal) {
                worm_entry<NS>(x, rec, p, pos, e);
                return uni(e);
            } else {
                const uint32_t ew = NS > 2 && pos >= 2u ? rdlane(rs.e1, j) : rdlane(rs.e0, j);
                return (pos & 1u) ? ew >> 16 : ew & 0xFFFFu;
            }
        }
        rs.off = off + 2u * (uint32_t)__popcll(cand);
    }
}

// The exact scatter (vertex_data.jl:113-125) of entry (c, port) for a word whose
// exit entry holds none: more than four exits, a fall-through, an invalid
// transition.  Wide exit word, or kWormSpecial for the last two.
template <int NS>
__device__ __noinline__ uint64_t worm_exact(const DevModel *mp, uint32_t c, uint32_t port, uint64_t m53)
{
    const DevModel &m = *mp;
    constexpr int LG = WormNS<NS>::LG;
    const uint32_t code = c >> LG, pos = c & ((1u << LG) - 1u);
    const uint32_t side = port & 1u, wf = port >> 1;
    const uint2 wc = m.wcode[code];
    const DevVD &vd = m.types[wc.y >> 10];
    const uint32_t v = (wc.y & 1023u) >> 1;
    if ((int)wf >= vd.max_worm)
        return kWormSpecial;
    const int ix = ((int)v * vd.max_worm + (int)wf) * 2 * NS + (int)(pos + NS * side);
    const int32_t o = vd.toff[ix], cnt = vd.tcnt[ix];
    if (o < 0)
        return kWormSpecial;
    const double r = (double)m53 * 0x1.0p-53;
    for (int32_t j = o; j < o + cnt; ++j)
        if (r < vd.cum[j]) {
            const uint32_t lo = vd.eleg[j], up = lo >= (uint32_t)NS ? 1u : 0u;
            // the worm enters the next operator on the far side
            return worm_word(worm_leg(NS, pos, lo), 2u * ((uint32_t)vd.ewrm[j] - 1u) + (up ^ 1u),
                             (code - v + ((uint32_t)vd.tgt[j] >> 1)) << LG);
        }
    return kWormSpecial;
}

// The entries behind an operator's legs, packed ahead of the exit, and the one
// that the exit leg leads to.
template <int NS, bool kWide>
struct WormHop {
    uint64_t all;
    // members of their own: of an array the compiler makes a select between its
    // elements' addresses, and keeps it in scratch memory (a step of three-site bonds
    // with partners in global memory: 404 ns with it, 298 without)
    uint32_t q0, q1, q2, q3;
    __device__ __forceinline__ explicit WormHop(const uint32_t *e)
    {
        q0 = e[0];
        q1 = NS > 1 ? e[NS > 1 ? 1 : 0] : 0u;
        q2 = NS > 2 ? e[NS > 2 ? 2 : 0] : 0u;
        q3 = NS > 3 ? e[NS > 3 ? 3 : 0] : 0u;
        if constexpr (!kWide && NS == 2) {
            const uint32_t pe = e[0] | e[1] << 16;
            all = (uint64_t)(pe - 0x00010001u) | (uint64_t)(pe + 0x00010001u) << 32;
        } else if constexpr (!kWide && NS >= 3) {
            all = (uint64_t)(e[0] | e[1] << 16) | (uint64_t)e[2] << 32;
            if constexpr (NS == 4)
                all |= (uint64_t)e[NS - 1] << 48;
        }
    }
    __device__ __forceinline__ uint32_t next(uint32_t sh) const
    {
        if constexpr (!kWide && NS == 2) {
            return (uint32_t)(all >> (sh & 63u)) & 0xFFFFu;
        } else if constexpr (!kWide && NS >= 3) {
            const uint32_t t = (uint32_t)(all >> (sh & 0x30u)) & 0xFFFFu;
            return (sh & 64u) ? t + 1u : t - 1u;
        } else {
            const bool up = NS <= 2 ? (sh & 32u) != 0u : (sh & 64u) != 0u;
            uint32_t t = q0;
            if constexpr (NS >= 2)
                t = (sh & 16u) ? q1 : t;
            if constexpr (NS >= 3) {
                const uint32_t h = NS == 4 && (sh & 16u) ? q3 : q2;
                t = (sh & 32u) ? h : t;
            }
            return up ? t + 1u : t - 1u;
        }
    }
};

// All worms of one walker (sse.jl:193-303).  Returns an error code (0 = ok).
template <int NS, class R, class T>
__device__ __forceinline__ int worm_chase(const WormCtx &x, const DevModel &m, WormStream &rs, const R &rec,
                                          const T &tab, int64_t nworms, double &total, int64_t &scat)
{
    if (x.n == 0u)
        return 0;  // worm_traverse! returns 0 without draws (sse.jl:234-236)
    // a vector zero: what is added to it stays in vector registers
    uint32_t vz;
    asm volatile("v_mov_b32 %0, 0" : "=v"(vz));
    // read once: every store would make the compiler read them again
    const uint32_t wdim = uni((uint32_t)m.w_dim), wmw = uni((uint32_t)m.w_mw);
    for (int64_t k = 0; k < nworms; ++k) {
        uint32_t p0, leg0;
        const uint32_t e0 = worm_start<NS>(x, rec, rs, tab, p0, leg0);
        const uint32_t pos0 = NS == 1 ? 0u : leg0 % NS, up0 = leg0 >= NS ? 1u : 0u;
        uint32_t dim0 = wdim;
        if (dim0 == 0u) {
            const uint4 b = x.wbond[op_bond(x.ops[p0])];
            const uint32_t w = pos0 < 2u ? b.x : b.y;
            dim0 = uni((uint32_t)x.site_dims[(pos0 & 1u) ? w >> 16 : w & 0xFFFFu]);
        }
        // worm function, 0-based (sse.jl:251); rand(1:1) still takes a word
        uint32_t wf0 = 0;
        if (dim0 == 2u)
            (void)rs.next(tab);
        else
            wf0 = uni((uint32_t)rs.range((uint64_t)(dim0 - 1u), tab));
        if (wf0 >= wmw)
            return SSE_ERR_STATE;
        // closing tests (sse.jl:290-297): the worm leaves through its start leg
        // with the inverse worm (it arrives at ea, the entry behind that leg,
        // with port porta), or re-enters the start leg (entry e0, port port0)
        const uint32_t port0 = 2u * wf0 + up0;
        const uint32_t ea = up0 ? e0 + 1u : e0 - 1u;
        const uint32_t porta = 2u * (dim0 - wf0 - 2u) + (up0 ^ 1u);
        uint32_t e = e0 + vz, port = port0 + vz;
        uint32_t c = rec.code(e);
        typename R::Part pt = rec.part(e);
        const typename R::Part part0 = uni_part(pt), parta = uni_part(rec.part(ea + vz));
        rec.set_part(e0 + vz, R::flagged(part0));
        rec.set_part(ea + vz, R::flagged(parta));
        const uint64_t ctr0 = rs.ctr();
        const uint32_t row0 = rdlane(rs.row, rs.off & 63u);
        uint32_t row = row0;
        typename T::Word wd = tab.load(row, c, port);
        // sse.jl:274-300.  A run of steps ends at a flag, at a word without an
        // exit or when the buffered words are used up; the entry, its code and
        // the exit word of the next step are loaded already.
        uint32_t reentry = 0;
        for (;;) {
            if (__builtin_expect(rs.off >= 64u, 0)) {
                rs.reload(tab);
                row = rdlane(rs.row, rs.off);
                wd = tab.load(row, c, port);
            }
            uint32_t off = uni(rs.off);
            row = uni(row);
            uint32_t q[NS], cq, pq, rq, none, ends;
            bool stop = false;  // (kScalar)
            // scalar loads return out of order: with one in flight from before the
            // loop, its first instruction would wait for the table in every step
            if constexpr (T::kScalar)
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            do {
                q[0] = e;
                rec_others<NS>(rec, pt, q);
                const WormHop<NS, R::kGlobal> hop(q);
                cq = c;
                pq = port;
                rq = T::kScalar ? 0u : row;
                // the exit's own chain starts here, with all that does not
                // need it done under its load
                __builtin_amdgcn_sched_barrier(0);
                const typename T::Pick pick = tab.pick(wd, row);
                uint32_t nx = hop.next(T::sh(pick));
                if constexpr (R::kGlobal) {
                    bool out = nx >= rec.n;
#pragma unroll
                    for (int j = 1; j < NS; ++j)
                        out |= q[j] >= rec.n;
                    if (wave_any(out && (int32_t)tab.exit(pick, cq).none >= 0))
                        return SSE_ERR_STATE;
                    nx = out ? 0u : nx;
                }
                // the next entry is never one of the operator's own (those
                // lie in other sites' ranges or behind a guard), so its loads
                // go before the stores
                c = rec.code(nx);
                pt = rec.part(nx);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (T::kScalar)
                    rq = T::unsure(wd, row);
                const WormExit<NS> ex = tab.exit(pick, cq);
                none = ex.none;
                if constexpr (!T::kScalar) {
#pragma unroll
                    for (int j = 0; j < NS; ++j)
                        rec.set_code(q[j], ex.c[j]);
                }
                off += 1u;
                e = nx;
                port = ex.port;
                row = rdlane(rs.row, off & 63u);
                if constexpr (!T::kScalar)
                    wd = tab.load(row, c, port);
                // one condition, one branch: a flag, no exit, or no word left
                ends = (63u - off) | (T::kNone ? rq : 0u);
                if constexpr (T::kNone)
                    ends |= none;
                // a wait for LDS is a wait for the scalar load too, so that one
                // leaves after the test of the flag
                if constexpr (T::kScalar) {
                    stop = wave_any((int32_t)(R::top(pt) | ends) < 0);
                    __builtin_amdgcn_sched_barrier(0);
                    wd = tab.load(row, c, port);
#pragma unroll
                    for (int j = 0; j < NS; ++j)
                        rec.set_code(q[j], ex.c[j]);
                }
            } while (T::kScalar ? !stop : !wave_any((int32_t)(R::top(pt) | ends) < 0));
            rs.off = off;
            if constexpr (T::kNone) {
                if (__builtin_expect(wave_any((int32_t)(none | rq) < 0), 0)) {
                    // take the step back and look its exit up exactly
                    const uint64_t o = worm_exact<NS>(&m, uni(cq), uni(pq), rs.word_at(off - 1u) >> 11);
                    if ((int64_t)uni64(o) < 0)
                        return SSE_ERR_SCATTER;
                    const uint32_t nc = (uint32_t)(o >> 32);
                    uint32_t pos = cq & ((1u << WormNS<NS>::LG) - 1u);
#pragma unroll
                    for (int j = 0; j < NS; ++j) {
                        rec.set_code(q[j], nc | pos);
                        pos = pos + 1u == NS ? 0u : pos + 1u;
                    }
                    e = WormHop<NS, R::kGlobal>(q).next((uint32_t)o & 0x7Fu) + vz;
                    port = (uint32_t)o >> 8;
                    if constexpr (R::kGlobal) {
                        if (wave_any(e >= rec.n))
                            return SSE_ERR_STATE;
                    }
                    c = rec.code(e);
                    pt = rec.part(e);
                    wd = tab.load(row, c, port);
                }
            }
            if (!wave_any((int32_t)R::top(pt) < 0))
                continue;
            // a flagged entry: the worm's end, a guard, or neither
            if (wave_any(e == ea && port == porta))
                break;
            if (wave_any(c == x.guard)) {
                e = R::other_end(pt);
                c = rec.code(e);
                pt = rec.part(e);
                wd = tab.load(row, c, port);
                if (!wave_any((int32_t)R::top(pt) < 0))
                    continue;
                // the start leg may be the one behind the guard
            }
            if (wave_any(e == e0 && port == port0)) {
                reentry = 1u;
                break;
            }
            pt = R::plain(pt);
        }
        rec.set_part(e0 + vz, part0);
        rec.set_part(ea + vz, parta);
        const uint64_t steps = rs.ctr() - ctr0;
        scat += (int64_t)steps;
        // worm length: scatters, + 1 when the worm closed on re-entry
        total += (double)(steps + reentry);
    }
    return 0;
}

// The worm-updated vertex codes back into the operator string, K chunks of 64
// slots per pass, their loads in flight together.
template <int NS, class R>
__device__ __noinline__ void worm_writeback(R rec, WormCtx x)
{
    constexpr int LG = WormNS<NS>::LG, K = 8;
    const uint32_t lane = threadIdx.x;
    gmem<uint32_t> *ops = as_global((uint32_t *)x.ops);
    const gmem<uint2> *wc = as_global(x.wcode);
    for (uint32_t b0 = 0; b0 < x.L; b0 += 64 * K) {
        uint32_t op[K], c[K];
        uint32_t ew[K];
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const uint32_t p = b0 + 64u * u + lane;
            op[u] = p < x.L ? ops[p] : 0u;
            if constexpr (!R::kGlobal)
                ew[u] = p < x.L ? as_global(x.ent)[(NS <= 2 ? 1u : 2u) * (size_t)p] & 0xFFFFu : 0u;
        }
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const uint32_t p = b0 + 64u * u + lane;
            c[u] = 0u;
            if (op[u] != 0u) {
                if constexpr (R::kGlobal) {
                    uint32_t e = 0;
                    worm_entry<NS>(x, rec, p, 0u, e);
                    ew[u] = e;
                }
                c[u] = rec.code(ew[u]) >> LG;
            }
        }
        uint32_t v[K];
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const gmem<uint2> &q = wc[c[u]];
            v[u] = q.y & 1023u;
        }
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const uint32_t nop = (op[u] & ~(1023u << 1)) | (v[u] << 1);
            if (op[u] != 0u && nop != op[u])
                ops[b0 + 64u * u + lane] = nop;
        }
    }
}

// State refresh (sse.jl:219-228): a site without operators draws a new state, in
// site order; one with operators takes the lower leg state of its first.
template <int NS, class R, class RS>
__device__ __forceinline__ void worm_refresh(const R &rec, const WormCtx &x, RS &rs, uint8_t *spins)
{
    constexpr int LG = WormNS<NS>::LG;
    const int lane = threadIdx.x;
    // sites in blocks of 32 so that one block draws at most 32 words (the
    // stream holds 64)
    for (uint32_t sb = 0; sb < x.N; sb += 32) {
        const uint32_t s = sb + lane;
        const bool vs = lane < 32 && s < x.N;
        const int32_t cnt = vs ? as_global(x.last)[s] : 1;
        const bool fr = vs && cnt == 0;
        const uint64_t frm = __ballot(fr);
        const int D = popc(frm);
        const uint64_t dim = vs ? (uint64_t)x.site_dims[s] : 1;
        bool reject = false;
        uint8_t val = 0;
        if (D > 0) {
            rs.ensure((uint32_t)D);
            // every lane takes part in the cross-lane read; lane s of the
            // refreshed sites uses word off + (its rank among them)
            const uint64_t w = rs.peek(fr ? (uint32_t)popc(frm & below_mask(lane)) : 0u);
            if (fr) {
                uint64_t lo = w * dim;
                if (lo < dim && lo < (0ull - dim) % dim)
                    reject = true;
                val = (uint8_t)(1 + __umul64hi(w, dim));
            }
        }
        if (vs && !fr) {
            uint32_t f;
            if constexpr (R::kGlobal)
                f = (uint32_t)as_global(x.first)[s];
            else
                f = x.sb[s];
            const uint32_t c = rec.code(f);
            val = (uint8_t)(x.wcode[c >> LG].x >> (8u * (c & ((1u << LG) - 1u))));
        }
        if (__ballot(reject)) {
            for (int i = 0; i < 32 && sb + i < x.N; ++i) {
                const bool fi = (frm >> i) & 1ull;
                uint8_t vi = 0;
                if (fi)
                    vi = (uint8_t)(1 + rs.range((uint64_t)x.site_dims[sb + i]));
                if (lane == i && fi)
                    val = vi;
            }
        } else {
            rs.advance((uint32_t)D);
        }
        if (vs)
            spins[s] = val;
    }
}

// stage, chase, refresh and write back with record layout R and exit table T
template <int NS, class R, class T>
__device__ __forceinline__ int worm_update(const DevWalker &w, const DevModel &m, const WormCtx &x,
                                           const R &rec, const T &tab, double &total, int64_t &scat,
                                           uint64_t &ctr)
{
    if (!worm_stage<NS, R>(rec, x))
        return SSE_ERR_STATE;
    __syncthreads();
    WormStream rs;
    rs.ent = x.ent;
    rs.L = x.L;
    rs.legs = 2u * NS;
    // worms of up to twice the buffered words' steps: every other buffer at
    // least starts one.  1536 dimer ladders (worms of 10 steps) 1.09 ms per sweep
    // against 1.11 without; above, no difference beyond the runs' own
    rs.ahead = !R::kGlobal && x.n != 0u && w.avg_worm_length < 128.0 ? 1u : 0u;
    rs.start(w.key, w.ctr, tab);
    const int err = worm_chase<NS>(x, m, rs, rec, tab, (int64_t)ceil(w.num_worms), total, scat);
    if (err)
        return err;
    __syncthreads();
    K2RegStream fs;
    fs.init(w.key, rs.ctr());
    worm_refresh<NS>(rec, x, fs, w.spins);
    ctr = fs.ctr();
    worm_writeback<NS, R>(rec, x);
    return 0;
}

// ------------------------------------------------------------------ layout choice
// LDS bytes of a walker's records with code width cb behind a table of tab bytes
__host__ __device__ inline size_t worm_lds_bytes(int ns, int64_t n, int64_t N, int cb, size_t tab)
{
    const size_t e = (size_t)(ns * n + 2 * N);
    return tab + ((cb * e + 15) & ~(size_t)15) + 2 * e + 2 * (size_t)N;
}
// 8-bit codes hold every code and the guard's
__host__ __device__ inline bool worm_small_codes(const DevModel &m)
{
    return ((int64_t)m.w_ncode << m.w_lg) <= 255;
}
__host__ __device__ inline size_t worm_table_bytes(const DevModel &m)
{
    if (m.wrow)
        return ((size_t)(m.w_nthr + 1) * m.w_nent * 4 + 15) & ~(size_t)15;
    return m.wexit ? (size_t)m.w_nent * 16 : 0;
}
// the table and, behind it, the copy of the threshold search
__host__ __device__ inline size_t worm_tables_bytes(const DevModel &m)
{
    const size_t t = worm_table_bytes(m);
    return t ? t + (size_t)m.w_rank : 0;
}
// LDS bytes with which a walker of n operators takes its fastest layout
__host__ __device__ inline size_t worm_lds_need(const DevModel &m, int64_t n)
{
    return worm_lds_bytes(m.nsb, n, m.n_sites, worm_small_codes(m) ? 1 : 2, worm_tables_bytes(m));
}

// copy a table into LDS (whole wave)
__device__ __forceinline__ void worm_copy_table(uint32_t dst, const void *src, size_t bytes)
{
    const gmem<u32x4> *g = as_global((const u32x4 *)src);
    lds_u32x4 *d = lds_at<lds_u32x4>(dst);
    const uint32_t n = (uint32_t)((bytes + 15) / 16);
    for (uint32_t i = threadIdx.x; i < n; i += 64)
        d[i] = g[i];
}

// the model's exit table and threshold search into LDS at byte address dst
__device__ __forceinline__ void worm_copy_tables(const DevModel &m, uint32_t dst, WormRank &rank)
{
    const size_t t = worm_table_bytes(m);
    worm_copy_table(dst, m.wrow ? (const void *)m.wrow : (const void *)m.wexit, t);
    if (m.w_rank) {
        worm_copy_table(dst + (uint32_t)t, m.wthr, (size_t)m.w_rank);
        rank.lds = dst + (uint32_t)t;
    }
}

// Worm update of walker wi.  mode (SSE_OPT_WORM_RECORDS) 0: records and table in
// LDS where they fit, the codes as narrow as they can be; 1: 16-bit codes and
// the global table; 2: global records; 3: as 0 with the global table.
template <int NS>
__device__ __forceinline__ void worm_walker(DevWalker *W, const DevModel *models, DevPool *pool, int wi,
                                            int full_sweep, int lds_bytes, int mode, char *lds_generic)
{
    const int lane = threadIdx.x;
    DevWalker w = W[wi];
    if (w.error || !w.active || w.retire)
        return;
    const DevModel &m = models[w.model];
    const bool therm = w.sweeps > w.thermalization;
    // byte address of the workgroup's LDS
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_u8 *)lds_generic;
    WormCtx x;
    x.ops = w.ops;
    x.idx = (const uint32_t *)w.links;
    x.ent = (uint32_t *)w.links + (size_t)NS * w.cap;
    x.first = w.first;
    x.last = w.last;
    x.wbond = m.wbond;
    x.wcode = m.wcode;
    x.site_dims = m.site_dims;
    x.sb = nullptr;
    x.L = (uint32_t)w.L;
    x.n = (uint32_t)w.n;
    x.N = (uint32_t)m.n_sites;
    x.n_bonds = (uint32_t)m.n_bonds;
    x.guard = (uint32_t)m.w_ncode << m.w_lg;
    WormRank rank{m.wthr, m.w_nthr, ~0u};
    const uint32_t ports = 2u * (uint32_t)m.w_mw;
    double total = 1.0;
    int64_t scat = 0;
    uint64_t ctr = w.ctr;
    int err = SSE_ERR_STATE;
    const bool small = worm_small_codes(m) && mode != 1;
    const int cb = small ? 1 : 2;
    const bool u16codes = x.guard <= 65535u;
    const size_t E = (size_t)NS * x.n + 2u * x.N;
    size_t tb = mode == 1 || mode == 3 ? 0 : worm_tables_bytes(m);
    auto fits = [&](size_t t) {
        return mode != 2 && u16codes && worm_lds_bytes(NS, x.n, x.N, cb, t) <= (size_t)lds_bytes &&
               (t + 1024) / cb + E < kWormIds;
    };
    bool in_lds = fits(tb);
    if (!in_lds && tb && fits(0)) {
        in_lds = true;
        tb = 0;
    }
    const uint32_t id0 = (lds + (uint32_t)tb) / (uint32_t)cb;
    const uint32_t pbase = lds + (uint32_t)(tb + ((cb * E + 15) & ~(size_t)15));
    const uint32_t poff = pbase - 2u * id0;
    if (in_lds)
        x.sb = lds_at<lds_u16>(pbase + 2u * (uint32_t)E);
    const TabWide<NS> wide{ports, m.wwide};
    const bool rows = NS <= 2 && m.wrow != nullptr;
#define WORM_RUN(R, T) err = worm_update<NS>(w, m, x, R, T, total, scat, ctr)
    if (in_lds && tb) {
        worm_copy_tables(m, lds, rank);
        if (rows) {
            if constexpr (NS <= 2) {
                const TabRows<NS> t{rank, lds, (uint32_t)m.w_nent * 4u, ports};
                WORM_RUN((RecL8{id0, poff}), t);
            }
        } else {
            const TabExits<NS> t{rank, lds, ports};
            if (small)
                WORM_RUN((RecL8{id0, poff}), t);
            else
                WORM_RUN((RecL16{id0, poff}), t);
        }
    } else if (in_lds) {
        if (small)
            WORM_RUN((RecL8{id0, poff}), wide);
        else
            WORM_RUN((RecL16{id0, poff}), wide);
    } else {
        gmem<uint32_t> *gp = as_global(x.ent);
        const uint32_t ne = (uint32_t)E;
        const size_t cofs = (size_t)NS * w.cap + 2u * (size_t)pool->max_sites;
        if (!u16codes) {
            WORM_RUN((RecG<uint32_t>{gp, gp + cofs, ne}), wide);
        } else if (rows && worm_tables_bytes(m) <= (size_t)lds_bytes) {
            if constexpr (NS <= 2) {
                worm_copy_tables(m, lds, rank);
                const TabRows<NS> t{rank, lds, (uint32_t)m.w_nent * 4u, ports};
                WORM_RUN((RecG<uint16_t>{gp, (gmem<uint16_t> *)(gp + cofs), ne}), t);
            }
        } else {
            // 8 bytes of partners per entry where the slab, which has 4 per
            // possible one, holds them: cutoffs are about twice the operator
            // count and more
            const size_t room = (4u + (size_t)worm_code_bytes(m)) * ((size_t)NS * w.cap + 2u * (size_t)pool->max_sites);
            bool all = false;
            if constexpr (NS >= 3) {
                all = 10u * E <= room && E <= RecGAll<NS>::kMaxIds;
                gmem<uint64_t> *ga = (gmem<uint64_t> *)gp;
                if (all && mode != 2 && E * (size_t)cb <= (size_t)lds_bytes) {
                    if (small)
                        WORM_RUN((RecHAll<NS, uint8_t>{ga, lds, ne}), wide);
                    else
                        WORM_RUN((RecHAll<NS, uint16_t>{ga, lds, ne}), wide);
                } else if (all) {
                    WORM_RUN((RecGAll<NS>{ga, (gmem<uint16_t> *)(ga + ne), ne}), wide);
                }
            }
            if (!all)
                WORM_RUN((RecG<uint16_t>{gp, (gmem<uint16_t> *)(gp + cofs), ne}), wide);
        }
    }
#undef WORM_RUN
    if (err) {
        if (lane == 0) {
            W[wi].error = err;
            flag_error(pool, err);
        }
        return;
    }
    w.last_scatter = scat;
    worm_controller(w, total, therm);
    if (lane == 0) {
        DevWalker &o = W[wi];
        o.ctr = ctr;
        o.avg_worm_length = w.avg_worm_length;
        o.num_worms = w.num_worms;
        o.last_scatter = w.last_scatter;
        o.last_total = w.last_total;
        o.last_wlf = w.last_wlf;
        if (full_sweep) {
            o.sweeps = w.sweeps + 1;
            o.acc_L = w.acc_L + w.L;
            o.acc_n = w.acc_n + w.n;
            o.acc_W = w.acc_W + scat;
            o.acc_sweeps = w.acc_sweeps + 1;
            if (w.remaining > 0) {
                o.remaining = w.remaining - 1;
                if (w.remaining == 1)
                    o.retire = 1;
            }
        }
    }
}
