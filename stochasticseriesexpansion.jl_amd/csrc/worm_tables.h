// worm_tables.h -- host side of the worm update's exit tables: the images that
// sse_worm.h reads, from the transition lists of a model.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../../include/ssegpu.h"
#include "sse_common.h"

// Host image of a model's worm tables (DevModel::w*).
struct WormTables {
    std::vector<uint4> bond;
    std::vector<uint2> code;
    std::vector<uint64_t> thr;
    std::vector<uint32_t> row;
    std::vector<uint4> exit;
    std::vector<uint32_t> wide;
    int nthr = 0, lg = 0, mw = 1, dim = 0, rank = 0, nent = 0;
};

// Exit rows save a step its compares: against 16-byte exits 90 instead of 126 ns (one
// walker) and 2.0 instead of 2.7 ms per sweep of 1536 walkers on 16x16 squares at
// beta = 8, spin-1 honeycombs 95 and 130 ns, 1.42 and 1.96 ms.  They take LDS beside
// every walker's records; a limit of 48 KB gave no model of the repository's
// workloads rows that it does not have with this one.
constexpr size_t kWormRowBytes = 16384;
// 16-byte exits against the wide table in global memory: a step of an XXZ square in a
// field with 8 different bonds 136 ns, with 32 (wide) 171.  Beyond this they are read there.
constexpr size_t kWormExitBytes = 16384;

// Builds t; returns the reason why the model is refused, or null.
inline const char *build_worm_tables(const sse_model_desc &m, WormTables &t)
{
    const int ns = m.bond_n_sites, legs = 2 * ns;
    t.lg = ns == 1 ? 0 : ns == 2 ? 1 : 2;
    for (int i = 0; i < m.n_types; ++i)
        t.mw = std::max(t.mw, (int)m.types[i].max_worm_count);
    t.dim = m.site_dims[0];
    for (int i = 1; i < m.n_sites; ++i)
        if (m.site_dims[i] != t.dim)
            t.dim = 0;
    // r < c  <=>  (word >> 11) < ceil(c * 2^53)
    auto thr = [](double c) {
        return c <= 0.0 ? 0ull : c >= 1.0 ? (1ull << 53) : (uint64_t)std::ceil(std::ldexp(c, 53));
    };
    // bond types with equal vertices and transitions share a range of codes
    std::map<std::string, int> seen;
    std::vector<int> base(m.n_types), rep;  // code base per type; representative types
    for (int i = 0; i < m.n_types; ++i) {
        const sse_vertex_data_desc &vd = m.types[i];
        std::string key;
        auto add = [&](const void *p, size_t bytes) { key.append((const char *)p, bytes); };
        const int nt = vd.n_vertices * vd.max_worm_count * legs;
        add(&vd.n_vertices, sizeof vd.n_vertices);
        add(&vd.max_worm_count, sizeof vd.max_worm_count);
        add(vd.leg_states, (size_t)legs * vd.n_vertices);
        for (int k = 0; k < nt; ++k) {
            const int off = vd.transition_offset[k], cnt = off < 0 ? -1 : vd.transition_count[k];
            if (cnt >= 4096)
                return "transition with more than 4095 exits";
            add(&cnt, sizeof cnt);
            for (int j = 0; j < cnt; ++j) {
                add(vd.exit_cumprob + off + j, sizeof(double));
                add(vd.exit_target + off + j, sizeof(int32_t));
                add(vd.exit_leg + off + j, 1);
                add(vd.exit_worm + off + j, 1);
            }
        }
        auto it = seen.find(key);
        if (it != seen.end()) {
            base[i] = it->second;
            continue;
        }
        base[i] = (int)t.code.size();
        seen.emplace(std::move(key), base[i]);
        rep.push_back(i);
        for (int v = 0; v < vd.n_vertices; ++v) {
            const uint8_t *ls = vd.leg_states + (size_t)legs * v;
            uint32_t lower = 0;
            bool diag = true;
            for (int k = 0; k < ns; ++k) {
                lower |= (uint32_t)ls[k] << (8 * k);
                diag &= ls[k] == ls[ns + k];
            }
            t.code.push_back(make_uint2(lower, (uint32_t)diag | (uint32_t)v << 1 | (uint32_t)i << 10));
        }
        // a vertex's diagonal flag is the one its exits' targets carry (equal to
        // the comparison of its leg states in the reference's tables,
        // vertex_data.jl:171-187)
        for (int e = 0; e < vd.n_exits; ++e) {
            uint32_t &y = t.code[(size_t)base[i] + ((uint32_t)vd.exit_target[e] >> 1)].y;
            y = (y & ~1u) | ((uint32_t)vd.exit_target[e] & 1u);
        }
    }
    const size_t nc = t.code.size(), ports = 2 * (size_t)t.mw;
    const size_t nent = ((nc << t.lg) + 1) * ports;
    const size_t ww = worm_wide_words(ns);
    if (nent * ww * 4 >= ((size_t)1 << 32))  // the kernel's offsets have 32 bits
        return "too many worm table entries";
    for (int i : rep) {
        const sse_vertex_data_desc &vd = m.types[i];
        for (int e = 0; e < vd.n_exits; ++e) {
            const uint64_t k = thr(vd.exit_cumprob[e]);
            if (k < kWormTail)
                t.thr.push_back(k);
        }
    }
    std::sort(t.thr.begin(), t.thr.end());
    t.thr.erase(std::unique(t.thr.begin(), t.thr.end()), t.thr.end());
    t.nthr = (int)t.thr.size();
    // m < k  <=>  q < rank(k), for words below kWormTail
    auto rank = [&](uint64_t k) {
        return k >= kWormTail ? 0xFFFFFFFFu
                                 : (uint32_t)(std::lower_bound(t.thr.begin(), t.thr.begin() + t.nthr, k) -
                                              t.thr.begin()) + 1u;
    };
    const uint32_t always = 0xFFFFFFFFu;
    t.nent = (int)nent;
    t.wide.assign(nent * ww, 1u << 31);
    for (size_t e = 0; e < nent; ++e)
        for (int j = 0; j < 4; ++j)
            t.wide[ww * e + (j < 3 ? j : 7)] = always;
    // 16-byte entries: exits of 16 bits (selector, port, code; bit 15: none, with
    // selector and port 0, which the step follows before it sees the bit), ranks in
    // three 10-bit fields (511: always), for four sites per bond a fifth exit
    const int lcb = ns <= 2 ? 2 : 3;
    const bool small = t.nthr <= 509 && nc <= 128 && ports <= ((size_t)1 << (8 - lcb)) && nent * 16 <= kWormExitBytes;
    const uint4 none = make_uint4(0x80008000u, 0x80008000u, 511u | 511u << 10 | 511u << 20, 511u | 0x8000u << 16);
    std::vector<uint4> exits(small ? nent : 0, none);
    bool rows = ns <= 2 && ports <= 128 && (nc << t.lg) <= 255 &&
                (size_t)(t.nthr + 1) * nent * 4 <= kWormRowBytes;
    std::vector<uint32_t> row(rows ? (size_t)(t.nthr + 1) * nent : 0, 0u);
    // A site of dimension d starts worms of max(d - 1, 1) types; an exit into
    // another type than its leg's site has makes all types possible.  Rows do not
    // see that a bond type has no list for a worm.
    bool foreign = false;
    for (int i : rep)
        for (int e = 0; e < m.types[i].n_exits; ++e)
            foreign |= m.types[i].exit_worm[e] > std::max(1, m.types[i].dims[m.types[i].exit_leg[e] % ns] - 1);
    for (int i : rep)
        for (int k = 0; k < ns; ++k)
            rows = rows && (foreign ? t.mw : std::max(1, m.types[i].dims[k] - 1)) <= m.types[i].max_worm_count;
    for (int i : rep) {
        const sse_vertex_data_desc &vd = m.types[i];
        for (int v = 0; v < vd.n_vertices; ++v)
            for (int wv = 0; wv < vd.max_worm_count; ++wv)
                for (int l = 0; l < legs; ++l) {
                    const int src = (v * vd.max_worm_count + wv) * legs + l;
                    const int off = vd.transition_offset[src], cnt = off < 0 ? 0 : vd.transition_count[src];
                    const uint32_t pos = (uint32_t)(l % ns), side = (uint32_t)(l / ns);
                    const size_t ix = ((((size_t)base[i] + v) << t.lg) + pos) * ports + 2 * (size_t)wv + side;
                    const auto cum = [&](int j) { return thr(vd.exit_cumprob[off + j]); };
                    // leg selector, port behind the exit, new vertex
                    const auto leg = [&](int j) { return worm_leg(ns, pos, vd.exit_leg[off + j]); };
                    const auto port = [&](int j) {
                        return 2u * ((uint32_t)vd.exit_worm[off + j] - 1u) + (vd.exit_leg[off + j] < ns ? 1u : 0u);
                    };
                    const auto vertex = [&](int j) { return vd.exit_target[off + j] >> 1; };
                    const auto code = [&](int j) { return (uint32_t)(base[i] + vertex(j)); };
                    // the last exit stands for every word past the thresholds: it
                    // has to end the list at 1, else none (the exact search decides)
                    const auto held = [&](int nt) { return cnt == nt + 1 && cum(nt) >= kWormTail ? cnt : std::min(cnt, nt); };
                    uint32_t *x = &t.wide[ww * ix];
                    const int nt = ns == 4 ? 4 : 3;
                    for (int j = 0; j < held(nt); ++j) {
                        x[j < 4 ? 3 + j : 8] = worm_entry_word(leg(j), port(j), vertex(j) - v);
                        if (j < nt)
                            x[j < 3 ? j : 7] = cum(j) >= kWormTail ? always : (uint32_t)(cum(j) >> 21);
                        if (j > 0 && j < nt)
                            x[j < 3 ? j : 7] = std::max(x[j < 3 ? j : 7], x[j - 1]);
                    }
                    uint32_t r[3] = {511u, 511u, 511u}, o[5] = {0x8000u, 0x8000u, 0x8000u, 0x8000u, 0x8000u};
                    const auto narrow = [&](int j) { return leg(j) | port(j) << lcb | code(j) << 8; };
                    for (int j = 0; small && j < held(3); ++j) {
                        o[j] = narrow(j);
                        if (j < 3)
                            r[j] = std::min(rank(cum(j)), 511u);
                        if (j > 0 && j < 3)
                            r[j] = std::max(r[j], r[j - 1]);
                    }
                    if (small) {
                        uint32_t r3 = 511u;
                        if (ns == 4 && cnt == 5 && cum(4) >= kWormTail) {
                            r3 = std::min(rank(cum(3)), 511u);
                            o[3] = narrow(3);
                            o[4] = narrow(4);
                        }
                        exits[ix] = make_uint4(o[0] | o[1] << 16, o[2] | o[3] << 16, r[0] | r[1] << 10 | r[2] << 20,
                                               r3 | o[4] << 16);
                    }
                    // rows have no exact search behind them: the list has to
                    // end at 1, and no word of the tail (rank() takes its
                    // thresholds for 1) may belong to another exit
                    for (int j = 0; j < cnt; ++j) {
                        rows = rows && (cum(j) == (1ull << 53) || (j + 1 < cnt && cum(j) < kWormTail));
                    }
                    if (rows)
                        for (int q = 0; q <= t.nthr && rows; ++q) {
                            int j = 0;
                            while (j < cnt && (uint32_t)q >= rank(cum(j)))
                                ++j;
                            if (j >= cnt) {
                                rows = false;  // a word without an exit
                                break;
                            }
                            const uint32_t nc0 = code(j) << t.lg;
                            row[(size_t)q * nent + ix] =
                                leg(j) << 4 | port(j) << 8 | (nc0 | pos) << 16 | (nc0 | (pos ^ 1u)) << 24;
                        }
                }
    }
    if (rows)
        t.row.swap(row);
    else
        t.exit.swap(exits);
    std::vector<uint16_t> bkt;
    if (t.nthr > 8 && (!t.row.empty() || !t.exit.empty())) {  // the wide table needs no ranks
        bkt.resize(256);
        for (uint64_t b = 0; b < 256; ++b)
            bkt[b] = (uint16_t)(std::upper_bound(t.thr.begin(), t.thr.end(), b << 45) - t.thr.begin());
    }
    do
        t.thr.push_back(~0ull);
    while (t.thr.size() % 8);
    if (!bkt.empty()) {
        const size_t at = t.thr.size();
        t.thr.resize(at + 64);
        memcpy(t.thr.data() + at, bkt.data(), 512);
        t.rank = (int)(8 * t.thr.size());
    }
    // sites two per word: the wave kernels take lattices far below 65536 sites
    t.bond.resize(m.n_bonds);
    for (int b = 0; b < m.n_bonds; ++b) {
        uint32_t s[4] = {0, 0, 0, 0};
        for (int k = 0; k < ns; ++k)
            s[k] = (uint32_t)m.bond_sites[(size_t)ns * b + k];
        t.bond[b] = make_uint4((s[0] & 0xFFFFu) | s[1] << 16, (s[2] & 0xFFFFu) | s[3] << 16,
                               (uint32_t)base[m.bond_type[b]], 0u);
    }
    return nullptr;
}
