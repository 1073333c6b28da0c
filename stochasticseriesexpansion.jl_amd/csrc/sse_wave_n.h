// sse_wave_n.h -- the wave kernels (one wavefront per walker) for bonds of
// any site count NS = 1..4 (SSEData{NSites}, sse_data.jl:15-42; vertices of
// 2*NS legs, vertex_list.jl:24-62).
//
// These kernels take the site count as a template parameter and keep the
// structure of the two-site ones of sse_wave.h where it carries over:
//   K1n  diagonal update + vertex list, 64 slots per step (as K1: the same
//        draws, acceptance windows and slot-by-slot fallback), with one
//        per-site lane mask per bond position;
//   (the worm update, sse_worm.h, takes any site count itself);
//   K3n  measurement (sign and the magnetization estimators), 64 slots per step.
// Included by sse_wave.h after the two-site kernels it builds on (K1's
// stream and acceptance code, the worm controller, the measurement sums) and
// before the launch helpers that dispatch to it.
#pragma once

// LDS of K1n (one walker): Philox words u64[256], lane masks u64[NS][N],
// operators on the site so far u32[N], spins u8[N]
__host__ __device__ inline size_t k1n_lds_bytes(int N, int NS)
{
    size_t b = 2048 + 8 * (size_t)NS * N + 4 * (size_t)N + (size_t)N;
    return (b + 15) & ~(size_t)15;
}

// upper (after the operator) states of vertex v, one byte per bond position
template <int NS>
__device__ __forceinline__ uint32_t k1n_upper(const DevVD &vd, uint32_t v)
{
    const uint8_t *ls = vd.leg_states + 2 * NS * v + NS;
    uint32_t u = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k)
        u |= (uint32_t)ls[k] << (8 * k);
    return u;
}

// Slot-by-slot processing of one chunk in reference order (Lemire rejection
// in a bond draw, or forced); emits the same idx words as the parallel path.
template <int NS>
__device__ void k1n_serial_chunk(DevWalker &w, const DevModel &m, WaveStream &rs, int64_t base,
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
                const int32_t *bs = m.bond_sites + (size_t)NS * b;
                const DevVD &vd = m.types[m.bond_type[b]];
                int idx = 0, stride = 1;
                for (int k = 0; k < NS; ++k) {
                    idx += (sp[bs[k]] - 1) * stride;
                    stride *= vd.dims[k];
                }
                int32_t dv = vd.diag_vertex[idx];
                double wgt = dv < 0 ? 0.0 : vd.weights[dv >> 1];
                double p_make = pm_raw / (double)(L - n);
                if (rs.next_float() < p_make * wgt) {
                    nop = op_make(b, (uint32_t)dv);
                    n += 1;
                }
            } else {
                uint32_t vc = op_vcode(op);
                uint32_t b = op_bond(op);
                const DevVD &vd = m.types[m.bond_type[b]];
                if (vc & 1u) {
                    double wgt = vd.weights[vc >> 1];
                    double p_remove = (double)(L - n + 1) * pr_raw;
                    if (rs.next_float() * wgt < p_remove) {
                        nop = 0u;
                        n -= 1;
                    }
                } else {
                    const uint32_t up = k1n_upper<NS>(vd, vc >> 1);
                    __syncthreads();
                    if (lane == 0)
                        for (int k = 0; k < NS; ++k)
                            sp[m.bond_sites[(size_t)NS * b + k]] = (uint8_t)(up >> (8 * k));
                    __syncthreads();
                }
            }
        }
        if (do_vl && nop != 0u) {
            const uint32_t b = op_bond(nop);
            __syncthreads();
            if (lane == 0)
                for (int k = 0; k < NS; ++k) {
                    const int s = m.bond_sites[(size_t)NS * b + k];
                    gidx[(size_t)NS * p + k] = cnt[s];
                    cnt[s] += 1u;
                }
            __syncthreads();
        }
        if (lane == 0 && nop != op)
            w.ops[p] = nop;
    }
    __syncthreads();
}

// Model lookups of K1n: from the LDS copy of DevModel::k1ntab (N1Staged) or
// from the model's global arrays (N1Global).  Same values either way.
template <int NS>
struct N1Global {
    const DevModel *m;
    __device__ __forceinline__ void stage(char *) const {}
    __device__ __forceinline__ int type(uint32_t b) const { return m->bond_type[b]; }
    __device__ __forceinline__ int site(uint32_t b, int k) const { return m->bond_sites[(size_t)NS * b + k]; }
    __device__ __forceinline__ int nv(int t) const { return m->types[t].nv; }
    __device__ __forceinline__ int dim(int t, int j) const { return m->types[t].dims[j]; }
    __device__ __forceinline__ int diag(int t, int i) const { return m->types[t].diag_vertex[i]; }
    __device__ __forceinline__ double weight(int t, int v) const { return m->types[t].weights[v]; }
    __device__ __forceinline__ uint32_t upper(int t, int v) const { return k1n_upper<NS>(m->types[t], (uint32_t)v); }
};
template <int NS>
struct N1Staged {
    const DevModel *m;
    const char *t;  // the LDS copy of m->k1ntab
    // copy the table into LDS (whole wave; the caller's barrier follows)
    __device__ __forceinline__ void stage(char *dst) const
    {
        const uint32_t *g = (const uint32_t *)m->k1ntab;
        uint32_t *d = (uint32_t *)dst;
        for (int i = threadIdx.x; i < m->k1ntab_bytes / 4; i += 64)
            d[i] = g[i];
    }
    __device__ __forceinline__ const uint32_t *hdr(int ty) const { return (const uint32_t *)(t + 32 * ty); }
    __device__ __forceinline__ const int32_t *bond(uint32_t b) const
    {
        return (const int32_t *)(t + m->k1n_bond_off) + (size_t)(NS + 1) * b;
    }
    __device__ __forceinline__ int type(uint32_t b) const { return bond(b)[0]; }
    __device__ __forceinline__ int site(uint32_t b, int k) const { return bond(b)[1 + k]; }
    __device__ __forceinline__ int nv(int ty) const { return (int)hdr(ty)[3]; }
    __device__ __forceinline__ int dim(int ty, int j) const { return (int)((hdr(ty)[4] >> (8 * j)) & 255u); }
    __device__ __forceinline__ int diag(int ty, int i) const { return ((const int32_t *)(t + hdr(ty)[1]))[i]; }
    __device__ __forceinline__ double weight(int ty, int v) const
    {
        return ((const double *)(t + hdr(ty)[0]))[v];
    }
    __device__ __forceinline__ uint32_t upper(int ty, int v) const
    {
        return ((const uint32_t *)(t + hdr(ty)[2]))[v];
    }
};

// LDS bytes of K1n with the model's lookups staged
__host__ __device__ inline size_t k1n_lds_staged(int N, int NS, int k1ntab_bytes)
{
    return k1n_lds_bytes(N, NS) + (((size_t)k1ntab_bytes + 15) & ~(size_t)15);
}

// K1n of walker wi: diagonal update (sse.jl:137-191) and vertex list
// (vertex_list.jl:15-54), 64 slots per step.  phases: 1 diagonal update,
// 2 vertex list, 8 force the slot-by-slot path; warm >= 0: init warm-up
// round r (diagonal only, pending walkers with more warm-up sweeps).
template <int NS, class Tab>
__device__ void k1n_walker(DevWalker *W, const DevModel *models, DevPool *pool, int wi, int phases,
                           int warm, char *lds, int grp, Tab tab)
{
    const int lane = threadIdx.x;
    DevWalker w = W[wi];
    if (w.error)
        return;
    if (warm >= 0 ? (warm >= w.warmup || !w.pending) : (!w.active || w.retire))
        return;
    const DevModel &m = models[w.model];
    const int N = m.n_sites;
    uint64_t *rbuf = (uint64_t *)lds;
    uint64_t *tm = (uint64_t *)(lds + 2048);  // tm[k * N + site]
    uint32_t *cnt = (uint32_t *)(tm + (size_t)NS * N);
    uint8_t *sp = (uint8_t *)(cnt + N);
    uint32_t *tmw = (uint32_t *)tm;

    const bool do_diag = phases & 1;
    const bool do_vl = (phases & 2) && warm < 0;
    const bool force_serial = phases & 8;

    tab.stage(lds + k1n_lds_bytes(N, NS));
    for (int i = lane; i < NS * N; i += 64)
        tm[i] = 0ull;
    for (int i = lane; i < N; i += 64) {
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
    const int64_t L = w.L;
    const uint32_t Lu = (uint32_t)L;
    int64_t n0 = w.n;
    const uint64_t below = below_mask(lane), above = above_mask(lane);
    gmem<uint32_t> *gidx = as_global((uint32_t *)w.links);
    gmem<uint32_t> *ops = as_global(w.ops);

    // As in k1_walker_t: the operators come in blocks of K1_BLOCK chunks, a block
    // ahead (an operator loaded in one chunk for the next would be waited on with
    // the chunk's stores), the model's scalars are read before the loop, and the
    // lanes run one path.  Measured on 64 walkers: ring of three-site bonds (8711
    // slots) 343 -> 246 us per sweep, of four-site bonds (1439 slots) 78 -> 59 us.
    const uint32_t nbonds = uni((uint32_t)m.n_bonds);
    uint32_t cur[K1_BLOCK], pf[K1_BLOCK];
#pragma unroll
    for (int u = 0; u < K1_BLOCK; ++u) {
        const uint32_t q = 64u * u + lane;
        cur[u] = q < Lu ? ops[q] : 0u;
    }
#pragma unroll
    for (int u = 0; u < K1_BLOCK; ++u) {
        const uint32_t q = 64u * (K1_BLOCK + u) + lane;
        pf[u] = q < Lu ? ops[q] : 0u;
    }
    bool bad = false;
    for (uint32_t base = 0; base < Lu; base += 64) {
        const uint32_t p = base + lane;
        const bool valid = p < Lu;
        const uint32_t chunk = base >> 6;
        const int slot = (int)uni(chunk % K1_BLOCK);
        if (slot == 0 && chunk > 0) {
#pragma unroll
            for (int u = 0; u < K1_BLOCK; ++u)
                cur[u] = pf[u];
#pragma unroll
            for (int u = 0; u < K1_BLOCK; ++u) {
                const uint32_t q = base + 64u * (K1_BLOCK + u) + lane;
                pf[u] = q < Lu ? ops[q] : 0u;
            }
        }
        const uint32_t op = cur[slot];
        const uint32_t vc = op_vcode(op);
        const bool ident = valid && op == 0u;
        const bool isop = op != 0u;
        const bool dia = isop && (vc & 1u);
        const bool offd = isop && !(vc & 1u);
        const uint64_t identm = __ballot(ident), diam = __ballot(dia), offm = __ballot(offd);
        uint32_t b = op_bond(op);
        // an operator outside the model (a corrupted string): reported when the
        // walker ends, its bond and vertex replaced by ones that exist
        bad |= b >= nbonds;
        b = b < nbonds ? b : 0u;
        double u = 0.0;
        if (do_diag) {
            const uint32_t D = 2u * (uint32_t)popc(identm) + (uint32_t)popc(diam);
            const uint32_t off = 2u * bits_below(identm) + bits_below(diam);
            rs.ensure(D + 2u);  // as in k1_walker_t
            const uint64_t x0 = rs.peek(off), x1 = rs.peek(off + 1u);
            // rand(1:n_bonds): high half of word * n_bonds, rejected where the low
            // half could be below 2^64 mod n_bonds
            const uint64_t pl = (uint64_t)(uint32_t)x0 * nbonds;
            const uint64_t ph = (uint64_t)(uint32_t)(x0 >> 32) * nbonds + (pl >> 32);
            const bool maybe = ident && (uint32_t)ph == 0u && (uint32_t)pl < nbonds;
            if (__builtin_expect(force_serial || wave_any(maybe), 0)) {
                bad |= isop && (int)(vc >> 1) >= tab.nv(tab.type(b));
                if (wave_any(bad))  // its lookups take indexes as they are
                    break;
                k1n_serial_chunk<NS>(w, m, rs, base, n0, pm_raw, pr_raw, do_diag, do_vl, sp, cnt);
                continue;
            }
            b = ident ? (uint32_t)(ph >> 32) : b;
            u = word_to_float(ident ? x1 : x0);
            rs.advance(D);
        } else if (force_serial) {
            bad |= isop && (int)(vc >> 1) >= tab.nv(tab.type(b));
            if (wave_any(bad))
                break;
            k1n_serial_chunk<NS>(w, m, rs, base, n0, pm_raw, pr_raw, do_diag, do_vl, sp, cnt);
            continue;
        }

        const bool has = isop || (ident && do_diag);
        const int type = tab.type(b);
        int st[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k)
            st[k] = tab.site(b, k);
        // per-site lane masks, one per bond position
        if (has) {
#pragma unroll
            for (int k = 0; k < NS; ++k)
                atomicOr(&tmw[2 * ((size_t)k * N + st[k]) + (lane >> 5)], 1u << (lane & 31));
        }
        int vx = (int)(vc >> 1);
        const bool vbad = vx >= tab.nv(type);
        bad |= isop && vbad;
        vx = vbad ? 0 : vx;
        const uint32_t up = tab.upper(type, vx);  // an off-diagonal operator's states after it
        double wgt = tab.weight(type, vx);        // a diagonal operator's weight
        uint32_t s0[NS], c0[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            s0[j] = sp[st[j]];
            c0[j] = cnt[st[j]];
        }
        wave_lds_sync();
        // M[j][k]: lanes whose bond has the site of this lane's position j at
        // position k; A[j]: lanes whose bond touches that site at all
        uint64_t M[NS][NS], A[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            A[j] = 0ull;
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                M[j][k] = tm[(size_t)k * N + st[j]];
                A[j] |= M[j][k];
            }
        }

        uint64_t plus = 0, minus = 0;
        uint32_t fop = op;
        if (do_diag) {
            // states at the slot: of the latest off-diagonal operator on the site
            // earlier in the chunk, else at the chunk's start
            int idx = 0, stride = 1;
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                const uint64_t cand = A[j] & offm & below;
                const uint32_t q = cand ? (uint32_t)hi_bit(cand) : 0u;
                const uint32_t uq = from_lane(up, q);
                uint32_t pos = 0;  // of the site in that operator's bond
#pragma unroll
                for (int k = 1; k < NS; ++k)
                    pos = ((M[j][k] >> q) & 1ull) ? 8u * k : pos;
                const int v = (int)(cand ? (uq >> pos) & 255u : s0[j]);
                idx += (v - 1) * stride;
                stride *= tab.dim(type, j);
            }
            const int32_t dv = ident ? tab.diag(type, idx) : -1;
            const double wd = tab.weight(type, dv < 0 ? 0 : dv >> 1);
            wgt = ident ? (dv < 0 ? 0.0 : wd) : wgt;
            // as in k1_walker_t
            const uint32_t room = Lu - (uint32_t)n0 + (ident ? 0u : 1u);
            const uint32_t dl = room + (uint32_t)lane < Lu ? room + (uint32_t)lane : Lu;
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
                const int64_t na = n0 + popc(plus & ba) - popc(minus & ba);
                bool d = false;
                if (lane == a) {
                    if (ident)
                        d = u < (pm_raw / (double)(L - na)) * wgt;
                    else
                        d = u * wgt < (double)(L - na + 1) * pr_raw;
                }
                const uint64_t dm = __ballot(d);
                if ((identm >> a) & 1ull)
                    plus |= dm;
                else
                    minus |= dm;
                ambm &= ambm - 1;
            }
            n0 += popc(plus) - popc(minus);
            if (ident && ((plus >> lane) & 1ull))
                fop = op_make(b, (uint32_t)dv);
            if (dia && ((minus >> lane) & 1ull))
                fop = 0u;
            if (fop != op)
                ops[p] = fop;
        }

        // vertex list over the chunk's final non-identity operators: how many
        // earlier operators act on each of the operator's sites
        const uint64_t NI = do_diag ? ((identm & plus) | (diam & ~minus) | offm) : (diam | offm);
        if (do_vl && ((NI >> lane) & 1ull)) {
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                gidx[(size_t)NS * p + j] = c0[j] + bits_below(A[j] & NI);
                atomicAdd(cnt + st[j], 1u);
            }
        }
        // spins after the chunk: the last off-diagonal operator on a site wins
        if (do_diag && offd) {
#pragma unroll
            for (int j = 0; j < NS; ++j)
                if (((A[j] & offm) & above) == 0ull)
                    sp[st[j]] = (uint8_t)(up >> (8 * j));
        }
        if (has) {
#pragma unroll
            for (int k = 0; k < NS; ++k)
                tm[(size_t)k * N + st[k]] = 0ull;
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

// Measurement (sse.jl:70-87, 305-376) of walker wi, 64 slots per step.  With
// the model's per-(bond, vertex) tables it is k3_walker's (their values do not
// depend on the bond size); otherwise the sign and operator count in one pass
// over the operator string, then one pass per magnetization estimator.  mode
// as in k3_walker.
template <int NS>
__device__ __forceinline__ void k3n_walker(DevWalker *W, const DevModel *models, double *out, double *sum,
                           double *sumsq, int64_t *count, double *wlf, int wi, int mode,
                           int32_t *done)
{
    constexpr int LEGS = 2 * NS;
    const int lane = threadIdx.x;
    if (models[W[wi].model].est_dtab) {
        k3_walker(W, models, out, sum, sumsq, count, wlf, wi, mode, done);
        return;
    }
    const DevWalker w = W[wi];
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
    const int N = m.n_sites, D = m.est_max_dim;
    const int64_t L = w.L;
    const gmem<uint32_t> *ops = as_global((const uint32_t *)w.ops);
    int neg = 0;
    int64_t cnt = 0;
    double sign = 1.0;
    // the sign and the operator count
    for (int64_t base = 0; base < L; base += 64) {
        const int64_t p = base + lane;
        const uint32_t op = p < L ? ops[p] : 0u;
        bool ng = false;
        if (op != 0u) {
            const DevVD &vd = m.types[m.bond_type[op_bond(op)]];
            ng = vd.signs[op_vcode(op) >> 1] < 0;
        }
        neg += popc(__ballot(ng));
        cnt += popc(__ballot(op != 0u));
    }
    sign = (neg & 1) ? -1.0 : 1.0;
    for (int e = 0; e < m.n_est; ++e) {
        const gmem<double> *cf = as_global(m.est_coef + (size_t)e * N);
        const gmem<double> *mk = as_global(m.est_mval + (size_t)e * N * D);
        double t0 = 0.0;
        for (int i = lane; i < N; i += 64)
            t0 += cf[i] * mk[(size_t)i * D + w.spins[i] - 1];
        const double tmp0 = wave_sum(t0);
        double run = tmp0, mag = 0.0, absmag = 0.0, mag2 = 0.0, mag4 = 0.0;
        for (int64_t base = 0; base < L; base += 64) {
            const int64_t p = base + lane;
            const uint32_t op = p < L ? ops[p] : 0u;
            double delta = 0.0;
            if (op != 0u && !(op_vcode(op) & 1u)) {
                const uint32_t b = op_bond(op);
                const DevVD &vd = m.types[m.bond_type[b]];
                const uint8_t *ls = vd.leg_states + (size_t)LEGS * (op_vcode(op) >> 1);
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    const int s = m.bond_sites[(size_t)NS * b + k];
                    delta += cf[s] * (mk[(size_t)s * D + ls[NS + k] - 1] - mk[(size_t)s * D + ls[k] - 1]);
                }
            }
            const double inc = wave_incl_scan(delta);
            if (op != 0u) {
                const double t = run + inc;
                const double t2 = t * t;
                mag += t;
                absmag += fabs(t);
                mag2 += t2;
                mag4 += t2 * t2;
            }
            run += __shfl(inc, 63);
        }
        // as k3_finish: the estimator's five values (magnetization_estimator.jl:125-165,205-230)
        const double Nn = m.norm;
        const double en = 1.0 + (double)cnt;
        const double norm = 1.0 / Nn;
        double smag = tmp0 + wave_sum(mag);
        double sabs = fabs(tmp0) + wave_sum(absmag);
        double s2 = tmp0 * tmp0;
        double smag2 = s2 + wave_sum(mag2);
        double smag4 = s2 * s2 + wave_sum(mag4);
        smag *= norm;
        sabs *= norm;
        smag2 *= norm * norm;
        smag4 *= (norm * norm) * (norm * norm);
        if (lane == 0) {
            double *oe = o + 5 + 5 * e;
            oe[0] = sign * smag / en;
            oe[1] = sign * sabs / en;
            oe[2] = sign * smag2 / en;
            oe[3] = sign * smag4 / en;
            const double chi = 1.0 / w.T / (en + 1.0) / en * (smag * smag + smag2) * Nn;
            oe[4] = sign * chi;
        }
    }
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

// ------------------------------------------------------------------ kernels
// The site count of a walker's model selects the instantiation (all bonds of
// a model have the same count).
#define SSE_NS_DISPATCH(ns, CALL) \
    switch (ns) {                 \
    case 1: CALL(1); break;       \
    case 2: CALL(2); break;       \
    case 3: CALL(3); break;       \
    default: CALL(4); break;      \
    }

// budget non-null: sweep `step` of a budgeted call; walker wi takes part
// only while step < budget[wi]
// K1n of walker wi with the model's lookups in LDS when the launch's LDS
// (lds_bytes) holds them
template <int NS>
__device__ __forceinline__ void k1n_walker_sel(DevWalker *W, const DevModel *models, DevPool *pool, int wi,
                                               int phases, int warm, char *lds, int grp, int lds_bytes)
{
    const DevModel *m = &models[W[wi].model];
    if (k1n_lds_staged(m->n_sites, NS, m->k1ntab_bytes) <= (size_t)lds_bytes)
        k1n_walker<NS>(W, models, pool, wi, phases, warm, lds, grp,
                       N1Staged<NS>{m, lds + k1n_lds_bytes(m->n_sites, NS)});
    else
        k1n_walker<NS>(W, models, pool, wi, phases, warm, lds, grp, N1Global<NS>{m});
}

__global__ __launch_bounds__(64) void waven_diag_vlist_kernel(DevWalker *W, const DevModel *models,
                                                              DevPool *pool, int w_begin, int w_end,
                                                              int phases, int warm,
                                                              const int32_t *order, int grp,
                                                              const int32_t *budget, int step,
                                                              int lds_bytes)
{
    extern __shared__ __align__(16) char lds[];
    const int pos = w_begin + (int)blockIdx.x;
    if (pos >= w_end)
        return;
    const int wi = walker_at(order, pos);
    if (budget && step >= budget[wi])
        return;
    const int ns = models[W[wi].model].nsb;
#define K1N_CALL(K) k1n_walker_sel<K>(W, models, pool, wi, phases, warm, lds, grp, lds_bytes)
    SSE_NS_DISPATCH(ns, K1N_CALL)
#undef K1N_CALL
}

__global__ __launch_bounds__(64) void waven_worm_kernel(DevWalker *W, const DevModel *models,
                                                        DevPool *pool, int w_begin, int w_end,
                                                        int full_sweep, const int32_t *order,
                                                        const int32_t *budget, int step,
                                                        int lds_bytes, int rec_mode)
{
    extern __shared__ __align__(16) char lds[];
    const int pos = w_begin + (int)blockIdx.x;
    if (pos >= w_end)
        return;
    const int wi = walker_at(order, pos);
    if (budget && step >= budget[wi])
        return;
    const int ns = models[W[wi].model].nsb;
#define K2N_CALL(K) worm_walker<K>(W, models, pool, wi, full_sweep, lds_bytes, rec_mode, lds)
    SSE_NS_DISPATCH(ns, K2N_CALL)
#undef K2N_CALL
}

__global__ __launch_bounds__(64) void waven_measure_kernel(DevWalker *W, const DevModel *models,
                                                           double *out, double *sum, double *sumsq,
                                                           int64_t *count, double *wlf, int w_begin,
                                                           int w_end, int mode, int32_t *done,
                                                           const int32_t *order,
                                                           const int32_t *budget, int step)
{
    const int pos = w_begin + (int)blockIdx.x;
    if (pos >= w_end)
        return;
    const int wi = walker_at(order, pos);
    if (budget && step >= budget[wi])
        return;
    const int ns = models[W[wi].model].nsb;
#define K3N_CALL(K) k3n_walker<K>(W, models, out, sum, sumsq, count, wlf, wi, mode, done)
    SSE_NS_DISPATCH(ns, K3N_CALL)
#undef K3N_CALL
}
