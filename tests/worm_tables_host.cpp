// Host build of csrc/worm_tables.h for tests/test_worm_tables_cpu.py: builds a
// model's worm tables and hands the images out.
#include "../stochasticseriesexpansion.jl_amd/csrc/worm_tables.h"

extern "C" {

void *wt_build(const sse_model_desc *m, const char **why)
{
    WormTables *t = new WormTables;
    *why = build_worm_tables(*m, *t);
    return t;
}
void wt_free(void *h) { delete (WormTables *)h; }

// thresholds, code stride (log2), worm types, entries
void wt_info(void *h, int64_t *out)
{
    const WormTables &t = *(WormTables *)h;
    out[0] = t.nthr;
    out[1] = t.lg;
    out[2] = t.mw;
    out[3] = t.nent;
}

// bytes of a slab (csrc/sse_common.h) of cap slots, codes chase codes and sites
// sites of the batch's largest lattice
int64_t wt_slab_bytes(int64_t cap, int ns, int codes, int sites)
{
    DevModel m;
    memset(&m, 0, sizeof m);
    m.nsb = ns;
    m.w_ncode = codes;
    return (int64_t)slab_bytes(cap, m, sites, true);
}

// image 0 thresholds, 1 rows, 2 16-byte exits, 3 wide entries, 4 codes, 5 bonds
const void *wt_image(void *h, int which, int64_t *bytes)
{
    const WormTables &t = *(WormTables *)h;
    auto give = [&](const auto &v) {
        *bytes = (int64_t)(v.size() * sizeof v[0]);
        return (const void *)v.data();
    };
    switch (which) {
    case 0: return give(t.thr);
    case 1: return give(t.row);
    case 2: return give(t.exit);
    case 3: return give(t.wide);
    case 4: return give(t.code);
    default: return give(t.bond);
    }
}
}
