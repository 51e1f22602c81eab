// host_long_runs.cpp -- test harness: what draws_in_place (pda_layout.cpp) goes
// by, and the units of random bursts with their draws made in place (BroadAll)
// against the general form, compiled for the host.
#include <cstdint>
#include <string>
#include <vector>

#include "pda_layout.h"
#include "pda_walk.h"

using namespace pda;

static bool same(float a, float b) { return fbits(a) == fbits(b) || (a != a && b != b); }

struct Data {
    std::vector<BurstDesc> bursts;
    std::vector<uint32_t> ticks;
    std::vector<uint2> links;
};

// out: [0], [1] donor and acceptor photons looked at with at least k of their
// run to come, [2] long bursts, [3], [4] draws_in_place of a single set and of a
// population over `range` bursts; units in place (R > 0): [5] units, [6]
// abandoned, [7] different, [8] acceptors.
extern "C" int hl_run(const int64_t* start, const int64_t* stop, const int64_t* istart,
                      const int32_t* phcount, int64_t nb, const int64_t* times,
                      const uint8_t* mask_ad, const uint8_t* mask_dd, int64_t np, const float* T,
                      float clk_p, float bg_ad, float bg_dd, float gamma, float crosstalk,
                      float dexdir, uint32_t k, int64_t range, int n, const float* args, int R,
                      uint32_t seed, int64_t* out) {
    Data d;
    LongRuns r;
    std::string err;
    PhotonSrc src{times, mask_ad, mask_dd, nullptr, nullptr};
    int rc = encode_bursts(start, stop, istart, phcount, nb, src, np, T, clk_p, bg_ad, bg_dd,
                           d.bursts, d.ticks, d.links, err, &r);
    if (rc) return rc;
    Photophysics ph;
    ph.gamma = gamma;
    ph.crosstalk = crosstalk;
    ph.dexdir = dexdir;
    const bool bg_on = !(bg_dd < 1e-4f);
    for (int c = 0; c < 2; ++c)
        out[c] = k < r.at_least[c].size() ? int64_t(r.at_least[c][k]) : 0;
    out[2] = r.long_bursts;
    const int64_t photons = int64_t(d.ticks.size());
    for (int p = 0; p < 2; ++p)
        out[3 + p] = draws_in_place(r, nb, photons, range, ph, bg_on, p != 0);
    Model M;
    rc = build_model(ph, n, args, n * (n + 1), M, err);
    if (rc) return rc;
    RunArgs a{};
    a.bg_on = bg_on ? 1 : 0;
    a.clk_p = clk_p;
    a.bg_ad = bg_ad;
    a.bg_dd = bg_dd;
    for (int i = 5; i < 9; ++i) out[i] = 0;
    const BroadAll draw{};
    for (int64_t b = 0; b < nb; ++b) {
        const BurstDesc& u = d.bursts[size_t(b)];
        for (int i = 0; i < R; ++i) {
            const UnitKey key{seed, 5u, uint32_t(i), uint32_t(b)};
            const uint32_t* tk = d.ticks.data() + u.off;
            const uint2* lk = d.links.data() + u.off;
            const WalkOut f = walk_unit<true, BroadAll>(M, &draw, key, u.P, u.stop_rel, u.T, tk, lk, a);
            const WalkOut g = walk_unit<false>(M, nullptr, key, u.P, u.stop_rel, u.T, tk, lk, a);
            ++out[5];
            out[6] += f.replay;
            out[7] += !f.replay && !(same(f.acc, g.acc) && same(f.F, g.F));
            out[8] += int64_t(g.acc);
        }
    }
    return 0;
}
