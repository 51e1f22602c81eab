// host_fast_form.cpp -- test harness: the pieces of the walk's fast form
// (pda_math.h, pda_walk.h) against the general form's, compiled for the host.
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "pda_layout.h"
#include "pda_walk.h"

using namespace pda;

static uint64_t splitmix(uint64_t& x) {
    uint64_t z = (x += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

static bool same(float a, float b) { return fbits(a) == fbits(b) || (a != a && b != b); }

// out: [0] uniforms compared, [1] logs that differ; every 24-bit uniform
// (with random low bits of the word).
extern "C" void hf_log(int64_t* out) {
    uint64_t st = 1;
    out[0] = out[1] = 0;
    for (uint32_t k = 0; k < (1u << 24); ++k) {
        const uint32_t x = (k << 8) | uint32_t(splitmix(st) & 255u);
        ++out[0];
        if (!same(flog_uniform24(x), flog(uniform24(x)))) ++out[1];
    }
}

// out: [0], [1] quotient() against the division; [2], [3] fexp_minus() against
// fexp(); [4], [5] gauss_uniform24() against gauss(); [6], [7]
// distance_efficiency_quick() against distance_efficiency().
extern "C" void hf_math(int64_t n, uint64_t seed, int64_t* out) {
    uint64_t st = seed;
    auto unit = [&]() { return double(splitmix(st) >> 11) * 0x1p-53; };
    for (int i = 0; i < 8; ++i) out[i] = 0;
    for (int64_t i = 0; i < n; ++i) {
        // divisors over the whole range, among them significands next to a
        // power of two; dividends the logs of uniforms, times, and random
        uint32_t mant = uint32_t(splitmix(st)) & 0x7FFFFFu;
        if (i % 8 == 0) mant = i % 16 ? 0x7FFFFFu - uint32_t(i / 16 % 4) : uint32_t(i / 16 % 4);
        const float b = std::ldexp(bitsf(0x3F800000u | mant), int(splitmix(st) % 80) - 40);
        float a;
        switch (i % 3) {
            case 0: a = flog_uniform24(uint32_t(splitmix(st))); break;
            case 1: a = float(unit()); break;
            default: a = std::ldexp(float(unit()), int(splitmix(st) % 40) - 20);
        }
        const float d = i % 2 ? b : -b;
        out[0]++;
        out[1] += quotient_range(b) && !same(quotient(a, d, 1.0f / d), a / d);
        const float lam = i % 5 ? float(64.0 * unit()) : std::ldexp(float(unit()), -int(i % 60));
        out[2]++;
        out[3] += !same(fexp_minus(lam), fexp(-lam));
        const uint32_t w0 = uint32_t(splitmix(st)), w1 = i % 7 ? uint32_t(splitmix(st))
                                                              : uint32_t(i / 7 % 9) * 0x1FFFFFFFu;
        out[4]++;
        out[5] += !same(gauss_uniform24(w0, w1), gauss(w0, w1));
        const float r0 = i % 4 ? 52.0f : float(1.0 + 200.0 * unit());
        float rd;
        switch (i % 6) {
            case 0: rd = float(-20.0 + 200.0 * unit()); break;
            case 1: rd = std::ldexp(float(unit()), int(splitmix(st) % 250) - 125); break;
            case 2: rd = 0.0f; break;
            case 3: rd = i % 9 ? INFINITY : NAN; break;
            default: rd = r0 * float(0.3 + 2.0 * unit());
        }
        out[6]++;
        out[7] += !same(distance_efficiency_quick(rd, r0, 1.0f / r0), distance_efficiency(rd, r0));
    }
}

// binomial_broad() against binomial() for n = 1 .. 127 and n_p efficiencies:
// out[0] draws compared, [1] different counts, [2] random uniforms it leaves
// to the general form, [3] uniforms at a threshold compared, [4] those of
// them that it decides within 2^10 grid steps of the threshold.
extern "C" void hf_binomial(int n_p, int n_u, uint64_t seed, int64_t* out) {
    uint64_t st = seed;
    for (int i = 0; i < 5; ++i) out[i] = 0;
    const UnitKey key{1u, 2u, 3u, 4u};
    for (int ip = 0; ip < n_p; ++ip) {
        float p;
        switch (ip) {
            case 0: p = 0.0f; break;
            case 1: p = 1.0f; break;
            case 2: p = 0.5f; break;
            case 3: p = 0x1p-140f; break;
            case 4: p = 1.0f - 0x1p-24f; break;
            case 5: p = NAN; break;
            case 6: p = 0.50000006f; break;
            default: p = float(double(splitmix(st) >> 11) * 0x1p-53);
        }
        for (int n = 1; n < kBinomTable; ++n) {
            auto draw = [&](int64_t u, int64_t* a, int64_t* b) {
                const uint32_t hi = uint32_t(u >> 26) << 5;
                const uint32_t lo = uint32_t(u & ((int64_t(1) << 26) - 1)) << 6;
                *a = binomial(n, double(p), hi, lo, key, 7u);
                *b = binomial_broad(n, p, hi, lo);
            };
            int64_t a, b;
            for (int i = 0; i < n_u; ++i) {
                draw(int64_t(splitmix(st) >> 11), &a, &b);
                ++out[0];
                if (b < 0) ++out[2];
                else if (a != b) ++out[1];
            }
            // around the cumulative sums of the exact pmf and at the ends
            const double pp = p > 0.5f ? 1.0 - double(p) : double(p);
            long double px = powl(1.0L - (long double)pp, n), C = 0.0L;
            for (int k = 0; k <= n && p >= 0.0f && p <= 1.0f; ++k) {
                C += px;
                px = px * (long double)(n - k) * (long double)pp /
                     ((long double)(k + 1) * (1.0L - (long double)pp));
                const int64_t t = int64_t(C * 0x1p53L);
                for (int64_t e : {-(int64_t(1) << 20), int64_t(-1025), int64_t(-1), int64_t(0),
                                  int64_t(1), int64_t(1025), int64_t(1) << 20}) {
                    const int64_t u = t + e;
                    if (u < 0 || u >= (int64_t(1) << 53)) continue;
                    draw(u, &a, &b);
                    ++out[3];
                    if (b >= 0 && a != b) ++out[1];
                    if (b >= 0 && e > -1024 && e < 1024) ++out[4];
                }
            }
        }
    }
}

// Units of random bursts in the fast form for models with broadening against
// the general form: out[0] units, [1] abandoned, [2] different, [3] windows'
// acceptors in all.
extern "C" int hf_walk(const int64_t* start, const int64_t* stop, const int64_t* istart,
                       const int32_t* phcount, int64_t nb, const int64_t* times,
                       const uint8_t* mask_ad, const uint8_t* mask_dd, int64_t np, const float* T,
                       float clk_p, float bg_ad, float bg_dd, int n, const float* args, float r0,
                       int R, uint32_t seed, int64_t* out) {
    std::vector<BurstDesc> bursts;
    std::vector<uint32_t> ticks;
    std::vector<uint2> links;
    std::string err;
    PhotonSrc src{times, mask_ad, mask_dd, nullptr, nullptr};
    int rc = encode_bursts(start, stop, istart, phcount, nb, src, np, T, clk_p, bg_ad, bg_dd,
                           bursts, ticks, links, err);
    if (rc) return rc;
    Photophysics ph;
    ph.gamma = 1.0f;
    ph.dexdir = 0.0f;
    ph.crosstalk = 0.05f;
    ph.r0 = r0;
    Model M;
    rc = build_model(ph, n, args, n * (n + 1), M, err);
    if (rc) return rc;
    RunArgs a{};
    a.bg_on = bg_dd < 1e-4f ? 0 : 1;
    a.clk_p = clk_p;
    a.bg_ad = bg_ad;
    a.bg_dd = bg_dd;
    for (int i = 0; i < 4; ++i) out[i] = 0;
    const BroadDraw draw{};
    for (int64_t b = 0; b < nb; ++b) {
        const BurstDesc& d = bursts[size_t(b)];
        for (int r = 0; r < R; ++r) {
            const UnitKey key{seed, 5u, uint32_t(r), uint32_t(b)};
            const uint32_t* tk = ticks.data() + d.off;
            const uint2* lk = links.data() + d.off;
            const WalkOut f = walk_unit<true, BroadDraw>(M, &draw, key, d.P, d.stop_rel, d.T, tk, lk, a);
            const WalkOut g = walk_unit<false>(M, nullptr, key, d.P, d.stop_rel, d.T, tk, lk, a);
            ++out[0];
            out[1] += f.replay;
            out[2] += !f.replay && !(same(f.acc, g.acc) && same(f.F, g.F));
            out[3] += int64_t(g.acc);
        }
    }
    return 0;
}
