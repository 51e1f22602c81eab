// pda_walk.h -- one (burst, resample) unit of the Monte-Carlo PDA walk:
// the body of gSMFRETda's mc_kernel (src/mc.cu:92-196) over the resident
// photon layout of pda_types.h.  Host-and-device code: the gfx950 walk
// kernels run it per lane; a host build of the same source checks the
// algorithm against the oracle without a GPU.
//
// Two forms of the same computation:
//   * general: every branch of the reference (distance broadening, BTPE,
//     inversion restarts, Poisson chunking for large background means);
//   * fast: the common case -- counts below 128, inversion without restarts,
//     background means <= 64.  The acceptor draw is by thresholds or tables of
//     the states' efficiencies (v == 0), or of an efficiency drawn per window
//     (broadening), where larger counts and means may be drawn in place
//     (BroadAll).  A unit that would leave the common case is abandoned
//     (replay = true) and recomputed from scratch by the general form; the
//     keyed random streams make the replay produce exactly the draws the fast
//     form would have consumed.
#pragma once
#include <type_traits>

#include "pda_math.h"
#include "pda_types.h"

namespace pda {

constexpr uint32_t kMaxWindows = 1u << 22;

// drawDisIdx (src/gen_rand.cuh:35-50) on precomputed running sums: the first
// i with cum[i] > u, else n - 1.  n is the same for every lane (the model's),
// so the loop runs n passes with no early exit; unrolled to kMaxStates it
// would keep one compare mask per bound live in scalar registers.
PDA_HD int first_above(const float* cum, int n, float u) {
    int idx = n - 1;
    bool found = false;
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
        const bool hit = !found && cum[i] > u;
        idx = hit ? i : idx;
        found = found || hit;
    }
    return idx;
}

struct WalkOut {
    float acc;    // sum of acceptor draws (float accumulation, as mcE[t] += ai)
    float F;      // sum of corrected photon counts
    bool replay;  // fast form only: the unit needs the general form
};

// Binomial(n, ep0[s]) by inversion from the per-state tables; -1 when the
// general sampler is needed (BTPE regime, n beyond the table, a restart).
// Same operations as binomial()/binomial_inversion() in pda_math.h.
PDA_HD int64_t binomial_table(int n, int s, const Model& M, const BinomTable& tab, uint32_t hi,
                              uint32_t lo) {
    if (n <= 0) return 0;
    const double pp = M.pp[s];
    if (n >= kBinomTable || !(n < kInversionMaxN || pp * double(n) <= 30.0)) return -1;
    const double q = M.qq[s];
    double px = tab.qn[s][n];
    const int bound = tab.bound[s][n];
    double U = uniform53(hi, lo);
    int X = 0;  // < kBinomTable: 32-bit counters convert to double exactly
    while (U > px) {
        ++X;
        if (X > bound) return -1;
        U -= px;
        px = (double(n - X + 1) * pp * px) / (double(X) * q);
    }
    return M.flip[s] ? int64_t(n - X) : int64_t(X);
}

static_assert(kInversionMaxN >= kBinomTable, "every tabulated count draws by inversion");

constexpr int64_t kU53Max = (int64_t(1) << 53) - 1;  // largest 53-bit grid index

// Rows of the guided inversion: binomial_table's X as a function of the
// uniform's grid index u (U = u 2^-53 exactly, uniform53).
//
// The loop keeps U_0 = U, U_{i+1} = fl(U_i - px_i) and goes past i while
// U_i > px_i, where px_i does not depend on U.  Rounding is monotone, so
// every U_i is a non-decreasing function of U, and so is X(U): X >= k + 1
// exactly for U at or above some grid point.  Locating it: every subtraction
// rounds a value in (0, 1), so U_i is within i 2^-54 of U - S_{i-1}, with
// S_k = px_0 + ... + px_k exact; hence U > S_k + k 2^-54 gives X >= k + 1
// and U <= S_k - k 2^-54 gives X <= k.
//
// The rows hold C_k, an approximation of S_k computed in parallel (below),
// with |C_k - S_k| + k 2^-54 < 2^-42 = kGuideBand grid steps, and
//   up_k = floor(C_k 2^53) + kGuideBand + 1:  u >= up_k  =>  X >= k + 1
//   lo_k = ceil(C_k 2^53) - kGuideBand - 1:   u <= lo_k  =>  X <= k
// The error bound, with eps = 2^-53 and k <= 127: the loop's px_k is
// qn rho_0 ... rho_{k-1} (rho_i = (m - i) p / ((i + 1) q), qn = q^m as
// tabulated) times 1 + t with |t| <= gamma(4k) (four roundings a step); here
// each ratio is rounded three times and the prefix product of k of them and
// qn k times more, also gamma(4k); both are within 2 gamma(4k + 1) < 1019 eps
// relative of the same exact product, whose sum over k is qn / q^m <= 1.0001.
// Any order of summing k + 1 such terms adds at most gamma(k) < 128 eps.
// With k 2^-54 <= 64 eps that is < 1211 eps < 2048 eps.
//
// A row ends at the bound (then a sentinel makes X = bound + 1 a replay, as
// the loop's "X > bound") or at the first k whose lo_k covers the whole grid
// (X <= k for every uniform).  guide[j] is the number of leading entries
// with up <= j 2^47, the least X of any u in bucket j.
constexpr int64_t kGuideBand = 2048;

// The device builds a row with one wave (guide_kernel): chunks of 64
// entries, lane l of chunk c holding k = 64 c + l; ratio r_k (r_0 = 1),
// Hillis-Steele inclusive scans (offsets 1, 2, ..., 32) of the ratios'
// product and of px_k = qn P_k, each chunk continuing from the last lane of
// the one before.  This host function performs the same operations in the
// same order, so its rows equal the device's bit for bit.
inline int build_guide_row_host(const Model& M, const BinomTable& tab, int s, int m, ThrPair* thr,
                                uint8_t* guide) {
    const double pp = M.pp[s];
    const double q = M.qq[s];
    const int bound = tab.bound[s][m];
    const double qn = tab.qn[s][m];
    double carryP = 1.0, carryC = 0.0;
    int end = -1;
    bool covered = false;
    for (int c = 0; c * kWave < kBinomTable && end < 0; ++c) {
        double P[kWave], C[kWave], t[kWave];
        for (int l = 0; l < kWave; ++l) {
            const int k = c * kWave + l;
            P[l] = k == 0 ? 1.0 : (double(m - k + 1) * pp) / (double(k) * q);
        }
        for (int off = 1; off < kWave; off <<= 1) {
            for (int l = 0; l < kWave; ++l) t[l] = l >= off ? P[l] * P[l - off] : P[l];
            for (int l = 0; l < kWave; ++l) P[l] = t[l];
        }
        for (int l = 0; l < kWave; ++l) C[l] = qn * (P[l] * carryP);
        for (int off = 1; off < kWave; off <<= 1) {
            for (int l = 0; l < kWave; ++l) t[l] = l >= off ? C[l] + C[l - off] : C[l];
            for (int l = 0; l < kWave; ++l) C[l] = t[l];
        }
        for (int l = 0; l < kWave && end < 0; ++l) {
            const int k = c * kWave + l;
            const double cs = (C[l] + carryC) * 0x1p53;
            const int64_t lo = int64_t(ceil(cs)) - kGuideBand - 1;
            thr[k] = ThrPair{int64_t(floor(cs)) + kGuideBand + 1, lo};
            if (lo >= kU53Max) covered = true;
            if (covered || k >= bound) end = k;
        }
        carryP = P[kWave - 1] * carryP;
        carryC = C[kWave - 1] + carryC;
    }
    thr[end + 1] = ThrPair{INT64_MAX, covered ? INT64_MAX : int64_t(-1)};
    for (int j = 0; j < kGuideBuckets; ++j) {
        const int64_t u0 = int64_t(j) << kGuideShift;
        int x = 0;
        while (x <= end && thr[x].up <= u0) ++x;
        guide[j] = uint8_t(x);
    }
    return end + 1;
}

// ThrPair at index i of a table, as one load.
PDA_HD ThrPair load_pair(const ThrPair* t, uint32_t i) {
#ifdef __HIP_DEVICE_COMPILE__
    typedef long Pair __attribute__((ext_vector_type(2)));
    const Pair v = *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(t) + i * 16u);
    return ThrPair{v.x, v.y};
#else
    return t[i];
#endif
}
static_assert(sizeof(ThrPair) == 16, "a pair is one load");

// binomial_table by the thresholds: the same X for every uniform, or -1
// where binomial_table returns -1 and where u falls between lo_X and up_X
// (2 kGuideBand + 2 grid points around each threshold, ~5e-13 of the grid:
// the general form then runs the loop).
// Two dependent loads instead of X + 1 loop passes whose count differs from
// lane to lane.
//
// guided_count: X before the flip of p > 1/2, for 0 < n < kBinomTable; row is
// the state's in the table.  Offsets are 32-bit from the tables' starts (a
// table holds at most 1 GiB), and a pair is one 16-byte load.
PDA_HD int guided_count(int n, uint32_t row, const BinomGuide& G, uint32_t hi, uint32_t lo) {
    const int64_t u = (int64_t(hi >> 5) << 26) | int64_t(lo >> 6);
    int X = G.guide[(row * uint32_t(kBinomTable) + uint32_t(n)) * uint32_t(kGuideBuckets) +
                    (hi >> 26)];
    uint32_t at = row * uint32_t(kGuideStatePairs) + uint32_t(n) * uint32_t(n + 3) / 2u + uint32_t(X);
    ThrPair e = load_pair(G.thr, at);
    while (u >= e.up) {
        ++X;
        e = load_pair(G.thr, ++at);
    }
    return u > e.lo ? -1 : X;
}

PDA_HD int64_t binomial_guided(int n, int s, const Model& M, const BinomGuide& G, uint32_t hi,
                               uint32_t lo) {
    if (n <= 0) return 0;
    if (n >= kBinomTable) return -1;
    const int X = guided_count(n, uint32_t(s), G, hi, lo);
    return X < 0 ? -1 : M.flip[s] ? n - X : X;
}

// binomial() for n < kBinomTable trials of any p, or -1 where the uniform lies
// too near a threshold to tell or the inversion restarts.  As for the rows
// above, X is a non-decreasing function of the uniform that passes from k to
// k + 1 where U = S_k + d, |d| <= k 2^-54, S_k the exact sum of the loop's
// px_0 .. px_k; here C_k, the running sum of products computed with a power
// instead of exp(n log q) and one reciprocal instead of a division a step,
// stands for it, and a uniform within kBroadBand = 2^-38 of C_k is left to
// the general form (about 10^-11 of the draws).  Errors of C_k, all relative
// to sums of at most 1.0001: the power's 14 and the products' 4 k roundings
// and the reciprocal's 2^-50, below 800 x 2^-53 + 127 x 2^-50; the loop's own
// 5 k roundings; its q^n = exp(n log q), whose argument is at most 88.1 in
// magnitude and within 3 units of 2^-53 relative of the exact one, and
// exp itself: below 300 x 2^-53.  Together less than 2^-41.
constexpr double kBroadBand = 0x1p-38;
PDA_HD int binomial_broad(int n, float p, uint32_t hi, uint32_t lo) {
    if (n <= 0 || !(p >= 0.0f && p <= 1.0f)) return 0;
    if (n >= kBinomTable) return -1;
    const bool flip = p > 0.5f;
    const double pp = flip ? 1.0 - double(p) : double(p);
    const double q = 1.0 - pp;
    double C = 1.0;  // q^n by squaring
    double sq = q;
    for (int e = n; e > 0; e >>= 1) {
        if (e & 1) C *= sq;
        sq *= sq;
    }
    const double ratio = pp * reciprocal_close(q);
    const double U = uniform53(hi, lo);
    double px = C;
    double left = double(n);  // n - X
    int X = 0;
    while (U > C && X < n) {
        ++X;
        const double inv = reciprocal_close(double(X));
        px = (px * ratio) * (left * inv);
        left -= 1.0;
        if (U < C + kBroadBand) return -1;  // too near the threshold passed
        C += px;
    }
    if (U > C - kBroadBand) return -1;
    // past the loop's bound, 10 standard deviations above the mean: a restart
    const double np = double(n) * pp;
    const double over = double(X) - np;
    if (over > 0.0 && over * over > 99.0 * (np * q + 1.0)) return -1;
    return flip ? n - X : X;
}

// Division of a unit index by the resample count without a divide
// instruction sequence: for d >= 1, l = ceil(log2 d) and m = ceil(2^(31+l) / d)
// (< 2^32), floor(u m / 2^(31+l)) = floor(u / d) for every u < 2^31 (m d =
// 2^(31+l) + e with 0 <= e < d, so u m / 2^(31+l) exceeds u / d by less than
// u / 2^(31+l) * e / d < 2^-l <= 1 / d, which cannot reach the next integer).
// Unit indices stay below 2^31 (every run checks it).  Built on the host, an
// argument of the launch.
struct UnitDiv {
    uint32_t m, sh;
};
PDA_HD UnitDiv make_unit_div(uint32_t d) {
    uint32_t l = 0;
    while (l < 32u && (uint64_t(1) << l) < uint64_t(d)) ++l;
    const uint64_t m = ((uint64_t(1) << (31u + l)) + uint64_t(d) - 1u) / uint64_t(d);
    return UnitDiv{uint32_t(m), 31u + l};
}
PDA_HD uint32_t unit_div(uint32_t u, const UnitDiv& q) {
    return uint32_t((uint64_t(u) * uint64_t(q.m)) >> q.sh);
}

template <class T>
struct NoDeduce {
    using type = T;
};

// background_count() for means <= 64 (one inversion chunk) and caps below 2^30
// photons, which a 32-bit counter cannot pass (background_single: -1 for
// others).
// The inversion's first two steps run for every lane without a branch: their
// divisions by 1 and 2 are exact (the identity and a power-of-two scaling),
// so pk * lam and (pk * lam) * 0.5 round to the loop's values; the loop then
// continues from k = 3 only for the lanes whose uniform lies beyond the
// cumulative probability of 2 photons and whose cap allows it, so a wave no
// longer runs the loop as often as its longest draw needs.  (The cumulative
// sums do not decrease, so a uniform beyond one is beyond those before; a
// mean of 0 or less has exp(0) = 1, which no uniform exceeds.)
PDA_HD float background_capped(float lam, float cap, float u_first, float u_cap) {
    lam = fmaxf(lam, 0.0f);
    const float pk0 = fexp_minus(lam);
    const float pk1 = pk0 * lam;
    const float cdf1 = pk0 + pk1;
    const float pk2 = (pk1 * lam) * 0.5f;
    const float cdf2 = cdf1 + pk2;
    int32_t k = (u_first > pk0 ? 1 : 0) + (u_first > cdf1 ? 1 : 0);
    if (u_first > cdf2) {
        k = 3;
        float pk = pk2, cdf = cdf2;
        while (float(k) <= cap) {
            pk = (pk * lam) / float(k);
            cdf = cdf + pk;
            if (!(u_first > cdf)) break;
            ++k;
        }
    }
    return float(k) <= cap ? float(k) : floorf(cap * u_cap);
}
PDA_HD float background_single(float lam, float cap, float u_first, float u_cap) {
    if (lam > 64.0f || !(cap < 0x1p30f)) return -1.0f;
    return background_capped(lam, cap, u_first, u_cap);
}

// Walk state of one unit between windows.  The fast form keeps the window
// ends in 32 bits (ticks < 2^31; a larger end is replayed), the general
// form in 64 bits as the reference.
template <bool kFast>
struct WalkState {
    using Tick = typename std::conditional<kFast, uint32_t, int64_t>::type;
    int s;        // current state
    float tsum;   // mcSpendTime
    Tick w0;      // start tick of the current window (bin0clk_t)
    uint32_t c;   // photon cursor (binIdxStart)
    uint32_t w;   // window index
    float acc, F;
};

enum StepResult : int { kStepMore = 0, kStepDone = 1, kStepReplay = 2 };

// What one window drew, for the counts form (kCounts): the state it dwelt
// in, the next state, the dwell time and the photon count the binomial
// acceptor draw would have taken (int(m), <= 0 draws nothing).
struct WindowInfo {
    int s, j;
    float tau;
    int32_t m;
};

#ifdef __HIPCC__
// Writes the GPU's clock (hipDeviceAttributeWallClockRate) to *t, which may be
// host memory, unless t is null; for one thread of a launch.
__device__ __forceinline__ void stamp(uint64_t* t) {
    if (t) *t = wall_clock64();
}
#endif

// What a work counter hands out: of a single set's units a contiguous share,
// of a population's batches (set 0's, set 1's, ...) every queues-th.
struct QueueRange {
    uint32_t begin, end;
};
PDA_HD QueueRange queue_range(uint32_t queue, uint32_t share, uint32_t n) {
    const uint64_t b = uint64_t(queue) * share;
    const uint32_t begin = b < n ? uint32_t(b) : n;
    return QueueRange{begin, n - begin < share ? n : begin + share};
}

// A unit that has been started: its burst and its key.
struct StartedUnit {
    BurstDesc d;
    uint32_t r, b;
};

// Start of a unit (src/mc.cu:92-116): initial state from genMatP's inflow.
// Returns kStepDone when the unit has no window that counts anything
// (zero or one photon, or T <= 0: E = 0).
template <bool kFast>
PDA_HD int begin_unit(const FastModel& M, const UnitKey& key, uint32_t P, float T,
                      WalkState<kFast>& st) {
    st.s = 0;
    st.tsum = 0.0f;
    st.w0 = 0;
    st.c = 0;
    st.w = 0;
    st.acc = 0.0f;
    st.F = 0.0f;
    if (P <= 1u || !(T > 0.0f)) return kStepDone;
    st.s = M.init_state >= 0
               ? M.init_state
               : first_above(M.p0cum, M.n,
                             uniform24(draw_block(key, kInitWindow, kSubMain).w[0]));
    return kStepMore;
}

// Where a window that ends at tick w1 closes: the first channel photon at or
// after w1 (photons in neither channel carry its tick, the links its index),
// else the last photon.  A bound past the last but one is the last photon
// whatever its tick; c < last, as a unit whose cursor reaches it ends.
PDA_HD uint32_t window_close(const uint32_t* tick, const uint2* link, uint32_t c, uint32_t last,
                             uint32_t w1) {
    uint32_t lo = c, hi = last;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (tick[mid] < w1) lo = mid + 1u;
        else hi = mid;
    }
    if (lo < last) {
        const uint32_t f1 = link[lo].x & kIndexMask;
        if (f1 < last) return f1;
    }
    return last;
}

// One dwell window of the walk (one pass of the while loop, src/mc.cu:117-191)
// in the general form.  tick/link point at the burst's photons.
// kCounts: no acceptor draw; the window is described in *wi instead, for the
// Rao-Blackwellised form that sums the binomial pmf.
template <bool kCounts = false>
PDA_HD int general_window(const Model& M, const UnitKey& key, uint32_t P, uint32_t stop_rel,
                          float T, const uint32_t* tick, const uint2* link, const RunArgs& a,
                          WalkState<false>& st, WindowInfo* wi = nullptr) {
    const int n = M.n;
    const int s = st.s;
    const uint32_t w = st.w;
    const uint32_t last = P - 1u;
    const Block A = draw_block(key, w, kSubMain);
    // next state (drawJ_Si2Sj, src/gen_rand.cuh:78-89); forced for n == 2
    int j;
    if (n == 2) {
        j = 1 - s;
    } else {
        const int jj = first_above(M.nscum[s], n - 1, uniform24(A.w[0]));
        j = jj >= s ? jj + 1 : jj;
    }
    // dwell at the chosen transition's rate (drawTau, src/mc.cu:122)
    const float tau = flog(uniform24(A.w[1])) / (-M.krate[s][j]);
    const float tsum = st.tsum + tau;
    int64_t w1;
    uint32_t w1c;
    if (!(tsum < T)) {
        w1 = stop_rel;
        w1c = stop_rel;
    } else {
        const float wf = float(st.w0) + tsum / a.clk_p;  // src/mc.cu:132
        w1 = wf >= 0x1p62f ? (int64_t(1) << 62) : int64_t(wf);
        w1c = w1 <= 0 ? 0u : (w1 >= int64_t(kTickSentinel) ? kTickSentinel : uint32_t(w1));
    }
    const uint32_t close = window_close(tick, link, st.c, last, w1c);
    // sticky-flag count over [c, close) (src/mc.cu:171-180)
    const uint2 L = link[st.c];
    const uint32_t f = L.x & kIndexMask;
    uint32_t cnt = 0;
    if (f < close) cnt = (L.y < close ? L.y : close) - f;
    const uint32_t colour = L.x >> 30;
    const float nd = colour == 1u ? float(cnt) : 0.0f;
    const float na = colour == 2u ? float(cnt) : 0.0f;
    const float fv = M.gmx * nd + M.omdd * na;
    float m;
    if (!a.bg_on) {
        m = floorf(fv + 0.5f);
    } else {  // background photons (src/mc.cu:153-166), one channel's (see fast_window)
        const Block Bk = draw_block(key, w, kSubBackground);
        const float dt = float(w1 - st.w0) * a.clk_p;
        const bool donor = colour == 1u;
        const float bg = background_count(
            dt * (donor ? a.bg_dd : a.bg_ad), donor ? M.gmx * nd : M.omdd * na,
            uniform24(donor ? Bk.w[1] : Bk.w[0]), uniform24(donor ? Bk.w[3] : Bk.w[2]), key, w,
            donor ? kSubPoissonD : kSubPoissonA);
        m = floorf((fv - bg) + 0.5f);
    }
    int64_t x = 0;
    if (kCounts) {
        *wi = WindowInfo{s, j, tau, int32_t(m)};
    } else {
        // broadened efficiency (drawE, src/gen_rand.cuh:63-68)
        float de;
        if (M.v[s] == 0.0f) {
            de = M.ep0[s];
        } else {
            const Block C = draw_block(key, w, kSubNormal);
            de = distance_efficiency(gauss(C.w[0], C.w[1]) * M.v[s] + M.base[s], M.r0);
        }
        x = binomial(int(m), double(de), A.w[2], A.w[3], key, w);
    }
    st.F += fv;
    st.acc += float(x);
    st.tsum = tsum;
    st.w0 = w1;
    st.s = j;
    st.c = close;
    st.w = w + 1u;
    // loop condition of the next window; every window after the cursor
    // reached the last photon is empty
    if (close == last || !(T > tsum) || st.w >= kMaxWindows) return kStepDone;
    return kStepMore;
}

// What the fast form needs besides the model, the same for every unit of a
// launch: jumps = the largest state count - 2, the comparisons of the
// next-state draw; quick: the rates and the tick length are in quotient()'s
// range; clk_r: 1 / clk_p rounded to float; r0_r: 1 / r0, or 0 when r0 is
// out of that range; top: the largest power of two up to the photons of the
// longest burst, the first step of the window ends' search.
//
// fast_args gives what follows from the resident bursts; the rest follows from
// the sets' models (fast_args_of).  A single set's launch takes it from the
// device's model when it runs: recorded into a graph it may be replayed after
// the slot's parameters or photophysics changed.
struct FastArgs {
    int32_t jumps;
    int32_t quick;
    float clk_r, r0_r;
    uint32_t top;
};
PDA_HD FastArgs fast_args(float clk_p, uint32_t max_photons) {
    uint32_t top = 1;
    while (top <= max_photons / 2u) top *= 2u;
    return FastArgs{kMaxStates - 2, quotient_range(clk_p) ? 1 : 0, 1.0f / clk_p, 0.0f, top};
}
PDA_HD FastArgs fast_args_of(FastArgs fa, int max_states, int quick_rates, float r0_r) {
    fa.jumps = max_states - 2;
    fa.quick = quick_rates ? fa.quick : 0;
    fa.r0_r = r0_r;
    return fa;
}

// window_close() by steps of decreasing powers of two, the same for every
// lane: pos is the last photon found so far whose tick is below w1 (c - 1:
// none).  A step past the burst looks at its last photon: were that below w1,
// so were all.  Five vector instructions a step and a uniform loop, where the
// halving of each lane's own interval took eight and the wave's exec mask.
PDA_HD uint32_t step_close(const uint32_t* tick, const uint2* link, uint32_t c, uint32_t last,
                           uint32_t w1, uint32_t top) {
    uint32_t pos = c - 1u;
    uint32_t step = top;
#ifdef __HIP_DEVICE_COMPILE__
    while (step > 1u && !__any(last - c >= step)) step >>= 1;
#else
    while (step > 1u && !(last - c >= step)) step >>= 1;  // a wave of one lane
#endif
#pragma unroll 1
    for (; step > 0u; step >>= 1) {
        const uint32_t next = pos + step;
        const uint32_t i = next < last ? next : last;
        pos = tick[i] < w1 ? i : pos;
    }
    const uint32_t at = pos + 1u < last ? pos + 1u : last;
    const uint32_t f1 = link[at].x & kIndexMask;
    return f1 < last ? f1 : last;
}

// Tab of fast_window for models with distance broadening: the efficiency is
// drawn per window, so there is no table of its binomials.  BroadAll: counts
// beyond the table and background means above 64 are drawn in place instead of
// abandoning the unit.
struct BroadDraw {};
struct BroadAll {};

// The same window in the fast form, the same values from fewer operations;
// kStepReplay where the window needs the general form.  Tab: BinomGuide
// (thresholds) or BinomTable (inversion loop) for the acceptor draw of a
// model without distance broadening, BroadDraw or BroadAll for one with.
template <bool kCounts = false, class Tab = BinomTable, class Mod = Model>
PDA_HD int fast_window(const Mod& M, const typename NoDeduce<Tab>::type* tab, const UnitKey& key,
                       uint32_t P, uint32_t stop_rel, float T, const uint32_t* tick,
                       const uint2* link, const RunArgs& a, const FastArgs& fa,
                       WalkState<true>& st, WindowInfo* wi = nullptr) {
    constexpr bool kAll = std::is_same<Tab, BroadAll>::value;
    constexpr bool kBroad = kAll || std::is_same<Tab, BroadDraw>::value;
    const int s = st.s;
    const uint32_t w = st.w;
    const uint32_t last = P - 1u;
    const Block A = draw_block(key, w, kSubMain);
    // next state: the running sums do not decrease, so the first one above u
    // comes after as many as are not above it (a rate sum of 0 makes them
    // NaN, never above); the entries from n - 2 on are +inf
    const float us = uniform24(A.w[0]);
    int j = (M.nscum[s][0] > us ? 0 : 1) + (M.nscum[s][1] > us ? 0 : 1);
#pragma unroll 1
    for (int i = 2; i < fa.jumps; ++i) j += M.nscum[s][i] > us ? 0 : 1;
    j += j >= s ? 1 : 0;
    const float lg = flog_uniform24(A.w[1]);
    const float mk = M.kdiv[s][j][0];
    const float tau = fa.quick ? quotient(lg, mk, M.kdiv[s][j][1]) : lg / mk;
    const float tsum = st.tsum + tau;
    const float ticks = fa.quick ? quotient(tsum, a.clk_p, fa.clk_r) : tsum / a.clk_p;
    const float wf = float(st.w0) + ticks;
    const bool ends = !(tsum < T);
    // bad: the window needs the general form (its values below are not used)
    bool bad = !ends && !(wf < 0x1p31f);
    const uint32_t w1 = ends ? stop_rel : bad ? 0u : uint32_t(wf);
    const uint32_t close = step_close(tick, link, st.c, last, w1, fa.top);
    // the count of the one colour the window has (0 for a photon in both
    // channels, whose run ends at itself)
    const uint2 L = link[st.c];
    const uint32_t f = L.x & kIndexMask;
    const uint32_t e = L.y < close ? L.y : close;
    const float cnt = float(e > f ? e - f : 0u);
    const bool donor = (L.x >> 30) == 1u;
    const float fv = (donor ? M.gmx : M.omdd) * cnt;
    float m = fv;
    if (a.bg_on) {
        // Background photons (src/mc.cu:153-166).  The window's photons carry
        // one colour, so one of the two capped draws has a cap of 0 and gives
        // 0 whatever its uniforms are (k = 0, or past the cap with
        // floor(0 u) = 0): only the other is made, on its channel's rate and
        // words (the window leaves the fast form when either mean is above
        // 64, unless kAll).  One exponential and one inversion loop per window instead of
        // two, whose lanes had each waited for the other channel's (with two
        // draws a 3-state evaluation of 100,000 bursts x 100 took 434 us and
        // the 256-set generation 19.9 ms, with one 417 us and 19.1 ms; under
        // a 30 kHz background 323 and 275 us).  (fv - bgd) - bga is fv - bg
        // then, exactly.
        const Block Bk = draw_block(key, w, kSubBackground);
        const float dt = float(int32_t(w1 - st.w0)) * a.clk_p;
        const bool many = dt * fmaxf(a.bg_ad, a.bg_dd) > 64.0f || !(fv < 0x1p30f);
        const float lam = dt * (donor ? a.bg_dd : a.bg_ad);
        const float u_first = uniform24(donor ? Bk.w[1] : Bk.w[0]);
        const float u_cap = uniform24(donor ? Bk.w[3] : Bk.w[2]);
        if (kAll && many && !bad) {
            m = fv - background_count(lam, fv, u_first, u_cap, key, w,
                                      donor ? kSubPoissonD : kSubPoissonA);
        } else {
            bad = bad || many;
            m = fv - background_capped(fminf(lam, 64.0f), bad ? 0.0f : fv, u_first, u_cap);
        }
    }
    m = floorf(m + 0.5f);
    if (kCounts) {
        *wi = WindowInfo{s, j, tau, int32_t(m)};
    } else {
        const int n = int(m);
        int x = 0;
        if constexpr (kBroad) {
            // broadened efficiency (drawE, src/gen_rand.cuh:63-68)
            float de = M.ep0[s];
            if (M.v[s] != 0.0f) {
                const Block C = draw_block(key, w, kSubNormal);
                const float rd = gauss_uniform24(C.w[0], C.w[1]) * M.v[s] + M.base[s];
                de = fa.r0_r != 0.0f ? distance_efficiency_quick(rd, M.r0, fa.r0_r)
                                     : distance_efficiency(rd, M.r0);
            }
            if (kAll && n >= kBinomTable && !bad)
                x = int(binomial(n, double(de), A.w[2], A.w[3], key, w));
            else
                x = binomial_broad(n, de, A.w[2], A.w[3]);
            bad = bad || x < 0;
        } else if constexpr (std::is_same<Tab, BinomGuide>::value) {
            bad = bad || n >= kBinomTable;
            if (n > 0 && !bad) {
                x = guided_count(n, uint32_t(M.guide_base + s), *tab, A.w[2], A.w[3]);
                bad = x < 0;
                x = M.flip[s] ? n - x : x;
            }
        } else {
            x = int(binomial_table(n, s, M, *tab, A.w[2], A.w[3]));
            bad = bad || x < 0;
        }
        st.acc += float(x);
    }
    st.F += fv;
    st.tsum = tsum;
    st.w0 = w1;
    st.s = j;
    st.c = close;
    st.w = w + 1u;
    if (bad) return kStepReplay;
    if (close == last || !(T > tsum) || st.w >= kMaxWindows) return kStepDone;
    return kStepMore;
}

// One (burst, resample) unit: the body of mc_kernel (src/mc.cu:92-196).
template <bool kFast, class Tab = BinomTable>
PDA_HD WalkOut walk_unit(const Model& M, const typename NoDeduce<Tab>::type* tab, const UnitKey& key,
                         uint32_t P, uint32_t stop_rel, float T, const uint32_t* tick,
                         const uint2* link, const RunArgs& a) {
    WalkState<kFast> st;
    int r = begin_unit<kFast>(M, key, P, T, st);
    if constexpr (kFast) {
        const FastArgs fa = fast_args_of(fast_args(a.clk_p, P), M.n, M.quick_rates, M.r0_r);
        while (r == kStepMore)
            r = fast_window<false, Tab>(M, tab, key, P, stop_rel, T, tick, link, a, fa, st);
    } else {
        while (r == kStepMore) r = general_window(M, key, P, stop_rel, T, tick, link, a, st);
    }
    return WalkOut{st.acc, st.F, r == kStepReplay};
}

}  // namespace pda
