// pda_kernels.hip -- gfx950 kernels of the Monte-Carlo PDA hot path.
//
// fast_walk_kernel and walk_kernel replace gSMFRETda's mc_kernel
// (src/mc.cu:83-197) together with the host histogram and chi2 of src/streamWorker.cpp:184-206:
//   * one-wave workgroups; every lane streams through (burst, resample)
//     units taken from per-XCD work counters, advancing one dwell window
//     per loop pass, so lanes and waves never wait for the longest unit;
//   * each window end is located by a binary search over burst-relative
//     uint32 ticks and the window's sticky-flag count read from per-photon
//     channel-run links, instead of rescanning photons;
//   * random numbers are stateless Philox4x32-10 blocks keyed by
//     (seed, set, window, sub-stream, resample, burst) -- no RNG state in
//     memory, nothing to initialise (replaces setup_kernel,
//     src/gen_rand.cuh:7-25);
//   * the common case runs in a lean form (fast_walk_kernel, at most 64 VGPRs,
//     with distance broadening 69 or 72, 80 where its rare draws are made in
//     place); the units that need more are listed and replayed in full by
//     walk_kernel over the whole grid, whose last workgroup sums the
//     accumulator rows, computes chi2 and writes both to the host's result
//     buffer.
#include <hip/hip_runtime.h>

#include "pda_math.h"
#include "pda_rb.h"
#include "pda_types.h"
#include "pda_walk.h"

namespace pda {

// Work counters of a replay pass: one per XCD, on the counter lines after the
// kMaxQueues lines of the walk (kAuxQueues of them).
constexpr uint32_t kReplayQueues = 8;
static_assert(kReplayQueues <= kAuxQueues, "replay counters live on the auxiliary lines");

// Set in the work counters of a population's walk to end it; the batches it
// hands out are fewer.
constexpr uint32_t kStopped = 1u << 31;

// Lanes of the mask below this one.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}

// Orders the LDS accesses of the wave's lanes: what a lane wrote before is
// visible to every lane's reads after it (one-wave workgroups, no barrier).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// A unit's efficiency into the LDS histogram.
__device__ __forceinline__ void tally(int32_t* h, int B, float acc, float F) {
    const float E = F > 0.0f ? acc / F : 0.0f;
    if (E >= 0.0f && E < 1.0f) {
        const int bin = int(floor(double(E) * double(B)));
        if (bin < B) atomicAdd(&h[bin], 1);
    }
}

// The per-unit outputs of a run that keeps samples.
__device__ __forceinline__ void store_sample(uint32_t u, float acc, float F, float* outE,
                                             int32_t* outAcc, float* outF) {
    outE[u] = F > 0.0f ? acc / F : 0.0f;
    outAcc[u] = int32_t(acc);
    outF[u] = F;
}

// Adds an LDS histogram to an accumulator row and clears it.
__device__ __forceinline__ void flush_hist(int32_t* h, int32_t* __restrict__ row, int B,
                                           uint32_t lane) {
    for (uint32_t i = lane; i < uint32_t(B); i += kWave) {
        const int32_t v = h[i];
        if (v) {
            atomicAdd(&row[i], v);
            h[i] = 0;
        }
    }
}

// ---- walk in the fast form --------------------------------------------------------
//
// The fast form of a run (one parameter set) or of a population's generation,
// in one-wave workgroups.
//
// Work stealing at two levels.  A wave takes batches of consecutive units
// from a work counter; its lanes take units from the batch as they need
// them.  One loop pass advances every busy lane by one window, and a lane
// whose unit ends starts another in the same pass, so lanes do not wait
// for the wave's longest unit and waves do not wait for the grid's
// slowest batch.  The units are split into a.queues contiguous ranges
// with a counter each, every counter on its own 256-byte line (device-
// scope atomics to one line serialise); workgroup g draws from queue
// g % a.queues, so with a multiple of 8 queues each queue is served by
// one XCD and its bursts stay in that XCD's L2.  Batches are small
// (about six grabs per wave, 32 for a population): the wave that grabs
// last still walks a whole batch, so the batch sets the grid's tail.
// Photons are read through L1/L2.
//
// A population's work is a flat list of batches: set s owns batches
// [s * bps, (s + 1) * bps), each covering up to a.batch consecutive units of
// that set; the list is dealt out to the counters in turn: a set's units take a
// multiple of another's under faster dynamics, and with contiguous shares a
// queue had whole sets, its waves (only they take from it) ending long after
// the others'.
// A wave's lanes may be walking units of two sets at once: the workgroup keeps
// two LDS model slots with an LDS histogram each, and a wave moves to a third
// set only after the older slot's lanes have finished, so it never drains to
// change sets.
//
// kPop: population (two LDS model slots with a histogram each); kPass: the
// acceptor draw (kPassGuided, kPassTable, kPassBroad, kPassBroadAll); kSamples:
// per-unit outputs.
//
// Bound by VALU issue on large runs (90 % of the cycles for 100,000 bursts x 100
// of 3 states, all of them for 256 sets; 68 % for 50,000 x 32 alone, whose end
// has idle lanes), so what counts is the instructions of fast_window: the
// window's arithmetic without the cases its arguments cannot have, correctly
// rounded quotients from reciprocals kept per model, and the launch's divisions
// done on the host (unit / R, the queues' shares) took a 3-state evaluation of
// 100,000 bursts x 100 from 459 to 407 us and the 256-set generation from 16.7
// to 14.7 ms; a search in uniform steps, 32-bit draws and windows without early
// returns from there to 387 us and 13.2 ms.  The register limit keeps 8 waves
// on a SIMD: the window loop waits on dependent loads, which the
// other waves hide (the 256-set generation 11.3 ms on the GPU with 7 and 10.6
// with 8, 64 sets of fast dynamics 12.1 and 11.3).
// A single set's bursts are started by falling duration within each quarter of
// a queue's share (burst_order in pda_layout.cpp), so that a run ends with units
// of few windows and not with some lane's thirtieth: 50,000 bursts x 50 of 3
// states under a 30 kHz background 272 -> 223 us, 100,000 x 100 of 3 states
// 315 -> 304 (one data set, its photons cached; 327 where three take turns).
// With whole shares sorted those take 244 and 313, with all bursts sorted and
// dealt out to the queues 248 and 318, and a population 6 % more; populations, whose other sets fill the end of each, and the RB walk, which
// writes per burst, start them as they come.
// Units are started 64 at a time into LDS and taken from there one lane at a
// time as lanes fall idle, and ended ones wait in LDS until 64 can be binned:
// a start (a Philox block and the unit's division) and a tally (a division and
// a floor in double) would otherwise run for the one or two lanes of a pass
// that need them.  64 sets of fast dynamics 11.27 -> 10.53 ms on the GPU,
// 100,000 x 100 of 3 states 293 -> 288 us; 256 sets of slow dynamics the same
// (10.62).  The population's workgroup has to stay within 5,120 bytes of LDS
// for 32 of them on a CU (LDS is handed out in 1,280), which is why the models
// come in parts.  That holds up to 96 bins (broadened 72); beyond, 25 share a CU
// and the 256 sets take 12.9 ms at 100 or 200 bins for 10.7 at 50, the 64 of
// fast dynamics 12.1 for 10.5 and the broadened ones 1.04 for 0.97.  (Starting
// units together with their first windows was slower: 14 % more instructions,
// the first window's close running for half of the lanes.)
// The draw of a broadened efficiency and its binomial (kPassBroad) need up to
// 72 registers (7 waves for populations: 0.94 ms against 0.98 with 6 on the
// 64 sets below; no difference for single sets).  They had been the general
// form's, at 186 registers and two waves per SIMD with logarithms,
// exponentials and divisions in double per window: 50,000 bursts x 50 of a
// 3-state model 371 -> 197 us, 64 sets x 20,000 x 16 2.74 -> 1.41 ms.
//
// kPassBroadAll: counts beyond the table and background means above 64 are
// drawn in the window.  A broadened unit had not been abandoned for them before
// it had a fast form; with each of them listed by one atomic and walked again
// (populations: the whole run again once the list was full), 64 sets of 8,000
// bursts x 64 at efficiencies near 0.99, 17 % of their units abandoned, took
// 8.5 ms where the general form had taken 3.5, and under a 60 kHz background
// 17.0 against 8.3; with the draws in place 1.9 and 2.1.  The draws spill up to
// 392 bytes where they are made; with 6 waves the 64 sets below take 1.06 ms,
// with 5 1.09, 4 1.23 and 3 1.44, against kPassBroad's 0.95: which of the two
// a run takes is decided by its bursts (draws_in_place in pda_layout.cpp).
constexpr bool is_broad(int pass) { return pass == kPassBroad || pass == kPassBroadAll; }
constexpr int fast_waves_per_eu(bool pop, int pass) {
    return !is_broad(pass) ? 8 : pop && pass == kPassBroad ? 7 : 6;
}

struct FastIO {
    const WalkBurst* bursts;
    const uint32_t* ticks;
    const uint2* links;
    const Model* models;       // [1], or the population's sets
    const BinomTable* tabs;    // kPassTable: [sets]
    const PopControl* ctl;     // population: the sets' stream keys
    BinomGuide guide;
    int32_t* hist_acc;
    void* replay;              // uint32 units; population: (set << 32 | unit)
    uint32_t* replay_count;
    uint32_t* work;
    float* outE;
    int32_t* outAcc;
    float* outF;
    RunTimes* times;           // or null
};

template <bool kPop, int kPass, bool kSamples>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(
    fast_waves_per_eu(kPop, kPass)))) void fast_walk_kernel(const FastIO io, const RunArgs a,
                                                            const FastArgs launch) {
    constexpr int kSlots = kPop ? 2 : 1;
    // (broadened walks choose their form so that the list suffices)
    constexpr bool kStops = kPop && !is_broad(kPass);
    using Mod = typename std::conditional<
        kPass == kPassGuided, FastModel,
        typename std::conditional<is_broad(kPass), BroadModel, Model>::type>::type;
    __shared__ Mod sM[kSlots];
    __shared__ StartedUnit s_start[kWave];    // units started and not yet taken
    __shared__ uint8_t s_state[kWave];        // their first states
    __shared__ float2 s_done[2 * kWave];      // (acc, F) of units not yet binned
    extern __shared__ int32_t s_hist[];       // [kSlots][a.B]
    const uint32_t lane = threadIdx.x;
    for (uint32_t i = lane; i < uint32_t(kSlots) * uint32_t(a.B); i += kWave) s_hist[i] = 0;
    auto load_model = [&](uint32_t into, uint32_t set) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(&io.models[set]);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&sM[into]);
        for (uint32_t i = lane; i < sizeof(Mod) / 4; i += kWave) dst[i] = src[i];
        wave_lds_sync();
    };
    FastArgs fa = launch;
    if constexpr (!kPop) {
        // from memory, beside the copy to LDS: from the copy they made 20,000
        // bursts x 4 of 3 broadened states walk for 30.0 us instead of 29.6
        const Model& M = io.models[0];
        fa = fast_args_of(launch, __builtin_amdgcn_readfirstlane(M.n),
                          __builtin_amdgcn_readfirstlane(M.quick_rates),
                          bitsf(__builtin_amdgcn_readfirstlane(fbits(M.r0_r))));
        load_model(0u, 0u);
    }

    // (as the first instruction it cost broadened runs of 50 us 0.6)
    if (!kPop && io.times && blockIdx.x == 0 && lane == 0) stamp(&io.times->start);

    const uint32_t seed = kPop ? io.ctl->seed : a.seed;
    const uint32_t queue = blockIdx.x % a.queues;
    const QueueRange q = queue_range(queue, a.q_share, kPop ? 0u : a.nunits);
    const uint32_t batches = a.nsets * a.bps;
    const uint32_t xrow = blockIdx.x & 7u;
    const UnitDiv divR{a.div_m, a.div_sh};
    int set0 = kPop ? -1 : 0, set1 = -1;  // the set each LDS slot holds
    uint32_t cur = 0;                     // slot whose units are being started
    uint32_t pool_set = 0, pool_next = 0, pool_end = 0;
    uint32_t started = 0, start_next = 0;  // entries of s_start, the next to take
    uint32_t done = 0;                     // entries of s_done
    bool drained = false;
    bool busy = false;
    uint32_t slot = 0;
    WalkState<true> st{};
    UnitKey key{seed, a.set, 0u, 0u};
    BurstDesc d{0u, 0u, 0u, 0.0f};
    // bins the first `count` (at most 64) waiting units, one per lane
    auto bin_done = [&](uint32_t first, uint32_t count) {
        wave_lds_sync();
        if (lane < count) {
            const float2 r = s_done[first + lane];
            const uint32_t sl = kPop ? fbits(r.y) >> 31 : 0u;  // F's sign: the slot
            tally(s_hist + sl * uint32_t(a.B), a.B, r.x, kPop ? fabsf(r.y) : r.y);
        }
    };
    while (true) {
        while (true) {
            const uint64_t want = __ballot(!busy);
            if (want == 0) break;
            if (start_next == started) {  // start 64 units
                if (pool_next >= pool_end) {
                    if (drained) break;
                    uint32_t k = 0;
                    if (lane == 0)
                        k = atomicAdd(&io.work[queue * kCounterStride], kPop ? 1u : a.batch);
                    k = __builtin_amdgcn_readfirstlane(k);
                    if (kPop) k = !kStops || k < kStopped ? k * a.queues + queue : k;
                    if (k >= (kPop ? batches : q.end - q.begin)) {
                        drained = true;
                        break;
                    }
                    if (kPop) pool_set = k / a.bps;
                    pool_next = kPop ? (k - pool_set * a.bps) * a.batch : q.begin + k;
                    const uint32_t end = kPop ? a.nunits : q.end;
                    pool_end = end - pool_next < a.batch ? end : pool_next + a.batch;
                }
                if (kPop && int(pool_set) != (cur ? set1 : set0)) {
                    const uint32_t other = cur ^ 1u;
                    if (__any(busy && slot == other)) break;  // the older set is still walking
                    const int old = other ? set1 : set0;
                    if (old >= 0) {
                        bin_done(0u, done);
                        done = 0;
                        wave_lds_sync();
                        flush_hist(s_hist + other * uint32_t(a.B),
                                   io.hist_acc + (size_t(old) * 8u + xrow) * size_t(a.B), a.B,
                                   lane);
                    }
                    load_model(other, pool_set);
                    if (other) set1 = int(pool_set);
                    else set0 = int(pool_set);
                    cur = other;
                }
                const uint32_t u = pool_next + lane;
                bool walks = false;
                int state = 0;
                StartedUnit e;
                if (u < pool_end) {
                    const uint32_t i = unit_div(u, divR);
                    e.d = io.bursts[a.begin + i].d;
                    e.b = io.bursts[a.begin + i].b;
                    e.r = u - i * a.R;
                    const UnitKey k{seed,
                                    kPop ? io.ctl->set_base + pool_set * io.ctl->set_stride : a.set,
                                    e.r, e.b};
                    WalkState<true> s0;
                    walks = begin_unit<true>(sM[kPop ? cur : 0u], k, e.d.P, e.d.T, s0) == kStepMore;
                    state = s0.s;
                    if (!walks) {
                        tally(s_hist + (kPop ? cur : 0u) * uint32_t(a.B), a.B, 0.0f, 0.0f);
                        if (kSamples)
                            store_sample((e.b - a.begin) * a.R + e.r, 0.0f, 0.0f, io.outE,
                                         io.outAcc, io.outF);
                    }
                }
                pool_next = pool_end - pool_next < kWave ? pool_end : pool_next + kWave;
                const uint64_t walking = __ballot(walks);
                if (walks) {
                    s_start[lanes_below(walking)] = e;
                    s_state[lanes_below(walking)] = uint8_t(state);
                }
                wave_lds_sync();
                start_next = 0;
                started = uint32_t(__popcll(walking));
                continue;
            }
            const uint32_t left = started - start_next;
            const uint32_t rank = lanes_below(want);
            if (!busy && rank < left) {
                const StartedUnit e = s_start[start_next + rank];
                d = e.d;
                key.r = e.r;
                key.b = e.b;
                slot = cur;
                if (kPop) key.set = io.ctl->set_base + uint32_t(cur ? set1 : set0) * io.ctl->set_stride;
                st = WalkState<true>{};
                st.s = s_state[start_next + rank];
                busy = true;
            }
            const uint32_t taken = uint32_t(__popcll(want));
            start_next += taken < left ? taken : left;
        }
        if (!__any(busy)) break;
        bool ended = false;
        if (busy) {
            const Mod& M = sM[kPop ? slot : 0u];
            const uint32_t set = kPop ? uint32_t(slot ? set1 : set0) : 0u;
            const uint32_t* ticks = io.ticks + d.off;
            const uint2* links = io.links + d.off;
            int r;
            if constexpr (is_broad(kPass)) {
                using Draw = typename std::conditional<kPass == kPassBroad, BroadDraw, BroadAll>::type;
                const Draw draw{};
                r = fast_window<false, Draw>(M, &draw, key, d.P, d.stop_rel, d.T, ticks, links, a,
                                             fa, st);
            } else if constexpr (kPass == kPassGuided) {
                r = fast_window<false, BinomGuide>(M, &io.guide, key, d.P, d.stop_rel, d.T, ticks,
                                                   links, a, fa, st);
            } else {
                r = fast_window<false, BinomTable>(M, &io.tabs[set], key, d.P, d.stop_rel,
                                                   d.T, ticks, links, a, fa, st);
            }
            busy = r == kStepMore;
            ended = r == kStepDone;
            if (r == kStepReplay) {
                const uint32_t u = (key.b - a.begin) * a.R + key.r;
                const uint32_t i = atomicAdd(io.replay_count, 1u);
                if (i < a.replay_cap) {
                    if (kPop) static_cast<uint64_t*>(io.replay)[i] = (uint64_t(set) << 32) | u;
                    else static_cast<uint32_t*>(io.replay)[i] = u;
                } else if (kStops) {
                    // more than the list holds: the run is repeated as a whole
                    // (pda_get_population_result), what is left of it is not
                    // walked.  (Had the waves looked at the list's count instead
                    // where they take a batch, the looks and the atomics on that
                    // line would have held each other up: 11 sets x 8,547 x 25,
                    // 2 % abandoned, 2.4 ms for 0.75.)
                    atomicOr(&io.work[queue * kCounterStride], kStopped);
                }
            }
            if (kSamples && ended)
                store_sample((key.b - a.begin) * a.R + key.r, st.acc, st.F, io.outE, io.outAcc,
                             io.outF);
        }
        // ended units wait until 64 can be binned together
        const uint64_t ends = __ballot(ended);
        if (ended)
            s_done[done + lanes_below(ends)] =
                make_float2(st.acc, kPop ? bitsf(fbits(st.F > 0.0f ? st.F : 0.0f) | slot << 31)
                                         : st.F);
        done += uint32_t(__popcll(ends));
        if (done >= kWave) {
            done -= kWave;
            bin_done(done, kWave);  // the last 64: those before them keep their places
        }
    }
    bin_done(0u, done);
    wave_lds_sync();
    if (kPop) {
        if (set0 >= 0)
            flush_hist(s_hist, io.hist_acc + (size_t(set0) * 8u + xrow) * size_t(a.B), a.B, lane);
        if (set1 >= 0)
            flush_hist(s_hist + uint32_t(a.B),
                       io.hist_acc + (size_t(set1) * 8u + xrow) * size_t(a.B), a.B, lane);
    } else {
        flush_hist(s_hist, io.hist_acc + size_t(xrow) * kMaxBins, a.B, lane);
    }
}

// The bursts as the walks start them, formed here from their indices: the two
// arrays made on the host and copied were a twentieth of a load's time.
__global__ __launch_bounds__(256) void order_kernel(const BurstDesc* __restrict__ bursts,
                                                    const uint32_t* __restrict__ idx, uint32_t n,
                                                    WalkBurst* __restrict__ plain,
                                                    WalkBurst* __restrict__ order) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const uint32_t b = idx[i];
    plain[i] = WalkBurst{bursts[i], i, {0u, 0u, 0u}};
    order[i] = WalkBurst{bursts[b], b, {0u, 0u, 0u}};
}

// chi2 of one histogram by one wave, as src/streamWorker.cpp:194-206: the
// reference's float accumulation and FP64.  Reads the 8 accumulator rows
// (`pitch` apart, left zero for the next run) and writes their sum.
//
// The reference's sum is a chain of dependent conversions and additions, one
// per bin.  Lane b forms bin b's terms, 64 bins at a time; the chain then
// runs over the lanes by readlane, a bin's terms ready before its turn.  An
// empty bin's terms are zero, which adds nothing: no branch in the chain.
// (It had been a loop of one thread over LDS: 24 us for 200 bins, 8.6 for
// 50, of which the rest of the kernel is 3.)
struct Chi2Sum {
    float c32;
    double c64;
    int filled;  // bins of the sum that are not empty
};
__device__ __forceinline__ double lane_value(double v, int l) {
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(b), l);
    const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(b >> 32), l);
    return __longlong_as_double((long long)(uint64_t(hi) << 32 | lo));
}
__device__ __forceinline__ Chi2Sum chi2_fold(const RunArgs& a, const float* __restrict__ obs,
                                             int32_t* __restrict__ rows, size_t pitch,
                                             int32_t* __restrict__ hist, uint32_t lane) {
    Chi2Sum r{0.0f, 0.0, 0};
    const uint32_t B = uint32_t(a.B);
    const float Rf = float(a.R);
    int32_t next[8];  // the next 64 bins' rows, on their way during the chain
    float next_obs = 0.0f;
    auto fetch = [&](uint32_t b) {
        if (b < B) {
#pragma unroll
            for (uint32_t x = 0; x < 8u; ++x)
                next[x] = __hip_atomic_load(&rows[x * pitch + b], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
            next_obs = obs[b];
        }
    };
    fetch(lane);
    for (uint32_t base = 0; base < B; base += kWave) {
        const uint32_t b = base + lane;
        int32_t Mb = 0;
        const float ob = next_obs;
        if (b < B) {
#pragma unroll
            for (uint32_t x = 0; x < 8u; ++x) {
                if (next[x]) rows[x * pitch + b] = 0;
                Mb += next[x];
            }
            hist[b] = Mb;
        }
        fetch(b + kWave);
        // per-bin terms: FP64, and the reference's double term of a float
        // difference (pow(float, 2) / float, src/streamWorker.cpp:200-201)
        double t64 = 0.0, t32 = 0.0;
        const bool filled = Mb > 0 && int(b) >= a.left_pad;
        if (filled) {
            const float Mf = float(Mb);
            const float dlt = ob - Mf / Rf;
            t32 = (double(dlt) * double(dlt)) / double(Mf / Rf);
            const double md = double(Mb) / double(a.R);
            const double dd = double(ob) - md;
            t64 = dd * dd / md;
        }
        r.filled += __popcll(__ballot(filled));
#pragma unroll 8
        for (int l = 0; l < kWave; ++l) {
            r.c32 = float(double(r.c32) + lane_value(t32, l));
            r.c64 += lane_value(t64, l);
        }
    }
    return r;
}

// Ends a single set's run (one wave): histogram, chi2, and the run's counters
// (walk and replay queues, replay count) back to zero.
__device__ __forceinline__ void finish_run(const RunArgs& a, const float* __restrict__ obs,
                                           int32_t* __restrict__ hist_acc,
                                           uint32_t* __restrict__ replay_count, uint32_t replays,
                                           uint32_t* __restrict__ work,
                                           ResultHeader* __restrict__ result, uint32_t lane) {
    const Chi2Sum c = chi2_fold(a, obs, hist_acc, kMaxBins,
                                reinterpret_cast<int32_t*>(result + 1), lane);
    if (lane == 0) {
        const int dof = c.filled - a.nstates * (a.nstates + 1);
        ResultHeader r{};
        r.chi2_ref = c.c32 / float(dof);
        r.chi2_64 = c.c64 / double(dof);
        r.effN = c.filled;
        r.units = int64_t(a.nunits);
        r.B = a.B;
        r.replays = int32_t(replays);
        *result = r;
        *replay_count = 0u;
    }
    for (uint32_t q = lane; q < kMaxQueues + kAuxQueues + 1u; q += kWave)
        work[q * kCounterStride] = 0u;
}

// ---- walk in the general form ---------------------------------------------------
//
// Walks this workgroup's share of a replay list in the general form and adds
// its histogram to its XCD's accumulator row (workgroups are dispatched to the
// 8 XCDs round-robin, so the atomics of a launch spread over 8 x B addresses).
__device__ __forceinline__ void replay_units(
    const BurstDesc* __restrict__ bursts, const uint32_t* __restrict__ ticks,
    const uint2* __restrict__ links, const Model* __restrict__ model, const RunArgs& a,
    int32_t* __restrict__ hist_acc, const uint32_t* __restrict__ replay, uint32_t nunits,
    uint32_t alive, uint32_t* __restrict__ work, float* __restrict__ outE,
    int32_t* __restrict__ outAcc, float* __restrict__ outF, uint32_t lane) {
    __shared__ Model sM;
    extern __shared__ int32_t s_hist[];  // [a.B]
    const uint32_t queues = alive < kReplayQueues ? alive : kReplayQueues;
    const uint32_t queue = blockIdx.x % queues;
    {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(model);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&sM);
        for (uint32_t i = lane; i < sizeof(Model) / 4; i += kWave) dst[i] = src[i];
        for (uint32_t i = lane; i < uint32_t(a.B); i += kWave) s_hist[i] = 0;
    }
    __syncthreads();

    // handed out as in fast_walk_kernel, a wave's worth at a time
    const uint32_t share = (nunits + queues - 1u) / queues;
    const uint32_t q_begin = queue * share < nunits ? queue * share : nunits;
    const uint32_t q_end = nunits - q_begin < share ? nunits : q_begin + share;
    uint32_t* counter = &work[(kMaxQueues + queue) * kCounterStride];
    uint32_t pool_next = 0, pool_end = 0;  // the wave's current batch
    bool busy = false;
    uint32_t u = 0;
    WalkState<false> st{};
    UnitKey key{a.seed, a.set, 0u, 0u};
    BurstDesc d{0u, 0u, 0u, 0.0f};
    const UnitDiv divR{a.div_m, a.div_sh};
    bool drained = false;
    while (true) {
        bool need = !busy;
        while (!drained) {
            const uint64_t want = __ballot(need);
            if (want == 0) break;
            if (pool_next >= pool_end) {
                uint32_t off = 0;
                if (lane == 0) off = atomicAdd(counter, uint32_t(kWave));
                off = __shfl(off, 0);
                if (off >= q_end - q_begin) {
                    drained = true;
                    break;
                }
                pool_next = q_begin + off;
                pool_end = q_end - pool_next < kWave ? q_end : pool_next + kWave;
            }
            const uint32_t rank = lanes_below(want);
            const uint32_t avail = pool_end - pool_next;
            if (need && rank < avail) {
                u = replay[pool_next + rank];
                const uint32_t bl = unit_div(u, divR);
                const uint32_t b = a.begin + bl;
                d = bursts[b];
                key.r = u - bl * a.R;
                key.b = b;
                if (begin_unit<false>(sM, key, d.P, d.T, st) == kStepMore) {
                    busy = true;
                    need = false;
                } else {
                    tally(s_hist, a.B, 0.0f, 0.0f);
                    if (outE) store_sample(u, 0.0f, 0.0f, outE, outAcc, outF);
                }
            }
            const uint32_t taken = uint32_t(__popcll(want));
            pool_next += taken < avail ? taken : avail;
        }
        if (!__any(busy)) break;
        if (busy) {
            const int r = general_window(sM, key, d.P, d.stop_rel, d.T, ticks + d.off,
                                         links + d.off, a, st);
            if (r != kStepMore) {
                tally(s_hist, a.B, st.acc, st.F);
                if (outE) store_sample(u, st.acc, st.F, outE, outAcc, outF);
                busy = false;
            }
        }
    }
    __syncthreads();
    flush_hist(s_hist, hist_acc + size_t(blockIdx.x & 7u) * kMaxBins, a.B, lane);
}

// The units the fast form abandoned, launched right after it on the same
// stream, so the replay list and its count are final; and the end of the run.
// The workgroup that adds its histogram last ends the run; where nothing was
// abandoned -- most runs -- that is workgroup 0 at once, without a counter.
// With the end as a launch of its own, on one thread's chain, and a copy of the
// result behind it, 5,000 bursts x 20 of 2 states at 50 bins took 80 us and
// 20,000 x 4 of 3 broadened states at 200 bins 115; now 69 and 89.
__global__ __launch_bounds__(kWave) void walk_kernel(
    const BurstDesc* __restrict__ bursts, const uint32_t* __restrict__ ticks,
    const uint2* __restrict__ links, const Model* __restrict__ model, const RunArgs a,
    int32_t* __restrict__ hist_acc, const uint32_t* __restrict__ replay,
    uint32_t* __restrict__ replay_count, uint32_t* __restrict__ work, float* __restrict__ outE,
    int32_t* __restrict__ outAcc, float* __restrict__ outF, const float* __restrict__ obs,
    ResultHeader* __restrict__ result, RunTimes* __restrict__ times) {
    if (times && blockIdx.x == 0 && threadIdx.x == 0) stamp(&times->walked);
    const uint32_t c = *replay_count;
    const uint32_t nunits = c < a.replay_cap ? c : a.replay_cap;
    // as many workgroups as the list needs a wave for, each queue served by
    // at least one of them
    const uint32_t waves = (nunits + kWave - 1u) / kWave;
    const uint32_t alive = waves < gridDim.x ? waves : gridDim.x;
    const uint32_t lane = threadIdx.x;
    if (blockIdx.x >= (alive ? alive : 1u)) return;  // uniform over the workgroup
    if (alive) {
        replay_units(bursts, ticks, links, model, a, hist_acc, replay, nunits, alive, work, outE,
                     outAcc, outF, lane);
        __threadfence();
        uint32_t ended = 0;
        if (lane == 0) ended = atomicAdd(&work[(kMaxQueues + kAuxQueues) * kCounterStride], 1u);
        if (__builtin_amdgcn_readfirstlane(ended) + 1u != alive) return;
        __threadfence();
    }
    // (a workgroup that has not yet read the replay count, and now reads
    // zero, is not workgroup 0, which has been counted: it returns)
    finish_run(a, obs, hist_acc, replay_count, c, work, result, lane);
    if (times && lane == 0) stamp(&times->end);
}

// One threshold row of the fast walk's binomial draws, by one wave: state s
// with m photons (the operations and their order are those of
// build_guide_row_host), in table row M.guide_base + s.
__device__ __forceinline__ void guide_row(const Model& M, int s, int m, ThrPair* __restrict__ thr,
                                          uint8_t* __restrict__ guide) {
    __shared__ int64_t s_up[kBinomTable + 1];
    const int srow = M.guide_base + s;
    const int lane = int(threadIdx.x);
    const double pp = M.pp[s];
    const double q = M.qq[s];
    double qn;
    int32_t bound;
    inversion_constants(m, pp, q, M.lq[s], &qn, &bound);
    ThrPair* t = thr + guide_row_offset(srow, m);
    double carryP = 1.0, carryC = 0.0;
    int end = -1;
    bool covered = false;
    for (int c = 0; c * kWave < kBinomTable && end < 0; ++c) {
        const int k = c * kWave + lane;
        double P = k == 0 ? 1.0 : (double(m - k + 1) * pp) / (double(k) * q);
        for (int off = 1; off < kWave; off <<= 1) {
            const double o = __shfl_up(P, off);
            if (lane >= off) P = P * o;
        }
        const double Pf = P * carryP;
        double C = qn * Pf;
        for (int off = 1; off < kWave; off <<= 1) {
            const double o = __shfl_up(C, off);
            if (lane >= off) C = C + o;
        }
        const double Cf = C + carryC;
        const double cs = Cf * 0x1p53;
        const int64_t up = int64_t(floor(cs)) + kGuideBand + 1;
        const int64_t lo = int64_t(ceil(cs)) - kGuideBand - 1;
        const bool full = lo >= kU53Max;
        const uint64_t stop = __ballot(full || k >= bound);
        const int first = stop ? int(__builtin_ctzll(stop)) : kWave;
        if (lane <= first && lane < kWave) {
            t[k] = ThrPair{up, lo};
            s_up[k] = up;
        }
        if (stop) {
            end = c * kWave + first;
            covered = __shfl(full ? 1 : 0, first) != 0;
        }
        carryP = __shfl(Pf, kWave - 1);
        carryC = __shfl(Cf, kWave - 1);
    }
    if (lane == 0) t[end + 1] = ThrPair{INT64_MAX, covered ? INT64_MAX : int64_t(-1)};
    __syncthreads();
    // guide: entries with up <= j 2^47, by binary search over the row
    const int64_t u0 = int64_t(lane) << kGuideShift;
    int lo_i = 0, hi_i = end + 1;  // count in [lo_i, hi_i]
    while (lo_i < hi_i) {
        const int mid = (lo_i + hi_i) >> 1;
        if (s_up[mid] <= u0) lo_i = mid + 1;
        else hi_i = mid;
    }
    guide[(size_t(srow) * kBinomTable + size_t(m)) * kGuideBuckets + size_t(lane)] = uint8_t(lo_i);
}

// A slot's parameter set: its model tables into the slot's device copy, and
// its threshold rows (one workgroup each: state * kBinomTable + count) for the
// walks behind on the stream.  The model is an argument of the launch, which
// is taken when it is made: no staging buffer, no copy in front of it.  With
// the copy, and the rows' constants formed on the host (131,072 exponentials
// for a generation of 256 sets of 4 states), 5,000 bursts x 20 of 2 states took
// 69 us and that generation 12.5 ms; now 52 us and 10.9 ms.
__global__ __launch_bounds__(kWave) void model_kernel(const Model M, Model* __restrict__ model,
                                                      ThrPair* __restrict__ thr,
                                                      uint8_t* __restrict__ guide) {
    if (blockIdx.x == 0) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(&M);
        uint32_t* dst = reinterpret_cast<uint32_t*>(model);
        for (uint32_t i = threadIdx.x; i < sizeof(Model) / 4; i += kWave) dst[i] = src[i];
    }
    if (M.any_v) return;  // draws by the loop, no rows
    guide_row(M, int(blockIdx.x) / kBinomTable, int(blockIdx.x) % kBinomTable, thr, guide);
}

// The threshold rows of a population's sets: blockIdx.x as above, blockIdx.y
// the set.
__global__ __launch_bounds__(kWave) void guide_kernel(const Model* __restrict__ models,
                                                      ThrPair* __restrict__ thr,
                                                      uint8_t* __restrict__ guide) {
    const Model& M = models[blockIdx.y];
    const int s = int(blockIdx.x) / kBinomTable;
    if (s >= M.n) return;  // uniform over the workgroup
    guide_row(M, s, int(blockIdx.x) % kBinomTable, thr, guide);
}

// The inversion tables of a population's sets (kPassTable), one workgroup per
// set, a thread per count: build_binom_table's values.  (Formed on the host and
// copied with every set_population, 49 MB for 4,000 sets, they took 28.5 ms of
// a generation of 500 bursts x 4; here 2.4.)
__global__ __launch_bounds__(kBinomTable) void table_kernel(const Model* __restrict__ models,
                                                            BinomTable* __restrict__ tabs) {
    const Model& M = models[blockIdx.x];
    BinomTable& T = tabs[blockIdx.x];
    const int m = int(threadIdx.x);
    for (int s = 0; s < M.n; ++s)
        inversion_constants(m, M.pp[s], M.qq[s], M.lq[s], &T.qn[s][m], &T.bound[s][m]);
}

// ---- population runs ---------------------------------------------------------
//
// A population of parameter sets (an optimiser generation) over the same
// resident bursts in one launch sequence: fast_walk_kernel walks every
// (set, burst, resample) unit, pop_replay_kernel recomputes the units it
// abandoned (where they are more than the list holds, pop_walk_kernel walks
// all of them again), pop_finish_kernel computes each set's histogram and
// chi2.  The reference evaluates one set per stream and per mc::run_kernel
// call (src/gpuWorker.cpp:71-80); the units and their random streams are the
// same as a single-set run with set id set_base + s * set_stride.

// The general form over every (set, unit) of a population whose replay list
// overflowed; work and sets as in fast_walk_kernel.
__global__ __launch_bounds__(kWave) void pop_walk_kernel(
    const BurstDesc* __restrict__ bursts, const uint32_t* __restrict__ ticks,
    const uint2* __restrict__ links, const PopControl* __restrict__ ctl,
    const Model* __restrict__ models, const RunArgs a, int32_t* __restrict__ hist_acc,
    uint32_t* __restrict__ work) {
    __shared__ Model sM[2];
    extern __shared__ int32_t s_hist[];  // [2][a.B]
    const uint32_t lane = threadIdx.x;
    for (uint32_t i = lane; i < 2u * uint32_t(a.B); i += kWave) s_hist[i] = 0;
    __syncthreads();

    const uint32_t seed = ctl->seed, set_base = ctl->set_base, set_stride = ctl->set_stride;
    const uint32_t queue = blockIdx.x % a.queues;
    const uint32_t batches = a.nsets * a.bps;
    const uint32_t xrow = blockIdx.x & 7u;
    int set0 = -1, set1 = -1;    // wave-uniform: the set each LDS slot holds
    uint32_t cur = 0;            // slot that receives new units
    uint32_t pool_set = 0, pool_next = 0, pool_end = 0;
    bool busy = false;
    uint32_t my_slot = 0;
    WalkState<false> st{};
    UnitKey key{seed, 0u, 0u, 0u};
    BurstDesc d{0u, 0u, 0u, 0.0f};
    const UnitDiv divR{a.div_m, a.div_sh};
    bool drained = false;
    while (true) {
        bool need = !busy;
        while (!drained) {
            const uint64_t want = __ballot(need);
            if (want == 0) break;
            if (pool_next >= pool_end) {
                uint32_t k = 0;
                if (lane == 0) k = atomicAdd(&work[queue * kCounterStride], 1u);
                k = __shfl(k, 0);
                k = k * a.queues + queue;
                if (k >= batches) {
                    drained = true;
                    break;
                }
                pool_set = k / a.bps;
                pool_next = (k - pool_set * a.bps) * a.batch;
                pool_end = pool_next + a.batch < a.nunits ? pool_next + a.batch : a.nunits;
            }
            if (int(pool_set) != (cur ? set1 : set0)) {
                const uint32_t other = cur ^ 1u;
                if (__any(busy && my_slot == other)) break;  // the older set is still walking
                const int old = other ? set1 : set0;
                if (old >= 0)
                    flush_hist(s_hist + other * uint32_t(a.B),
                               hist_acc + (size_t(old) * 8u + xrow) * size_t(a.B), a.B, lane);
                const uint32_t* src = reinterpret_cast<const uint32_t*>(&models[pool_set]);
                uint32_t* dst = reinterpret_cast<uint32_t*>(&sM[other]);
                for (uint32_t i = lane; i < sizeof(Model) / 4; i += kWave) dst[i] = src[i];
                __syncthreads();
                if (other) set1 = int(pool_set);
                else set0 = int(pool_set);
                cur = other;
            }
            const uint32_t rank = lanes_below(want);
            const uint32_t avail = pool_end - pool_next;
            if (need && rank < avail) {
                const uint32_t u = pool_next + rank;
                my_slot = cur;
                const uint32_t bl = unit_div(u, divR);
                const uint32_t b = a.begin + bl;
                d = bursts[b];
                key.set = set_base + pool_set * set_stride;
                key.r = u - bl * a.R;
                key.b = b;
                if (begin_unit<false>(sM[my_slot], key, d.P, d.T, st) == kStepMore) {
                    busy = true;
                    need = false;
                } else {
                    tally(s_hist + my_slot * uint32_t(a.B), a.B, 0.0f, 0.0f);
                }
            }
            const uint32_t taken = uint32_t(__popcll(want));
            pool_next += taken < avail ? taken : avail;
        }
        if (!__any(busy)) break;
        if (busy) {
            const int r = general_window(sM[my_slot], key, d.P, d.stop_rel, d.T,
                                         ticks + d.off, links + d.off, a, st);
            if (r != kStepMore) {
                tally(s_hist + my_slot * uint32_t(a.B), a.B, st.acc, st.F);
                busy = false;
            }
        }
    }
    __syncthreads();
    if (set0 >= 0)
        flush_hist(s_hist, hist_acc + (size_t(set0) * 8u + xrow) * size_t(a.B), a.B, lane);
    if (set1 >= 0)
        flush_hist(s_hist + uint32_t(a.B), hist_acc + (size_t(set1) * 8u + xrow) * size_t(a.B),
                   a.B, lane);
}

// Recomputes abandoned (set, unit) pairs in the general form, one per lane,
// and adds them to row 0 of the set's accumulator.
__global__ __launch_bounds__(kWave) void pop_replay_kernel(
    const BurstDesc* __restrict__ bursts, const uint32_t* __restrict__ ticks,
    const uint2* __restrict__ links, const PopControl* __restrict__ ctl,
    const Model* __restrict__ models, const RunArgs a, int32_t* __restrict__ hist_acc,
    const uint64_t* __restrict__ replay, const uint32_t* __restrict__ replay_count) {
    const uint32_t count = *replay_count;
    if (count > a.replay_cap) return;  // the run is repeated as a whole
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const uint64_t e = replay[i];
        const uint32_t set = uint32_t(e >> 32), u = uint32_t(e);
        const uint32_t bl = u / a.R;
        const uint32_t b = a.begin + bl;
        const BurstDesc d = bursts[b];
        const UnitKey key{ctl->seed, ctl->set_base + set * ctl->set_stride, u - bl * a.R, b};
        const WalkOut o = walk_unit<false>(models[set], nullptr, key, d.P, d.stop_rel, d.T,
                                           ticks + d.off, links + d.off, a);
        tally(hist_acc + size_t(set) * 8u * size_t(a.B), a.B, o.acc, o.F);
    }
}

// One workgroup per set: reduces the set's 8 accumulator rows (leaving them
// zero), computes its chi2 as finish_run does, with the set's own degrees
// of freedom; workgroup 0 reports and resets the replay count and the work
// counters.
__global__ __launch_bounds__(kWave) void pop_finish_kernel(
    const Model* __restrict__ models, const RunArgs a, const float* __restrict__ obs,
    int32_t* __restrict__ hist_acc, uint32_t* __restrict__ replay_count,
    uint32_t* __restrict__ work, PopStatus* __restrict__ status, SetResult* __restrict__ results,
    int32_t* __restrict__ hists) {
    const uint32_t set = blockIdx.x, lane = threadIdx.x;
    const size_t B = size_t(a.B);
    const Chi2Sum c = chi2_fold(a, obs, hist_acc + size_t(set) * 8u * B, B,
                                hists + size_t(set) * B, lane);
    if (lane == 0) {
        const int n = models[set].n;
        const int dof = c.filled - n * (n + 1);
        SetResult r;
        r.chi2_ref = c.c32 / float(dof);
        r.chi2_64 = c.c64 / double(dof);
        r.effN = c.filled;
        r.n = n;
        r.pad = 0;
        results[set] = r;
    }
    if (set == 0) {
        if (lane == 0) {
            const uint32_t n = *replay_count;
            *replay_count = 0u;
            PopStatus st;
            st.replays = n;
            st.overflow = n > a.replay_cap ? 1u : 0u;
            st.pad[0] = st.pad[1] = 0;
            *status = st;
        }
        for (uint32_t q = lane; q < kMaxQueues; q += kWave) work[q * kCounterStride] = 0u;
    }
}

// Evaluates shared-library primitives for the bit-exactness tests.
struct BinomItem {
    int32_t n;
    uint32_t pad0;
    double p;
    uint32_t seed, set, r, b, w, hi, lo, pad1;
};
struct BgItem {
    float lam, cap, u1, u2;
    uint32_t seed, set, r, b, w, sub;
};

__global__ void primitive_kernel(int op, const void* __restrict__ in, void* __restrict__ out,
                                 int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    switch (op) {
        case 0: {
            const uint32_t* q = static_cast<const uint32_t*>(in) + 6 * i;
            const Block x = philox10(q[0], q[1], q[2], q[3], q[4], q[5]);
            uint32_t* o = static_cast<uint32_t*>(out) + 4 * i;
            o[0] = x.w[0]; o[1] = x.w[1]; o[2] = x.w[2]; o[3] = x.w[3];
            break;
        }
        case 1: static_cast<float*>(out)[i] = flog(static_cast<const float*>(in)[i]); break;
        case 2: static_cast<float*>(out)[i] = fexp(static_cast<const float*>(in)[i]); break;
        case 3: static_cast<double*>(out)[i] = dlog(static_cast<const double*>(in)[i]); break;
        case 4: static_cast<double*>(out)[i] = dexp(static_cast<const double*>(in)[i]); break;
        case 5: static_cast<float*>(out)[i] = cos_turns(static_cast<const float*>(in)[i]); break;
        case 6: {
            const uint32_t* q = static_cast<const uint32_t*>(in) + 2 * i;
            static_cast<float*>(out)[i] = gauss(q[0], q[1]);
            break;
        }
        case 7: {
            const BinomItem it = static_cast<const BinomItem*>(in)[i];
            const UnitKey key{it.seed, it.set, it.r, it.b};
            static_cast<int64_t*>(out)[i] = binomial(it.n, it.p, it.hi, it.lo, key, it.w);
            break;
        }
        case 8: {
            const BgItem it = static_cast<const BgItem*>(in)[i];
            const UnitKey key{it.seed, it.set, it.r, it.b};
            static_cast<float*>(out)[i] =
                background_count(it.lam, it.cap, it.u1, it.u2, key, it.w, it.sub);
            break;
        }
        case 9: static_cast<uint32_t*>(out)[i] = static_cast<const uint32_t*>(in)[i]; break;
        case 10: static_cast<float*>(out)[i] = flog_uniform24(static_cast<const uint32_t*>(in)[i]); break;
        case 11: static_cast<float*>(out)[i] = fexp_minus(static_cast<const float*>(in)[i]); break;
        case 12: {
            const float* q = static_cast<const float*>(in) + 2 * i;
            static_cast<float*>(out)[i] = quotient(q[0], q[1], 1.0f / q[1]);
            break;
        }
        case 13: {
            const uint32_t* q = static_cast<const uint32_t*>(in) + 2 * i;
            static_cast<float*>(out)[i] = gauss_uniform24(q[0], q[1]);
            break;
        }
        case 14: {
            const float* q = static_cast<const float*>(in) + 2 * i;
            static_cast<float*>(out)[i] = distance_efficiency_quick(q[0], q[1], 1.0f / q[1]);
            break;
        }
        case 15: {
            const BinomItem it = static_cast<const BinomItem*>(in)[i];
            static_cast<int64_t*>(out)[i] = binomial_broad(it.n, float(it.p), it.hi, it.lo);
            break;
        }
        case 16: static_cast<double*>(out)[i] = reciprocal_close(static_cast<const double*>(in)[i]); break;
        default: break;
    }
}

// ---- microbenchmarks of the algorithm's events ---------------------------------
//
// The weights of the algorithmic cost model: each lane repeats one event of
// the walk -- a Philox block, the scalar work of a dwell window, a
// binary-search step, a background draw, a capped-Poisson iteration, a
// binomial draw, a binomial inversion iteration, the per-unit start and
// tally -- with a loop-carried dependence, counts the events it performed
// and writes a checksum.  Launched with 256-thread workgroups at full
// occupancy, the loops are bound by VALU issue, so the time per event times
// the device's 32-bit lane-operation rate is the event's weight in
// lane-issue-cycles.  Inputs vary with a 32-bit LCG step per event (part of
// the measured cost, standing in for reading a Philox word).
enum MicroOp : int {
    kMbPhilox = 0,   // one Philox4x32-10 block
    kMbWindow = 1,   // a dwell window's scalar work (next state, dwell, window end,
                     // corrected count, its rounding and sums)
    kMbSearch = 2,   // one step of the window-end binary search (LDS-resident ticks,
                     // whole 7-step searches)
    kMbPoisson = 3,  // one capped-Poisson draw (and its inversion iterations)
    kMbBinom = 4,    // one binomial inversion draw from the q^m table (and its
                     // iterations)
    kMbUnit = 5,     // a unit's initial state draw and its tally into the histogram
    kMbOutcome = 6,  // one outcome of the Rao-Blackwellised spread: the bin of E = a / F
                     // and the 2^-32 fixed-point weight of its probability
};
constexpr int kMicroOps = 7;
constexpr uint32_t kMbThreads = 256;

__device__ __forceinline__ uint32_t lcg(uint32_t x) { return x * 1664525u + 1013904223u; }

template <int kOp>
__global__ __launch_bounds__(kMbThreads) void microbench_kernel(int iters, float param,
                                                                const double* __restrict__ qn,
                                                                const int32_t* __restrict__ bound,
                                                                uint64_t* __restrict__ out) {
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t h = gid * 0x9E3779B9u + 0x7F4A7C15u;
    uint64_t events = 0, inner = 0;
    __shared__ uint32_t s_tick[128];
    __shared__ int32_t s_hist[kMbThreads];
    if (kOp == kMbSearch || kOp == kMbUnit) {
        for (uint32_t i = threadIdx.x; i < 128u; i += blockDim.x) s_tick[i] = i * 97u;
        for (uint32_t i = threadIdx.x; i < kMbThreads; i += blockDim.x) s_hist[i] = 0;
        __syncthreads();
    }
    if (kOp == kMbPhilox) {
        // every counter and key word changes per block (no part of the
        // rounds can be hoisted out of the loop)
        Block x{{h, gid, 0u, 0u}};
        for (int i = 0; i < iters; ++i)
            x = philox10(uint32_t(i) ^ x.w[3], x.w[0], gid ^ x.w[2], x.w[1], h ^ uint32_t(i),
                         x.w[2] ^ x.w[3]);
        h = x.w[0] ^ x.w[1] ^ x.w[2] ^ x.w[3];
        events = uint64_t(iters);
    } else if (kOp == kMbWindow) {
        const float cum[2] = {0.4f, 1.0f};
        const float krate[3] = {900.0f, 3000.0f, 5500.0f};
        const float T = 1e-3f, clk = 12.5e-9f, gmx = 0.95f, omdd = 1.0f;
        float tsum = 0.0f, F = 0.0f, acc = 0.0f;
        uint32_t w0 = 0;
        int st = 0;
        for (int i = 0; i < iters; ++i) {
            h = lcg(h);
            const int jj = first_above(cum, 2, uniform24(h));
            const int j = jj >= st ? jj + 1 : jj;
            h = lcg(h);
            const float kk = j == 0 ? krate[0] : (j == 1 ? krate[1] : krate[2]);
            const float tau = flog(uniform24(h)) / (-kk);
            tsum = tsum + tau;
            const bool end = !(tsum < T);
            const float wf = float(w0) + tsum / clk;
            const uint32_t w1 = end ? 80000u : uint32_t(wf);
            const uint32_t cnt = (w1 - w0) & 31u;
            const float nd = (h & 1u) ? float(cnt) : 0.0f;
            const float na = (h & 1u) ? 0.0f : float(cnt);
            const float fv = gmx * nd + omdd * na;
            const float m = floorf(fv + 0.5f);
            F += fv;
            acc += m;
            w0 = end ? 0u : w1;
            tsum = end ? 0.0f : tsum;
            st = j;
        }
        h ^= fbits(F) ^ fbits(acc);
        events = uint64_t(iters);
    } else if (kOp == kMbSearch) {
        // whole lower_bound searches over 127 ticks (7 steps each), a new
        // key per search
        uint32_t acc = 0;
        for (int i = 0; i < iters; ++i) {
            h = lcg(h);
            const uint32_t key = h & 0x3FFFu;
            uint32_t lo = 0, hi = 127;
#pragma unroll
            for (int k = 0; k < 7; ++k) {
                const uint32_t mid = (lo + hi) >> 1;
                if (s_tick[mid] < key) lo = mid + 1u;
                else hi = mid;
            }
            acc += lo;
        }
        h ^= acc;
        events = uint64_t(iters) * 7u;
    } else if (kOp == kMbPoisson) {
        uint64_t it = 0;
        for (int i = 0; i < iters; ++i) {
            h = lcg(h);
            const float u1 = uniform24(h);
            h = lcg(h);
            const float k = background_single(param, 1e6f, u1, uniform24(h));
            it += uint64_t(k);
            h ^= fbits(k);
        }
        events = uint64_t(iters);
        inner = it;
    } else if (kOp == kMbBinom) {
        const int n = int(param);
        const double pp = 0.3, q = 0.7;
        uint64_t it = 0;
        for (int i = 0; i < iters; ++i) {
            h = lcg(h);
            const uint32_t lo32 = h;
            h = lcg(h);
            // the inversion of binomial_table (pda_walk.h) on a q^m table
            double px = qn[n];
            const int bnd = bound[n];
            double U = uniform53(h, lo32);
            int X = 0;
            while (U > px) {
                ++X;
                if (X > bnd) break;
                U -= px;
                px = (double(n - X + 1) * pp * px) / (double(X) * q);
            }
            it += uint64_t(X);
            h ^= uint32_t(X);
        }
        events = uint64_t(iters);
        inner = it;
    } else if (kOp == kMbUnit) {
        const float p0cum[3] = {0.2f, 0.7f, 1.0f};
        float acc = 3.0f, F = 7.0f;
        for (int i = 0; i < iters; ++i) {
            h = lcg(h);
            const int s0 = first_above(p0cum, 3, uniform24(h));
            acc += float(s0);
            F += float(h & 7u);
            const float E = F > 0.0f ? acc / F : 0.0f;
            if (E >= 0.0f && E < 1.0f) {
                // the histogram update; one address per lane (how often lanes
                // collide on a bin depends on the data, not on the algorithm)
                const int bin = int(floor(double(E) * 50.0));
                if (bin < 50) atomicAdd(&s_hist[threadIdx.x], bin + 1);
            }
            acc = E * 3.0f;
        }
        h ^= fbits(acc);
        events = uint64_t(iters);
    } else if (kOp == kMbOutcome) {
        // rb_bin and rb_fixed of pda_rb.h on fresh (a, F, P) per event; the
        // sums carry the results out
        uint64_t fx = 0;
        int32_t bins = 0;
        for (int i = 0; i < iters; ++i) {
            h = lcg(h);
            const int a = int(h & 31u);
            const float F = 8.0f + float(h >> 27) + param;
            const float P = uniform24(h ^ 0x5bd1e995u);
            bins += rb_bin(a, F, 50);
            fx += rb_fixed(P);
        }
        h ^= uint32_t(fx) ^ uint32_t(fx >> 32) ^ uint32_t(bins);
        events = uint64_t(iters);
    }
    out[3u * gid] = h;
    out[3u * gid + 1u] = events;
    out[3u * gid + 2u] = inner;
}

// ---- launchers (called by the C-ABI layer) ---------------------------------

hipError_t walk_occupancy(int pass, int B, int* blocks_per_cu) {
    const size_t lds = sizeof(int32_t) * size_t(B);
    if (pass == kPassReplay)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, walk_kernel, kWave, lds);
    if (pass == kPassBroad)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(
            blocks_per_cu, fast_walk_kernel<false, kPassBroad, false>, kWave, lds);
    if (pass == kPassBroadAll)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(
            blocks_per_cu, fast_walk_kernel<false, kPassBroadAll, false>, kWave, lds);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        blocks_per_cu, fast_walk_kernel<false, kPassGuided, false>, kWave, lds);
}

template <bool kPop, int kPass, bool kSamples>
static void launch_fast(uint32_t grid, size_t lds, const FastIO& io, const RunArgs& a,
                        const FastArgs& fa, hipStream_t stream) {
    hipLaunchKernelGGL((fast_walk_kernel<kPop, kPass, kSamples>), dim3(grid), dim3(kWave), lds,
                       stream, io, a, fa);
}

hipError_t launch_walk(int pass, uint32_t grid, const BurstDesc* bursts, const WalkBurst* order,
                       const uint32_t* ticks,
                       const uint2* links, const Model* model, const BinomGuide& guide,
                       const RunArgs& a, const FastArgs& fa, int32_t* hist_acc, uint32_t* replay,
                       uint32_t* replay_count, uint32_t* work, float* outE, int32_t* outAcc,
                       float* outF, const float* obs, ResultHeader* result, RunTimes* times,
                       hipStream_t stream) {
    const size_t lds = sizeof(int32_t) * size_t(a.B);
    const FastIO io{order, ticks, links, model, nullptr, nullptr, guide, hist_acc, replay,
                    replay_count, work, outE, outAcc, outF, times};
    if (pass == kPassReplay)
        hipLaunchKernelGGL(walk_kernel, dim3(grid), dim3(kWave), lds, stream, bursts, ticks, links,
                           model, a, hist_acc, replay, replay_count, work, outE, outAcc, outF, obs,
                           result, times);
    else if (pass == kPassBroadAll && outE)
        launch_fast<false, kPassBroadAll, true>(grid, lds, io, a, fa, stream);
    else if (pass == kPassBroadAll)
        launch_fast<false, kPassBroadAll, false>(grid, lds, io, a, fa, stream);
    else if (pass == kPassBroad && outE)
        launch_fast<false, kPassBroad, true>(grid, lds, io, a, fa, stream);
    else if (pass == kPassBroad)
        launch_fast<false, kPassBroad, false>(grid, lds, io, a, fa, stream);
    else if (outE)
        launch_fast<false, kPassGuided, true>(grid, lds, io, a, fa, stream);
    else
        launch_fast<false, kPassGuided, false>(grid, lds, io, a, fa, stream);
    return hipGetLastError();
}

hipError_t launch_order(const BurstDesc* bursts, const uint32_t* idx, uint32_t n, WalkBurst* plain,
                        WalkBurst* order, hipStream_t stream) {
    hipLaunchKernelGGL(order_kernel, dim3((n + 255u) / 256u), dim3(256), 0, stream, bursts, idx, n,
                       plain, order);
    return hipGetLastError();
}

hipError_t launch_model(const Model& M, Model* model, ThrPair* thr, uint8_t* guide,
                        hipStream_t stream) {
    hipLaunchKernelGGL(model_kernel, dim3(M.any_v ? 1u : uint32_t(M.n) * kBinomTable), dim3(kWave),
                       0, stream, M, model, thr, guide);
    return hipGetLastError();
}

hipError_t launch_guide(const Model* models, int nsets, int max_states, ThrPair* thr,
                        uint8_t* guide, hipStream_t stream) {
    hipLaunchKernelGGL(guide_kernel, dim3(uint32_t(max_states) * kBinomTable, uint32_t(nsets)),
                       dim3(kWave), 0, stream, models, thr, guide);
    return hipGetLastError();
}

hipError_t launch_tables(const Model* models, int nsets, BinomTable* tabs, hipStream_t stream) {
    hipLaunchKernelGGL(table_kernel, dim3(uint32_t(nsets)), dim3(kBinomTable), 0, stream, models,
                       tabs);
    return hipGetLastError();
}

hipError_t pop_walk_occupancy(int pass, int B, int* blocks_per_cu) {
    const size_t lds = sizeof(int32_t) * 2u * size_t(B);
    if (pass == kPassGeneral)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, pop_walk_kernel, kWave,
                                                            lds);
    if (pass == kPassBroad)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(
            blocks_per_cu, fast_walk_kernel<true, kPassBroad, false>, kWave, lds);
    if (pass == kPassBroadAll)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(
            blocks_per_cu, fast_walk_kernel<true, kPassBroadAll, false>, kWave, lds);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        blocks_per_cu, fast_walk_kernel<true, kPassGuided, false>, kWave, lds);
}

hipError_t launch_pop_walk(int pass, uint32_t grid, const BurstDesc* bursts,
                           const WalkBurst* order, const uint32_t* ticks, const uint2* links, const PopControl* ctl,
                           const Model* models, const BinomTable* tabs,
                           const BinomGuide& guide, const RunArgs& a,
                           const FastArgs& fa, int32_t* hist_acc, uint64_t* replay,
                           uint32_t* replay_count, uint32_t* work, hipStream_t stream) {
    const size_t lds = sizeof(int32_t) * 2u * size_t(a.B);
    const FastIO io{order, ticks, links, models, tabs, ctl, guide, hist_acc, replay,
                    replay_count, work, nullptr, nullptr, nullptr, nullptr};
    if (pass == kPassGeneral)
        hipLaunchKernelGGL(pop_walk_kernel, dim3(grid), dim3(kWave), lds, stream, bursts, ticks,
                           links, ctl, models, a, hist_acc, work);
    else if (pass == kPassBroad)
        launch_fast<true, kPassBroad, false>(grid, lds, io, a, fa, stream);
    else if (pass == kPassBroadAll)
        launch_fast<true, kPassBroadAll, false>(grid, lds, io, a, fa, stream);
    else if (pass == kPassTable)
        launch_fast<true, kPassTable, false>(grid, lds, io, a, fa, stream);
    else
        launch_fast<true, kPassGuided, false>(grid, lds, io, a, fa, stream);
    return hipGetLastError();
}

hipError_t launch_pop_replay(const BurstDesc* bursts, const uint32_t* ticks, const uint2* links,
                             const PopControl* ctl, const Model* models, const RunArgs& a,
                             int32_t* hist_acc, const uint64_t* replay,
                             const uint32_t* replay_count, uint32_t grid, hipStream_t stream) {
    hipLaunchKernelGGL(pop_replay_kernel, dim3(grid), dim3(kWave), 0, stream, bursts, ticks,
                       links, ctl, models, a, hist_acc, replay, replay_count);
    return hipGetLastError();
}

hipError_t launch_pop_finish(const Model* models, const RunArgs& a, const float* obs,
                             int32_t* hist_acc, uint32_t* replay_count, uint32_t* work,
                             PopStatus* status, SetResult* results, int32_t* hists,
                             hipStream_t stream) {
    hipLaunchKernelGGL(pop_finish_kernel, dim3(a.nsets), dim3(kWave), 0, stream, models, a, obs,
                       hist_acc, replay_count, work, status, results, hists);
    return hipGetLastError();
}

hipError_t launch_primitive(int op, const void* in, void* out, int64_t n, hipStream_t stream) {
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(primitive_kernel, dim3(uint32_t(blocks)), dim3(256), 0, stream, op, in, out,
                       n);
    return hipGetLastError();
}

hipError_t microbench_shape(int op, uint32_t* grid, uint32_t* threads) {
    int per_cu = 0;
    hipError_t e = hipSuccess;
    switch (op) {
        case kMbPhilox: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbPhilox>, kMbThreads, 0); break;
        case kMbWindow: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbWindow>, kMbThreads, 0); break;
        case kMbSearch: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbSearch>, kMbThreads, 0); break;
        case kMbPoisson: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbPoisson>, kMbThreads, 0); break;
        case kMbBinom: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbBinom>, kMbThreads, 0); break;
        case kMbUnit: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbUnit>, kMbThreads, 0); break;
        case kMbOutcome: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, microbench_kernel<kMbOutcome>, kMbThreads, 0); break;
        default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess) return e;
    if (per_cu < 1) per_cu = 1;
    int dev = 0, cus = 0;
    e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    *grid = uint32_t(cus) * uint32_t(per_cu);
    *threads = kMbThreads;
    return hipSuccess;
}

hipError_t launch_microbench(int op, uint32_t grid, int iters, float param, const double* qn,
                             const int32_t* bound, uint64_t* out, hipStream_t stream) {
    const dim3 g(grid), b(kMbThreads);
    switch (op) {
        case kMbPhilox: hipLaunchKernelGGL(microbench_kernel<kMbPhilox>, g, b, 0, stream, iters, param, qn, bound, out); break;
        case kMbWindow: hipLaunchKernelGGL(microbench_kernel<kMbWindow>, g, b, 0, stream, iters, param, qn, bound, out); break;
        case kMbSearch: hipLaunchKernelGGL(microbench_kernel<kMbSearch>, g, b, 0, stream, iters, param, qn, bound, out); break;
        case kMbPoisson: hipLaunchKernelGGL(microbench_kernel<kMbPoisson>, g, b, 0, stream, iters, param, qn, bound, out); break;
        case kMbBinom: hipLaunchKernelGGL(microbench_kernel<kMbBinom>, g, b, 0, stream, iters, param, qn, bound, out); break;
        case kMbUnit: hipLaunchKernelGGL(microbench_kernel<kMbUnit>, g, b, 0, stream, iters, param, qn, bound, out); break;
        case kMbOutcome: hipLaunchKernelGGL(microbench_kernel<kMbOutcome>, g, b, 0, stream, iters, param, qn, bound, out); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace pda
