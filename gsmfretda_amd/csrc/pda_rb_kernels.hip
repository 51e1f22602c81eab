// pda_rb_kernels.hip -- gfx950 kernels of the Rao-Blackwellised (RB) PDA form.
//
//   rb_walk_kernel       the walk of every (burst, resample) unit with the
//                        keyed draws of the plain kernel (src/mc.cu:92-191)
//                        but no acceptor draw; per unit it stores the photon
//                        counts per state, F, and (for rate gradients) the
//                        score of the walk's draws, and lists the units whose
//                        acceptor total is too large for the memo; fast form,
//                        the rare units beyond it listed for
//   rb_replay_kernel     the general form over those units
//   rb_table_kernel      the binomial pmfs of every state, counts < 256
//   rb_memo_kernel       the pmf (a convolution of one binomial per state)
//                        of every count vector with a small acceptor total,
//                        a wave per few vectors, lanes over outcomes (the
//                        derivative passes' leave-one-trial-out pmfs are the
//                        pmfs of the vectors with one trial fewer)
//   rb_unit_kernel       every unit with a small total: its pmf from the
//                        memo spread into the E histogram as 2^-32 fixed
//                        point (forward), or the cotangent-weighted pmf and
//                        its derivatives (adjoint), or the derivatives of
//                        every bin (Jacobian); a lane per unit, the units of
//                        a tile sorted by length
//   rb_big_kernel        the same for the listed units, one wave per unit,
//                        lanes over acceptor totals, the pmf built in LDS
//   rb_score_mean_kernel per burst, the mean score of its R resamples
//   rb_finish_kernel     reduces the histogram rows, computes chi2 on the
//                        expected counts, resets the counters
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pda_math.h"
#include "pda_rb.h"
#include "pda_types.h"
#include "pda_walk.h"

namespace pda {

// A unit's pmf has Mt + 1 entries, Mt its acceptor total (the sum of its
// photon counts per state).  The pmfs of every count vector with
// Mt < kRbMemoCap are built once per forward (rb_memo_kernel) and the units
// look theirs up (rb_unit_kernel); the walk lists the units with larger
// totals for rb_big_kernel.  The mean Mt is about 6 on the 3-state
// workloads and 24 on the 4-state fast-dynamics one, where 97 % of the
// units have Mt < 48.
constexpr int kRbMemoWaves = 4;  // waves per workgroup of rb_memo_kernel
static_assert(kRbMemoCap <= kWave, "a memo pmf fits the lanes of a wave");
// rb_unit_kernel's work counters: the kAuxQueues lines after the walk's,
// workgroup g on counter g % kAuxQueues, each over a contiguous share of the
// units (one queue per XCD).
constexpr uint32_t kRbUnitCounter = kMaxQueues * kCounterStride;
// rb_big_kernel's LDS rows of the Jacobian hold the rates from column
// kRbMaxStates.
constexpr int kRbJacCols = kRbMaxStates + kRbMaxPairs;

constexpr int kRbFwd = 0, kRbGrad = 1, kRbJac = 2;

// Orders the LDS accesses of the wave's lanes: every lane's earlier LDS
// writes are visible to every lane's later LDS reads.  The lanes of a wave
// share data through LDS here without a workgroup barrier; the compiler
// treats each lane as a thread of its own and, without this fence, may keep
// a value a lane stored in a register instead of reading what another lane
// wrote over it, or move accesses across the exchange.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Lane l's value, in every lane.
__device__ __forceinline__ double lane_value(double v, int l) {
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(b), l);
    const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(b >> 32), l);
    return __longlong_as_double((long long)(uint64_t(hi) << 32 | lo));
}

// *dst = src by `threads` threads, this one being t.
template <class T>
__device__ __forceinline__ void store_words(T* dst, const T& src, uint32_t t, uint32_t threads) {
    const uint32_t* from = reinterpret_cast<const uint32_t*>(&src);
    uint32_t* to = reinterpret_cast<uint32_t*>(dst);
    for (uint32_t i = t; i < sizeof(T) / 4; i += threads) to[i] = from[i];
}

// Lanes of the mask below this one.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}

// What an RB walk accumulates over a unit's windows (kN states, known at
// compile time): the photon counts per state, in registers, and the score of
// the walk's draws per rate pair, in the lane's column of an LDS array,
//   d/dK(j', s) log[P(j | s) K(j, s) exp(-K(j, s) tau)]
//     = [j' = j] (2 / K(j, s) - tau) - 1 / sum_{j''} K(j'', s)
// summed over the windows in float, in the order of the oracle's
// restatement: per window, the taken pair's 2 / K - tau first, then
// 1 / sum K off every pair leaving the window's state.
template <int kN, bool kScores, int kStride>
struct RbAcc {
    static constexpr int kK = kN * (kN - 1);
    static constexpr bool kHasScores = kScores;
    uint32_t cnt[kN];
    float* S;  // the lane's scores, kStride apart

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int s = 0; s < kN; ++s) cnt[s] = 0u;
        if (kScores) {
#pragma unroll
            for (int i = 0; i < kK; ++i) S[i * kStride] = 0.0f;
        }
    }

    template <class R_t>
    __device__ __forceinline__ void absorb(const R_t& R, const WindowInfo& wi) {
        const uint32_t m = wi.m > 0 ? uint32_t(wi.m) : 0u;
#pragma unroll
        for (int s = 0; s < kN; ++s) cnt[s] += s == wi.s ? m : 0u;
        if (kScores) {
            const float v = R.two_over_k[wi.s][wi.j] - wi.tau;
            const float inv = R.inv_sum[wi.s];
            // the pairs leaving wi.s: rate_pair(kN, wi.s, to)
            float t[kN - 1];
#pragma unroll
            for (int k = 0; k < kN - 1; ++k) t[k] = S[out_pair(wi.s, k) * kStride];
#pragma unroll
            for (int k = 0; k < kN - 1; ++k) {
                const int to = k < wi.s ? k : k + 1;
                t[k] = to == wi.j ? t[k] + v : t[k];
                S[out_pair(wi.s, k) * kStride] = t[k] - inv;
            }
        }
    }

    // rate_pair(kN, s, to) of the k-th state `to` other than s
    __device__ __forceinline__ static int out_pair(int s, int k) {
        return k < s ? k * (kN - 1) + s - 1 : (k + 1) * (kN - 1) + s;
    }

    // rb_pack of the counts (states >= n hold 0)
    __device__ __forceinline__ uint2 packed() const {
        uint32_t c[kRbMaxStates] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int s = 0; s < kN; ++s) c[s] = cnt[s];
        return make_uint2((c[0] & 0xFFFFu) | (c[1] << 16), (c[2] & 0xFFFFu) | (c[3] << 16));
    }

    // Stores the unit: its packed counts, F and scores; a unit too long for
    // the memo joins the big list (total < kRbBigSplit, count big_count[0]) or the huge one (count
    // big_count[1]): one atomic per wave, list and call site, the lanes
    // storing now ranked among themselves.
    __device__ __forceinline__ void store(uint32_t unit, float F, uint32_t lane,
                                          uint2* __restrict__ cnt_out, float* __restrict__ F_out,
                                          float* __restrict__ S_out, uint32_t* __restrict__ big,
                                          uint32_t* __restrict__ huge,
                                          uint32_t* __restrict__ big_count) const {
        const uint2 c = packed();
        cnt_out[unit] = c;
        F_out[unit] = F;
        if (kScores) {
            // kK (2, 6 or 12) floats per unit, 8-byte aligned rows: as few
            // stores as there can be, each lane's going to a line of its own
            struct __attribute__((packed, aligned(8))) Quad {
                float v[4];
            };
            float* row = S_out + size_t(unit) * size_t(kK);
#pragma unroll
            for (int i = 0; i + 4 <= kK; i += 4)
                *reinterpret_cast<Quad*>(row + i) = Quad{{S[i * kStride], S[(i + 1) * kStride],
                                                          S[(i + 2) * kStride],
                                                          S[(i + 3) * kStride]}};
            if (kK % 4)
                *reinterpret_cast<float2*>(row + kK / 4 * 4) =
                    make_float2(S[(kK - 2) * kStride], S[(kK - 1) * kStride]);
        }
        const uint32_t mt = (c.x & 0xFFFFu) + (c.x >> 16) + (c.y & 0xFFFFu) + (c.y >> 16);
        append(mt >= uint32_t(kRbMemoCap) && mt < uint32_t(kRbBigSplit), unit, lane, big,
               &big_count[0]);
        append(mt >= uint32_t(kRbBigSplit), unit, lane, huge, &big_count[1]);
    }

    __device__ __forceinline__ static void append(bool take, uint32_t unit, uint32_t lane,
                                                  uint32_t* __restrict__ list,
                                                  uint32_t* __restrict__ count) {
        const uint64_t mk = __ballot(take);
        if (mk) {
            const int leader = __ffsll(static_cast<long long>(mk)) - 1;
            uint32_t base = 0;
            if (int(lane) == leader) base = atomicAdd(count, uint32_t(__popcll(mk)));
            base = __shfl(base, leader);
            if (take)
                list[base + __builtin_amdgcn_mbcnt_hi(uint32_t(mk >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(uint32_t(mk), 0u))] = unit;
        }
    }
};

// Units that rb_walk_kernel starts at a time: its LDS then stays within 5,120
// bytes, and 32 workgroups share a CU.
template <int kN>
constexpr uint32_t kRbWalkStart = kN > 3 ? 32u : 64u;

// A unit without a window: no counts, no scores.
template <class Acc>
__device__ __forceinline__ void zero_unit(uint32_t unit, uint2* __restrict__ cnt_out,
                                          float* __restrict__ F_out, float* __restrict__ S_out) {
    cnt_out[unit] = make_uint2(0u, 0u);
    F_out[unit] = 0.0f;
    if (Acc::kHasScores)
        for (int i = 0; i < Acc::kK; ++i) S_out[size_t(unit) * Acc::kK + i] = 0.0f;
}

// What absorb() reads of an RbModel.
struct RbScoreModel {
    float two_over_k[kRbMaxStates][kRbMaxStates];
    float inv_sum[kRbMaxStates];
};

// The walk of every unit in the fast form (32-bit window ends, background
// means <= 64: the plain walk's common case) with the work stealing of
// fast_walk_kernel; a unit that leaves the common case is listed for
// rb_replay_kernel, which walks it again from its start in the general form
// with the same keyed draws, so every unit's stored summary is the general
// form's.  As there, units are started into LDS many at a time.
//
// Bound by the memory its results go to (100,000 bursts x 64 of 3 states: 231
// MB of counts, F and scores, of which 400 MB arrive, lines being written back
// before the last of their five units ends; with the scores stored to one
// small region instead the walk takes 65 us less), VALU at 60 %.  Scores summed
// in LDS instead of registers: a window touches the n - 1 rates out of its
// state where the register form had to select among all n (n - 1), 594 VALU
// instructions against 835 and 59 registers against 71, so 8 waves on a SIMD.
// That run 324 -> 300 us, 4 states of fast dynamics 160 -> 157 us per set and
// derivative step.  (Ended units kept in LDS and stored 64 at a time: 315 us
// with 3 states, spills with 4.)
template <bool kScores, int kN>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(8))) void rb_walk_kernel(
    const WalkBurst* __restrict__ bursts, const uint32_t* __restrict__ ticks,
    const uint2* __restrict__ links, const Model* __restrict__ model,
    const RbModel* __restrict__ rbm, const RunArgs a, const FastArgs fa,
    uint2* __restrict__ cnt_out,
    float* __restrict__ F_out, float* __restrict__ S_out, uint32_t* __restrict__ work,
    uint32_t* __restrict__ big, uint32_t* __restrict__ huge, uint32_t* __restrict__ big_count,
    uint32_t* __restrict__ replay, uint32_t* __restrict__ replay_count) {
    using Acc = RbAcc<kN, kScores, kWave>;
    constexpr uint32_t kStart = kRbWalkStart<kN>;
    constexpr int kS = kScores ? Acc::kK : 1;
    __shared__ FastModel sM;
    __shared__ RbScoreModel sR;
    __shared__ StartedUnit s_start[kStart];   // units started and not yet taken
    __shared__ uint8_t s_state[kStart];       // their first states
    __shared__ float s_S[kS][kWave];          // the lanes' scores
    const uint32_t lane = threadIdx.x;
    {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(model);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&sM);
        for (uint32_t i = lane; i < sizeof(FastModel) / 4; i += kWave) dst[i] = src[i];
        const float* src2 = &rbm->two_over_k[0][0];
        float* dst2 = reinterpret_cast<float*>(&sR);
        static_assert(offsetof(RbModel, inv_sum) ==
                          offsetof(RbModel, two_over_k) + offsetof(RbScoreModel, inv_sum),
                      "the two lie together in both");
        for (uint32_t i = lane; i < sizeof(RbScoreModel) / 4; i += kWave) dst2[i] = src2[i];
    }
    __syncthreads();
    Acc acc;
    acc.S = &s_S[0][lane];

    const uint32_t queue = blockIdx.x % a.queues;
    const QueueRange q = queue_range(queue, a.q_share, a.nunits);
    uint32_t pool_next = 0, pool_end = 0;
    uint32_t started = 0, start_next = 0;  // entries of s_start, the next to take
    bool busy = false;
    WalkState<true> st{};
    UnitKey key{a.seed, a.set, 0u, 0u};
    BurstDesc d{0u, 0u, 0u, 0.0f};
    const UnitDiv divR{a.div_m, a.div_sh};
    bool drained = false;
    while (true) {
        while (true) {
            const uint64_t want = __ballot(!busy);
            if (want == 0) break;
            if (start_next == started) {  // start the next units
                if (pool_next >= pool_end) {
                    if (drained) break;
                    uint32_t k = 0;
                    if (lane == 0) k = atomicAdd(&work[queue * kCounterStride], a.batch);
                    k = __builtin_amdgcn_readfirstlane(k);
                    if (k >= q.end - q.begin) {
                        drained = true;
                        break;
                    }
                    pool_next = q.begin + k;
                    pool_end = q.end - pool_next < a.batch ? q.end : pool_next + a.batch;
                }
                const uint32_t v = pool_next + lane;
                bool walks = false;
                int state = 0;
                StartedUnit e;
                if (lane < kStart && v < pool_end) {
                    const uint32_t i = unit_div(v, divR);
                    e.d = bursts[a.begin + i].d;
                    e.b = bursts[a.begin + i].b;
                    e.r = v - i * a.R;
                    const UnitKey k{a.seed, a.set, e.r, e.b};
                    WalkState<true> s0;
                    walks = begin_unit<true>(sM, k, e.d.P, e.d.T, s0) == kStepMore;
                    state = s0.s;
                    if (!walks) {
                        zero_unit<Acc>((e.b - a.begin) * a.R + e.r, cnt_out, F_out, S_out);
                    }
                }
                pool_next = pool_end - pool_next < kStart ? pool_end : pool_next + kStart;
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
                st = WalkState<true>{};
                st.s = s_state[start_next + rank];
                acc.clear();
                busy = true;
            }
            const uint32_t taken = uint32_t(__popcll(want));
            start_next += taken < left ? taken : left;
        }
        if (!__any(busy)) break;
        if (busy) {
            WindowInfo wi;
            const uint32_t u = (key.b - a.begin) * a.R + key.r;
            const int r = fast_window<true, BinomGuide>(sM, nullptr, key, d.P, d.stop_rel, d.T,
                                                        ticks + d.off, links + d.off, a, fa, st,
                                                        &wi);
            if (r == kStepReplay) {
                replay[atomicAdd(replay_count, 1u)] = u;
                busy = false;
            } else {
                acc.absorb(sR, wi);
                if (r != kStepMore) {
                    acc.store(u, st.F, lane, cnt_out, F_out, S_out, big, huge, big_count);
                    busy = false;
                }
            }
        }
    }
}

// The units rb_walk_kernel listed, in the general form, one unit per lane
// over the list; workgroups beyond the list's need exit at once.  Launched
// after rb_walk_kernel on the same stream.
template <bool kScores, int kN>
__global__ __launch_bounds__(kWave) void rb_replay_kernel(
    const BurstDesc* __restrict__ bursts, const uint32_t* __restrict__ ticks,
    const uint2* __restrict__ links, const Model* __restrict__ model,
    const RbModel* __restrict__ rbm, const RunArgs a, uint2* __restrict__ cnt_out,
    float* __restrict__ F_out, float* __restrict__ S_out, uint32_t* __restrict__ big,
    uint32_t* __restrict__ huge, uint32_t* __restrict__ big_count,
    const uint32_t* __restrict__ replay, const uint32_t* __restrict__ replay_count) {
    const uint32_t count = *replay_count;
    if (blockIdx.x * kWave >= count) return;  // uniform over the workgroup
    __shared__ Model sM;
    __shared__ RbModel sR;
    __shared__ float s_S[kScores ? kN * (kN - 1) : 1][kWave];
    const uint32_t lane = threadIdx.x;
    {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(model);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&sM);
        for (uint32_t i = lane; i < sizeof(Model) / 4; i += kWave) dst[i] = src[i];
        const uint32_t* src2 = reinterpret_cast<const uint32_t*>(rbm);
        uint32_t* dst2 = reinterpret_cast<uint32_t*>(&sR);
        for (uint32_t i = lane; i < sizeof(RbModel) / 4; i += kWave) dst2[i] = src2[i];
    }
    __syncthreads();
    const uint32_t first = blockIdx.x * kWave;
    const uint32_t stride = gridDim.x * kWave;
    for (uint32_t base = first; base < count; base += stride) {
        const uint32_t i = base + lane;
        if (i < count) {
            const uint32_t u = replay[i];
            const uint32_t bl = u / a.R;
            const uint32_t b = a.begin + bl;
            const BurstDesc d = bursts[b];
            const UnitKey key{a.seed, a.set, u - bl * a.R, b};
            WalkState<false> st{};
            RbAcc<kN, kScores, kWave> acc;
            acc.S = &s_S[0][lane];
            acc.clear();
            int r = begin_unit<false>(sM, key, d.P, d.T, st);
            while (r == kStepMore) {
                WindowInfo wi;
                r = general_window<true>(sM, key, d.P, d.stop_rel, d.T, ticks + d.off,
                                         links + d.off, a, st, &wi);
                acc.absorb(sR, wi);
            }
            acc.store(u, st.F, lane, cnt_out, F_out, S_out, big, huge, big_count);
        }
    }
}

// Sum over the wave (every lane gets the total, the same on every run).
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Inclusive prefix sum over the lanes of the wave.
__device__ __forceinline__ int wave_scan_sum(int v, int lane) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int t = __shfl_up(v, d);
        if (lane >= d) v += t;
    }
    return v;
}

// What the passes compute per unit, with P(a), a = 0..Mt, the unit's pmf
// and bin(a) the histogram bin of E = a / F:
//
// Forward: P(a) into the bin of a, in 2^-32 fixed point (integer sums: the
// result does not depend on the order in which units or outcomes arrive).
//
// Adjoint, for a cotangent G over the bins: h = sum_a G(bin(a)) P(a) and,
// per state s with m_s photons,
//   d h / d p_s = m_s sum_c P_s(c) (G(bin(c + 1)) - G(bin(c)))
// where P_s is the pmf with one trial of state s removed,
// P(a) = q_s P_s(a) + p_s P_s(a - 1): for a memo unit the memo's pmf of its
// count vector with m_s - 1 (built by the same convolutions); rb_big_kernel
// gets it from P by a first-order recurrence, upwards when p_s <= 1/2 and
// downwards otherwise (the direction in which it damps rounding errors).
// The rate gradient is the likelihood
// ratio R / (R - 1) sum_units h (S - Sbar), S the unit's score and Sbar the
// mean score of its burst's R resamples: the per-burst leave-one-out
// baseline, sum_r h_r S_r - (sum_r h_r)(sum_r S_r) / R, summed per unit.
//
// Jacobian: the adjoint for every indicator cotangent G_b(a) = [bin(a) = b]
// at once.  G_b(c + 1) - G_b(c) is nonzero only where c and c + 1 fall in
// different bins, so d M_b / d p_s gathers m_s P_s(c) at the unit's bin
// boundaries; the rate columns add P(a) (S - Sbar) to the row of bin(a).

// The memo: the pmf of every count vector of the list's items into poolP.
// (The derivative passes' leave-one-out pmfs are the pmfs of the vectors with
// one trial fewer, in the same pool.)  An item is the counts of all states but
// the last and a run of counts of the last (kRbMemoRun at most); a wave takes
// it, lane q holding outcome q (Mt < 48 outcomes fit a wave).  The states'
// binomials are convolved in state order, each output summed k ascending from
// 0.0f, as the oracle does: z += Y[k] X[q - k], X moving up one lane per step,
// the lanes below getting 0.  Outcomes outside the overlap add an exact 0, so
// the result is the oracle's bit for bit; a count of 0 leaves X as it is (its
// binomial is [1]).  Y's index is the same for all lanes: its loads are scalar.
// Three instructions a step and no LDS.  With a lane per vector, each walking
// its own chain of convolutions in a strip of LDS (31 KB a wave: five waves a
// CU), the 249,900 vectors of four states took 411 us, longer than the walk
// they are built beside, and the 19,600 of three 101 us; like this 135 and
// 14 us beside the walk.  The prefix is convolved again for each run:
// about a tenth of the steps, and every wave independent of every other.
typedef float Floats4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float Floats8 __attribute__((ext_vector_type(8), aligned(4)));
static_assert(kRbMemoCap + 8 < kRbPmfTable, "rows of the pmf table follow the memo's");

template <int kN>
__global__ __launch_bounds__(kWave * kRbMemoWaves) void rb_memo_kernel(
    const float* __restrict__ pmf_tab, const uint4* __restrict__ items, uint32_t nitems,
    const uint32_t* __restrict__ rank_offP, float* __restrict__ poolP) {
    const int q = int(threadIdx.x) % kWave;
    const uint32_t i = blockIdx.x * uint32_t(kRbMemoWaves) +
                       uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave));
    if (i >= nitems) return;  // uniform over the wave; no barrier below
    const uint4 e = items[i];
    const uint2 c = make_uint2(uint32_t(__builtin_amdgcn_readfirstlane(int(e.x))),
                               uint32_t(__builtin_amdgcn_readfirstlane(int(e.y))));
    const int first = __builtin_amdgcn_readfirstlane(int(e.z));
    const int runs = __builtin_amdgcn_readfirstlane(int(e.w));
    // X (*) Binomial(m, p_s)
    auto convolve = [&](float X, int s, int m) {
        const float* Y = pmf_tab + size_t(s) * kRbPmfStride + m * (m + 1) / 2;
        float z = 0.0f;
        for (int k0 = 0; k0 <= m; k0 += 8) {  // entries past m: the next rows', taken as 0
            const Floats8 y = *reinterpret_cast<const Floats8*>(Y + k0);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                z = z + (k0 + k <= m ? y[k] : 0.0f) * X;
                X = bitsf(uint32_t(__builtin_amdgcn_update_dpp(0, int(fbits(X)), 0x138, 0xf, 0xf,
                                                               true)));  // wave_shr:1
            }
        }
        return z;
    };
    float X = q == 0 ? 1.0f : 0.0f;
    int mm[kRbMaxStates] = {0, 0, 0, 0};
    int total = 0;
#pragma unroll
    for (int s = 0; s < kN - 1; ++s) {
        mm[s] = int(rb_count(c, s));
        total += mm[s];
        if (mm[s] > 0) X = convolve(X, s, mm[s]);
    }
    for (int m = first; m < first + runs; ++m) {
        const float z = m > 0 ? convolve(X, kN - 1, m) : X;
        mm[kN - 1] = m;
        const uint32_t off = rank_offP[rb_rank(mm, kN, kRbMemoCap - 1)];
        if (q <= total + m) poolP[off + uint32_t(q)] = z;
    }
}

// ---- units with a small acceptor total ---------------------------------------
//
// rb_unit_kernel takes every unit with Mt < kRbMemoCap, a lane per unit.  A
// workgroup takes a tile of consecutive units, sorts them by Mt in LDS
// (counting sort, longest first), and its waves take 64 of the sorted units at
// a time, all lanes looping over their unit's outcomes a = 0..Mt together:
// sorted, the lanes' loops are nearly of one length.  What belongs to a unit
// (F and its reciprocal, the memo offsets, the scores, the sums over its
// outcomes) stays in the lane's registers.  The pmfs of the smallest totals
// (the pool's first floats) are kept in LDS, where 64 lanes read 64 blocks at
// once; longer units read the pool in memory.
//   forward: P(a) into the bin of a, 2^-32 fixed point;
//   adjoint: h and sum_c P_s(c) dG(c) of the unit in registers, the unit's
//     scores once per unit;
//   Jacobian: the outcome's n efficiency terms, as m_s (P_s(a - 1) - P_s(a))
//     at the bin of a (the bin boundaries' terms gathered by bin), and its
//     n (n - 1) rate terms, into the bin's row.
// The histogram and the rows are LDS accumulators with atomics.  The lanes of
// a group tend to the same bins (outcome 0 is bin 0 for all), so there are
// `copies` of each accumulator, lane l using copy l % copies, copies adjacent:
// lanes on different copies never meet in a bank.
// Spreading the concatenated outcomes of 64 units over the lanes instead
// (each lane finding its outcome's unit by a search over the lanes and
// fetching the unit's data by shuffles, about 25 LDS instructions per 64
// outcomes besides the atomics), every wave adding its sums to one line in
// memory at the end, took, at 3 states, 100,000 bursts x 64, 139 us forward,
// 667 adjoint and 579 Jacobian; like this it takes 77, 152 and 215.  The
// adjoint and the Jacobian of 4 states of fast dynamics, 50,000 x 8: 491 and
// 123 -> 68 and 83 us.
constexpr int kRbUnitPer = 4;  // units per thread of a full tile

// Totals whose pmfs a workgroup keeps in LDS (the pool begins with them), and
// their floats: sum over t < totals of C(t + n - 1, n - 1) (t + 1).
__host__ __device__ constexpr int rb_lds_totals(int n) { return n == 2 ? 24 : n == 3 ? 14 : 10; }
// Three more, for the reads of four that begin in the last block.
__host__ __device__ constexpr int rb_lds_floats(int n) {
    return (n == 2 ? 4900 : n == 3 ? 6020 : 5863) + 3;
}
// Accumulators of a workgroup per copy, in 8-byte entries: the forward's bins;
// the Jacobian's rows of n efficiency and n (n - 1) rate columns, where its
// lanes are turned (kTurn) an odd number of entries apart.  (The adjoint's
// cotangent is not an accumulator: one copy, and a 0 for the outcomes outside
// the histogram.)
__host__ __device__ constexpr int rb_jac_stride(int n, bool turn) {
    return turn ? n * n | 1 : n * n;
}
__host__ __device__ inline int rb_unit_acc(int B, int mode, int n, bool turn) {
    return mode == kRbJac ? B * rb_jac_stride(n, turn) : mode == kRbGrad ? B + 1 : B;
}
// Dynamic LDS: the accumulators, the pool's first floats, the tile's order
// and its 64 counters (one per total, one for the group to take next).
__host__ __device__ inline size_t rb_unit_lds(int B, int mode, int n, bool turn, int copies,
                                              int threads, bool pool) {
    return sizeof(double) * size_t(rb_unit_acc(B, mode, n, turn)) * size_t(copies) +
           (pool ? sizeof(float) * size_t(rb_lds_floats(n)) : 0) +
           sizeof(uint16_t) * size_t(threads) * kRbUnitPer + sizeof(uint32_t) * 64u;
}

// What one unit pass reads and writes, and its shape.
struct RbUnitArgs {
    const uint2* cnt;
    const float* F;
    const float* S;
    const double* Sbar;
    const double* g;
    const uint32_t* rank_offP;
    const uint4* rank_offD;
    const float* poolP;
    unsigned long long* hist_acc;
    double* grad;
    uint32_t* work;
    int32_t copies;  // accumulator copies, a power of two
    int32_t tile;    // units a workgroup takes at a time
    int32_t pool;    // the pool's first floats are kept in LDS
    RunTimes* times;  // forward: where the walk's end goes, or null
};

// Entry j becomes entry (j + turn) & 3, turn 0 .. 3.
__device__ __forceinline__ void turn_by(float (&v)[4], int turn) {
    const bool one = turn & 1, two = turn & 2;
    const float a = one ? v[1] : v[0], b = one ? v[2] : v[1], c = one ? v[3] : v[2],
                d = one ? v[0] : v[3];
    v[0] = two ? c : a;
    v[1] = two ? d : b;
    v[2] = two ? a : c;
    v[3] = two ? b : d;
}

// rb_bin() for F in quotient_range and its reciprocal rF rounded to float; B
// for outcomes outside the histogram.  floor(E B) from the float product: one
// too much where the product rounded up to the next integer, which the sign
// of the exact remainder tells.
__device__ __forceinline__ int rb_bin_quick(int a, float F, float rF, float Bf, int B) {
    const float E = quotient(float(a), F, rF);
    float b = floorf(E * Bf);
    b = fmaf(E, Bf, -b) < 0.0f ? b - 1.0f : b;
    return E < 1.0f ? int(b) : B;
}

constexpr int rb_unit_threads_of(int mode) { return mode == kRbJac ? 1024 : 256; }

// kTurn (Jacobian): the lanes of a wave go through their outcomes from different
// places, see pass_shape.
template <int kMode, int kN, bool kTurn>
__global__ __launch_bounds__(rb_unit_threads_of(kMode)) void rb_unit_kernel(const RunArgs a,
                                                                            const RbUnitArgs p) {
    constexpr bool kDeriv = kMode != kRbFwd;
    constexpr int K = kN * (kN - 1), kCols = kN * kN, kStride = rb_jac_stride(kN, kTurn);
    constexpr int kThreads = rb_unit_threads_of(kMode);
    extern __shared__ __align__(16) double s_acc[];
    const int tid = int(threadIdx.x), lane = tid % kWave;
    if (kMode == kRbFwd && p.times && blockIdx.x == 0 && tid == 0) stamp(&p.times->walked);
    const int B = a.B;
    const int nacc = rb_unit_acc(B, kMode, kN, kTurn) * p.copies;
    float* s_pool = reinterpret_cast<float*>(s_acc + nacc);
    uint16_t* s_order = reinterpret_cast<uint16_t*>(s_pool + (p.pool ? rb_lds_floats(kN) : 0));
    uint32_t* s_count = reinterpret_cast<uint32_t*>(s_order + kThreads * kRbUnitPer);
    unsigned long long* s_h = reinterpret_cast<unsigned long long*>(s_acc);
    for (int i = tid; i < nacc; i += kThreads) {
        if (kMode == kRbGrad) s_acc[i] = i < B ? p.g[i] : 0.0;
        else s_h[i] = 0ull;
    }
    if (p.pool)
        for (int i = tid; i < rb_lds_floats(kN); i += kThreads) s_pool[i] = p.poolP[i];
    const int copy = lane & (p.copies - 1);
    const float Bf = float(B);
    const UnitDiv divR{a.div_m, a.div_sh};

    const uint32_t nq = gridDim.x < kAuxQueues ? gridDim.x : kAuxQueues;
    const uint32_t queue = blockIdx.x % nq;
    const uint32_t q_begin = uint32_t(uint64_t(a.nunits) * queue / nq);
    const uint32_t q_len = uint32_t(uint64_t(a.nunits) * (queue + 1u) / nq) - q_begin;
    uint32_t* counter = &p.work[kRbUnitCounter + queue * kCounterStride];
    double gp[kN] = {};       // adjoint: d h / d p_s over the lane's units
    double gk[K] = {};        // adjoint: h (S - Sbar) over the lane's units
    unsigned long long acc0 = 0;  // forward: the units' outcomes 0 (bin 0)
    while (true) {
        __syncthreads();  // the last tile's order and counters are free
        if (tid < 64) s_count[tid] = 0u;
        if (tid == 63) s_count[63] = atomicAdd(counter, uint32_t(p.tile));
        __syncthreads();
        const uint32_t off = s_count[63];
        if (off >= q_len) break;
        const uint32_t base = q_begin + off;
        const uint32_t len = q_len - off < uint32_t(p.tile) ? q_len - off : uint32_t(p.tile);
        // counting sort by total, the longest first; units with Mt >=
        // kRbMemoCap are left out (the walk listed them for rb_big_kernel)
        uint32_t key[kRbUnitPer], rank[kRbUnitPer];
#pragma unroll
        for (int j = 0; j < kRbUnitPer; ++j) {
            const uint32_t i = uint32_t(tid + j * kThreads);
            key[j] = kRbMemoCap;
            if (i < len) {
                const uint2 c = p.cnt[base + i];
                const uint32_t mt = (c.x & 0xFFFFu) + (c.x >> 16) + (c.y & 0xFFFFu) + (c.y >> 16);
                if (mt < uint32_t(kRbMemoCap)) key[j] = uint32_t(kRbMemoCap) - 1u - mt;
            }
            rank[j] = key[j] < uint32_t(kRbMemoCap) ? atomicAdd(&s_count[key[j]], 1u) : 0u;
        }
        __syncthreads();
        if (tid < kWave) {
            const uint32_t v = lane < kRbMemoCap ? s_count[lane] : 0u;
            const uint32_t incl = uint32_t(wave_scan_sum(int(v), lane));
            s_count[lane] = lane <= kRbMemoCap ? incl - v : 0u;  // [kRbMemoCap]: how many
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kRbUnitPer; ++j)
            if (key[j] < uint32_t(kRbMemoCap))
                s_order[s_count[key[j]] + rank[j]] = uint16_t(tid + j * kThreads);
        const uint32_t count = s_count[kRbMemoCap];
        __syncthreads();

        while (true) {
            uint32_t first = 0;
            if (lane == 0) first = atomicAdd(&s_count[62], uint32_t(kWave));
            first = uint32_t(__builtin_amdgcn_readfirstlane(int(first)));
            if (first >= count) break;
            const bool valid = first + uint32_t(lane) < count;
            const uint32_t u = base + s_order[valid ? first + uint32_t(lane) : first];
            const uint2 c = p.cnt[u];
            const float F = p.F[u];
            int mm[kRbMaxStates] = {0, 0, 0, 0};
            int total = 0;
#pragma unroll
            for (int s = 0; s < kN; ++s) {
                mm[s] = int(rb_count(c, s));
                total += mm[s];
            }
            const int Mt = valid ? total : -1;
            const int longest = __builtin_amdgcn_readfirstlane(total);  // sorted
            const uint32_t rk = rb_rank(mm, kN, kRbMemoCap - 1);
            const uint32_t offP = p.rank_offP[rk];
            uint32_t offD[kN];  // the pmfs without a trial of state s (uncounted: any block)
            if (kDeriv) {
                const uint4 d = p.rank_offD[rk];
                int js = 0;
#pragma unroll
                for (int s = 0; s < kN; ++s) {
                    const bool counted = mm[s] > 0;
                    const uint32_t o = js == 0 ? d.x : js == 1 ? d.y : js == 2 ? d.z : d.w;
                    offD[s] = counted ? o : offP;
                    js += counted ? 1 : 0;
                }
            }
            double sc[kMode == kRbJac ? K : 1];  // Jacobian: S - Sbar
            const uint32_t bl = kDeriv ? unit_div(u, divR) : 0u;
            if (kMode == kRbJac) {
#pragma unroll
                for (int k = 0; k < K; ++k)
                    sc[k] = double(p.S[size_t(u) * size_t(K) + size_t(k)]) -
                            p.Sbar[size_t(bl) * size_t(K) + size_t(k)];
            }
            const bool in_range = quotient_range(F);
            const float rF = 1.0f / F;
            const bool quick = __all(in_range);  // F = 0, or far from 1: the plain quotient
            double h = 0.0, G_last = 0.0, hs[kN] = {};
            float pd_last[kN] = {};
            // four outcomes at a time; four(offset, v): entries offset ..
            // offset + 3.  Lanes past their unit's outcomes read on into the
            // blocks that follow.
            auto outcomes = [&](auto&& four) {
                const int turn = kTurn ? lane & 3 : 0;
                int at = kTurn ? (lane >> 2) % (longest / 4 + 1) * 4 : 0;
                for (int q0 = 0; q0 <= longest; q0 += 4) {
                    float P4[4], D4[kN][4], L4[kTurn ? kN : 1][4];
                    if (!kTurn) at = q0;
                    four(offP + uint32_t(at), P4);
                    if (kDeriv) {
#pragma unroll
                        for (int s = 0; s < kN; ++s) four(offD[s] + uint32_t(at), D4[s]);
                    }
                    if constexpr (kTurn) {
                        turn_by(P4, turn);
#pragma unroll
                        for (int s = 0; s < kN; ++s) {  // L4: the entries one before D4's
                            L4[s][0] = at > 0 ? p.poolP[offD[s] + uint32_t(at) - 1u] : 0.0f;
#pragma unroll
                            for (int j = 1; j < 4; ++j) L4[s][j] = D4[s][j - 1];
                            turn_by(D4[s], turn);
                            turn_by(L4[s], turn);
                        }
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int q = kTurn ? at + ((j + turn) & 3) : q0 + j;
                        const bool act = q <= Mt;
                        const float P = P4[j];
                        int b = 0;
                        if (quick) {
                            b = rb_bin_quick(q, F, rF, Bf, B);
                        } else {
                            b = rb_bin(q, F, B);
                            b = b < 0 ? B : b;
                        }
                        if constexpr (kMode == kRbFwd) {
                            const uint64_t w = act ? rb_fixed(P) : 0u;
                            if (q == 0) acc0 += w;  // E = 0: bin 0
                            else if (act && b < B)
                                atomicAdd(&s_h[b * p.copies + copy], (unsigned long long)w);
                        } else if constexpr (kMode == kRbGrad) {
                            // sum_c P_s(c) (G(bin(c + 1)) - G(bin(c))), c = q - 1
                            const double G = s_acc[b];
                            // (no difference before the first outcome: G alone
                            // may be beyond float)
                            const double dG = act && q > 0 ? double(float(G - G_last)) : 0.0;
                            h += G * double(act ? P : 0.0f);
                            G_last = G;
#pragma unroll
                            for (int s = 0; s < kN; ++s) {
                                hs[s] += double(pd_last[s]) * dG;
                                pd_last[s] = D4[s][j];
                            }
                        } else {
                            double e[kN];
#pragma unroll
                            for (int s = 0; s < kN; ++s) {
                                const float pd = q < Mt ? D4[s][j] : 0.0f;
                                const float before = kTurn ? L4[kTurn ? s : 0][j] : pd_last[s];
                                e[s] = double(mm[s]) * (double(before) - double(pd));
                                pd_last[s] = pd;
                            }
                            if (act && b < B) {
                                double* row = s_acc + size_t(b * kStride) * size_t(p.copies) + copy;
#pragma unroll
                                for (int s = 0; s < kN; ++s) atomicAdd(&row[s * p.copies], e[s]);
#pragma unroll
                                for (int k = 0; k < K; ++k)
                                    atomicAdd(&row[(kN + k) * p.copies], double(P) * sc[k]);
                            }
                        }
                    }
                    if (kTurn) at = at + 4 > longest ? 0 : at + 4;
                }
            };
            if (p.pool && longest < rb_lds_totals(kN))
                outcomes([&](uint32_t o, float* v) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = s_pool[o + uint32_t(j)];
                });
            else
                outcomes([&](uint32_t o, float* v) {
                    const Floats4 x = *reinterpret_cast<const Floats4*>(p.poolP + o);
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = x[j];
                });
            if (kMode == kRbGrad && valid) {
#pragma unroll
                for (int s = 0; s < kN; ++s) gp[s] += double(mm[s]) * hs[s];
#pragma unroll
                for (int k = 0; k < K; ++k)
                    gk[k] += h * (double(p.S[size_t(u) * size_t(K) + size_t(k)]) -
                                  p.Sbar[size_t(bl) * size_t(K) + size_t(k)]);
            }
        }
    }
    const double f = a.R > 1 ? double(a.R) / double(a.R - 1) : 0.0;
    if (kMode == kRbFwd) {
        atomicAdd(&s_h[copy], acc0);
        __syncthreads();
        unsigned long long* row = p.hist_acc + size_t(blockIdx.x & 7u) * kMaxBins;
        for (int i = tid; i < B; i += kThreads) {
            unsigned long long v = 0;
            for (int x = 0; x < p.copies; ++x) v += s_h[i * p.copies + x];
            if (v) atomicAdd(&row[i], v);
        }
    } else if (kMode == kRbGrad) {
        // the workgroup's sums, in the cotangent's place
        double* s_sum = reinterpret_cast<double*>(s_acc);
        __syncthreads();
        if (tid < kCols) s_sum[tid] = 0.0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kCols; ++i) {
            const double v = wave_sum(i < kN ? gp[i < kN ? i : 0] : f * gk[i < kN ? 0 : i - kN]);
            if (lane == 0) atomicAdd(&s_sum[i], v);
        }
        __syncthreads();
        double* row = p.grad + size_t(blockIdx.x % kRbGradRows) * kRbGradLen;
        if (tid < kCols) atomicAdd(&row[tid], s_sum[tid]);
    } else {
        // grad holds J[b][i], i < n + K (efficiencies, then rates in args
        // order), B rows of kRbGradLen, kRbJacRows times
        __syncthreads();
        double* J = p.grad + size_t(blockIdx.x % kRbJacRows) * size_t(B) * kRbGradLen;
        for (int i = tid; i < B * kCols; i += kThreads) {
            const int b = i / kCols, col = i - b * kCols;
            double v = 0.0;
            const double* from = s_acc + size_t(b * kStride + col) * size_t(p.copies);
            for (int x = 0; x < p.copies; ++x) v += from[x];
            if (col >= kN) v *= f;
            if (v != 0.0) atomicAdd(&J[size_t(b) * kRbGradLen + size_t(col)], v);
        }
    }
}

// Bytes of rb_big_kernel's dynamic LDS: B 8-byte entries (the forward's
// histogram, the adjoint's cotangent) or the Jacobian's [B][kRbJacCols]
// rows, then three pmf buffers (X, Y, Z) of cap floats.
__host__ __device__ inline size_t rb_big_lds(int B, int cap, int mode, bool wide) {
    const size_t head = size_t(mode == kRbJac ? B * kRbJacCols : B);
    return sizeof(double) * head +
           (mode != kRbFwd && wide ? sizeof(double) : sizeof(float)) * 3u * size_t(cap);
}

// The units the walk listed (Mt >= kRbMemoCap), one wave per unit, lanes
// over acceptor totals; cap = the largest Mt + 1 of the units of the list.
// The forward convolves in float, in the oracle's order (bit-exact).  The
// derivative passes take the leave-one-out pmfs from P by a recurrence
// whose factor has magnitude |alpha| = p / q (or q / p): it carries P's
// rounding errors, amplified up to 1 / (1 - |alpha|) -- 3x at p = 0.4, the
// length of the chain at p = 1/2, where a P rounded to float at every
// convolution step had put 1e-3 of an efficiency gradient off at
// Mt ~ 1,000.  kWide (sets with a state of 0.4 < p < 0.6): those passes
// convolve in double (from the same float binomial tables), at twice the
// LDS.
template <int kMode, bool kWide>
__global__ __launch_bounds__(kWave) void rb_big_kernel(
    const RbModel* __restrict__ rbm, const double* __restrict__ lf,
    const float* __restrict__ pmf_tab, const RunArgs a, const uint2* __restrict__ cnt_in,
    const float* __restrict__ F_in, const float* __restrict__ S_in,
    const double* __restrict__ Sbar, const double* __restrict__ g,
    const uint32_t* __restrict__ big, const uint32_t* __restrict__ big_count,
    unsigned long long* __restrict__ hist_acc, double* __restrict__ grad, int cap) {
    extern __shared__ double s_dyn[];
    __shared__ RbModel sR;
    const uint32_t lane = threadIdx.x;
    const int B = a.B;
    const uint32_t count = *big_count;
    if (blockIdx.x >= count) return;  // whole workgroup: no barrier below is skipped by part
    {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(rbm);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&sR);
        for (uint32_t i = lane; i < sizeof(RbModel) / 4; i += kWave) dst[i] = src[i];
    }
    const int head = kMode == kRbJac ? B * kRbJacCols : B;
    unsigned long long* s_h = reinterpret_cast<unsigned long long*>(s_dyn);
    double* s_d = s_dyn;
    using T = typename std::conditional<kMode != kRbFwd && kWide, double, float>::type;
    T* bufs = reinterpret_cast<T*>(s_dyn + head);
    for (int i = int(lane); i < head; i += kWave) {
        if (kMode == kRbGrad) s_d[i] = g[i];
        else if (kMode == kRbJac) s_d[i] = 0.0;
        else s_h[i] = 0ull;
    }
    __syncthreads();
    const int n = sR.n, K = sR.K;
    double gp_acc = 0.0, gk_acc = 0.0;  // adjoint: lane s holds d/dp_s, lane k d/dk_k
    for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
        const uint32_t u = big[i];
        const uint2 c = cnt_in[u];
        const float F = F_in[u];
        int bX = 0, bY = 1, bZ = 2;
        int xl = 1;
        if (lane == 0) bufs[0] = T(1);
#pragma unroll
        for (int s = 0; s < kRbMaxStates; ++s) {
            const int m = s < n ? int(rb_count(c, s)) : 0;
            T* Y = bufs + bY * cap;
            for (int k = int(lane); m > 0 && k <= m; k += kWave) {
                const double y = m < kRbPmfTable
                                     ? double(pmf_tab[rb_pmf_index(s, m, k)])
                                     : rb_binom_pmf(m, k, lf, sR.p[s], sR.lp[s], sR.lq[s]);
                Y[k] = kMode == kRbFwd ? T(float(y)) : T(y);
            }
            __syncthreads();
            if (m > 0) {
                if (xl == 1) {  // X = [1]: the product is Y itself, bit for bit
                    const int t = bX;
                    bX = bY;
                    bY = t;
                    xl = m + 1;
                } else {
                    const T* X = bufs + bX * cap;
                    T* Z = bufs + bZ * cap;
                    for (int q = int(lane); q < xl + m; q += kWave)
                        Z[q] = rb_conv_at(Y, m + 1, X, xl, q);
                    const int t = bX;
                    bX = bZ;
                    bZ = t;
                    xl += m;
                }
            }
            __syncthreads();
        }
        const T* P = bufs + bX * cap;
        if (kMode == kRbFwd) {
            for (int q = int(lane); q < xl; q += kWave) {
                const int bin = rb_bin(q, F, B);
                if (bin >= 0) atomicAdd(&s_h[bin], (unsigned long long)rb_fixed(P[q]));
            }
            __syncthreads();
            continue;
        }
        const int Mt = xl - 1;
        const uint32_t bl = u / a.R;
        double sc[kRbMaxPairs];  // Jacobian: the unit's score less its burst's mean
#pragma unroll
        for (int k = 0; k < kRbMaxPairs; ++k)
            sc[k] = kMode == kRbJac && k < K
                        ? double(S_in[size_t(u) * size_t(K) + size_t(k)]) -
                              Sbar[size_t(bl) * size_t(K) + size_t(k)]
                        : 0.0;
        T* dG = bufs + bY * cap;  // adjoint: G(bin(c + 1)) - G(bin(c)), rounded to float
        double hp = 0.0;
        for (int q = int(lane); q < xl; q += kWave) {
            const int b0 = rb_bin(q, F, B);
            if (kMode == kRbJac) {
                if (b0 >= 0) {
                    const double w = double(P[q]);
                    double* row = s_d + b0 * kRbJacCols + kRbMaxStates;
#pragma unroll
                    for (int k = 0; k < kRbMaxPairs; ++k)
                        if (k < K) atomicAdd(&row[k], w * sc[k]);
                }
                continue;
            }
            const double G0 = b0 >= 0 ? s_d[b0] : 0.0;
            hp += G0 * double(P[q]);
            if (q + 1 < xl) {
                const int b1 = rb_bin(q + 1, F, B);
                dG[q] = T(float((b1 >= 0 ? s_d[b1] : 0.0) - G0));
            }
        }
        __syncthreads();
        const double h = wave_sum(hp);
#pragma unroll
        for (int s = 0; s < kRbMaxStates; ++s) {
            const int m = s < n ? int(rb_count(c, s)) : 0;
            if (m == 0) continue;  // uniform over the wave
            const double p = double(sR.p[s]), q = 1.0 - p;
            const bool up = p <= 0.5;
            const double alpha = up ? -p / q : -q / p;
            const double inv = up ? 1.0 / q : 1.0 / p;
            double carry = 0.0, part = 0.0;
            for (int j0 = 0; j0 < Mt; j0 += kWave) {
                // lanes over 64 steps of the recurrence: a scan of the
                // affine maps x -> alpha x + P(.) inv
                const int j = j0 + int(lane);
                const bool v = j < Mt;
                double A = v ? alpha : 1.0;
                double Bv = v ? double(P[up ? j : Mt - j]) * inv : 0.0;
#pragma unroll
                for (int d = 1; d < kWave; d <<= 1) {
                    const double A2 = __shfl_up(A, d);
                    const double B2 = __shfl_up(Bv, d);
                    if (int(lane) >= d) {
                        Bv = A * B2 + Bv;
                        A = A * A2;
                    }
                }
                const double x = A * carry + Bv;  // P_s(up ? j : Mt - 1 - j)
                carry = __shfl(x, kWave - 1);
                const int ci = up ? j : Mt - 1 - j;
                if (kMode == kRbJac) {
                    const int b0 = rb_bin(ci, F, B), b1 = rb_bin(ci + 1, F, B);
                    if (v && b0 != b1) {
                        const double w = double(m) * x;
                        if (b1 >= 0) atomicAdd(&s_d[b1 * kRbJacCols + s], w);
                        if (b0 >= 0) atomicAdd(&s_d[b0 * kRbJacCols + s], -w);
                    }
                } else if (v) {
                    part += x * double(dG[ci]);
                }
            }
            if (kMode == kRbGrad) {
                part = wave_sum(part) * double(m);
                if (int(lane) == s) gp_acc += part;
            }
        }
        if (kMode == kRbGrad && int(lane) < K)
            gk_acc += h * (double(S_in[size_t(u) * size_t(K) + lane]) -
                           Sbar[size_t(bl) * size_t(K) + lane]);
        __syncthreads();
    }
    if (kMode == kRbFwd) {
        unsigned long long* row = hist_acc + size_t(blockIdx.x & 7u) * kMaxBins;
        for (int i = int(lane); i < B; i += kWave)
            if (s_h[i]) atomicAdd(&row[i], s_h[i]);
    } else if (kMode == kRbGrad) {
        const double f = a.R > 1 ? double(a.R) / double(a.R - 1) : 0.0;
        double* row = grad + size_t(blockIdx.x % kRbGradRows) * kRbGradLen;
        if (int(lane) < n) atomicAdd(&row[lane], gp_acc);
        if (int(lane) < K) atomicAdd(&row[n + int(lane)], f * gk_acc);
    } else {
        const double f = a.R > 1 ? double(a.R) / double(a.R - 1) : 0.0;
        const int w = n + K;
        double* J = grad + size_t(blockIdx.x % kRbJacRows) * size_t(B) * kRbGradLen;
        for (int i = int(lane); i < B * w; i += kWave) {
            const int b = i / w, col = i - b * w;
            const double v = col < n ? s_d[b * kRbJacCols + col]
                                     : f * s_d[b * kRbJacCols + kRbMaxStates + (col - n)];
            if (v != 0.0) atomicAdd(&J[size_t(b) * kRbGradLen + size_t(col)], v);
        }
    }
}

// Per burst bl and rate k: Sbar[bl K + k] = (1 / R) sum_r S[(bl R + r) K + k],
// summed r ascending in double.  A workgroup stages the scores of a run of
// whole bursts in LDS with coalesced loads, then one thread per (burst,
// rate) sums them; a burst whose R K scores exceed the stage is taken a part of
// its resamples at a time.  Bound by the scores' 154 MB (100,000 bursts x 64
// of 3 states): 33 us, 82 with single-float loads and half as many workgroups
// of twice the stage.  (Bursts beyond the stage had been summed straight from
// memory, a thread per burst and rate: 200 bursts x 1,000 of 3 states 182 us,
// now 21.)
constexpr uint32_t kRbSbarStage = 4096;  // floats
__global__ __launch_bounds__(256) void rb_score_mean_kernel(const RunArgs a, int K,
                                                            const float* __restrict__ S,
                                                            double* __restrict__ Sbar) {
    __shared__ __align__(8) float st[kRbSbarStage];
    const uint64_t nb = a.nunits / a.R;
    const uint32_t per = a.R * uint32_t(K);  // scores per burst
    // bursts at a time, or resamples of one burst
    const uint32_t bpb = per <= kRbSbarStage ? kRbSbarStage / per : 1u;
    const uint32_t rpb = per <= kRbSbarStage ? a.R : kRbSbarStage / uint32_t(K);
    for (uint64_t b0 = uint64_t(blockIdx.x) * bpb; b0 < nb; b0 += uint64_t(gridDim.x) * bpb) {
        const uint32_t nbh = uint32_t(nb - b0 < bpb ? nb - b0 : bpb);
        double part = 0.0;  // of thread k < K, where the burst is taken in parts
        for (uint32_t r0 = 0; r0 < a.R; r0 += rpb) {
            const uint32_t rh = a.R - r0 < rpb ? a.R - r0 : rpb;
            const uint32_t len = per <= kRbSbarStage ? nbh * per : rh * uint32_t(K);
            const float* src = S + b0 * per + uint64_t(r0) * uint64_t(K);
            __syncthreads();
            // K is even: whole pairs, 8-byte aligned
            const float2* src2 = reinterpret_cast<const float2*>(src);
            float2* st2 = reinterpret_cast<float2*>(st);
#pragma unroll 8
            for (uint32_t i = threadIdx.x; i < len / 2u; i += 256u) st2[i] = src2[i];
            __syncthreads();
            for (uint32_t t = threadIdx.x; t < nbh * uint32_t(K); t += blockDim.x) {
                const uint32_t bl = t / uint32_t(K), k = t - bl * uint32_t(K);
                const float* x = st + bl * per + k;
                double sum = part;
#pragma unroll 8
                for (uint32_t r = 0; r < rh; ++r) sum += double(x[r * uint32_t(K)]);
                if (r0 + rh == a.R) Sbar[(b0 + bl) * uint64_t(K) + k] = sum / double(a.R);
                else part = sum;
            }
        }
    }
}

// Start of a forward: the binomial pmfs of every state (blockIdx.y) for
// counts m < kRbPmfTable, one thread per entry, read by the pmf passes instead
// of recomputing them per unit; and from the first workgroup the run's device
// copies of its models and zeroed counters.  The models are arguments of the
// launch: no staging buffer whose reuse the host has to wait for, no copies
// and fills in front of the walk.  (With those, six small launches here and as
// many at the derivative passes' ends, 3 states of 100,000 bursts x 64 with
// their adjoint took 775 us; now 653.)
__global__ __launch_bounds__(256) void rb_table_kernel(
    const RbModel R, const Model M, RbModel* __restrict__ rbm, Model* __restrict__ model,
    const double* __restrict__ lf, float* __restrict__ pmf_tab, uint32_t* __restrict__ work,
    uint32_t* __restrict__ big_count, uint32_t* __restrict__ replay_count,
    RunTimes* __restrict__ times) {
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        const uint32_t t = threadIdx.x;
        if (times && t == 0u) stamp(&times->start);
        store_words(rbm, R, t, 256u);
        if (model) store_words(model, M, t, 256u);
        for (uint32_t i = t; i < kMaxQueues + kAuxQueues + 1u; i += 256u)
            work[i * kCounterStride] = 0u;
        if (t < 2u) big_count[t] = 0u;
        if (t == 0u) *replay_count = 0u;
    }
    const int r = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (r >= kRbPmfStride) return;
    const int s = int(blockIdx.y);
    // r = m (m + 1) / 2 + k with 0 <= k <= m
    int m = int((sqrt(8.0 * double(r) + 1.0) - 1.0) * 0.5);
    while (m * (m + 1) / 2 > r) --m;
    while ((m + 1) * (m + 2) / 2 <= r) ++m;
    const int k = r - m * (m + 1) / 2;
    pmf_tab[s * kRbPmfStride + r] = float(rb_binom_pmf(m, k, lf, R.p[s], R.lp[s], R.lq[s]));
}

// Start of a derivative pass: its accumulator rows and counters zero, and for
// the adjoint the cotangent from the host's buffer.
__global__ __launch_bounds__(256) void rb_begin_kernel(double* __restrict__ rows, uint32_t n,
                                                       uint32_t* __restrict__ work,
                                                       const double* __restrict__ g_host,
                                                       double* __restrict__ g, int B,
                                                       RunTimes* __restrict__ times) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (times && i == 0u) stamp(&times->start);
    if (i < n) rows[i] = 0.0;
    if (i < kMaxQueues + kAuxQueues + 1u) work[i * kCounterStride] = 0u;
    if (g_host && i < uint32_t(B)) g[i] = g_host[i];
}

// Sums the rows of a derivative pass: n sums of `rows` values `stride` apart, a
// group of kLanes lanes per sum.  The last workgroup stamps the end of the pass
// (a count of those that ended, for the very last one, took 5 us of a Jacobian
// of 1,000 bins).
template <int kLanes>
__global__ __launch_bounds__(256) void rb_rows_kernel(const double* __restrict__ rows_in, int n,
                                                      int rows, int stride,
                                                      double* __restrict__ out,
                                                      RunTimes* __restrict__ times) {
    const int t = int(blockIdx.x * blockDim.x + threadIdx.x);
    const int i = t / kLanes, l = t % kLanes;
    double v = 0.0;
    if (i < n)
        for (int r = l; r < rows; r += kLanes) v += rows_in[size_t(r) * size_t(stride) + size_t(i)];
#pragma unroll
    for (int o = kLanes / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (i < n && l == 0) out[i] = v;
    if (blockIdx.x != gridDim.x - 1u) return;
    __syncthreads();
    if (threadIdx.x == 0) stamp(&times->end);
}

// Device result of an RB run, followed by uint64 M[B] (2^-32 units).
struct RbResultHeader {
    double chi2;
    int32_t effN;
    int32_t B;
};

// One wave: sums the 8 rows (leaving them zero), chi2 of the expected
// counts M_b / R against the observed histogram with the reference's rules
// (src/streamWorker.cpp:197-206), into the host's result buffer.  Lane b forms
// bin b's term, 64 bins at a time, and the sum runs over the lanes; an empty
// bin's term is zero.
__global__ __launch_bounds__(kWave) void rb_finish_kernel(
    const RunArgs a, const float* __restrict__ obs, unsigned long long* __restrict__ hist_acc,
    RbResultHeader* __restrict__ res, RunTimes* __restrict__ times) {
    const uint32_t lane = threadIdx.x;
    unsigned long long* M = reinterpret_cast<unsigned long long*>(res + 1);
    double c = 0.0;
    int effN = 0;
    for (uint32_t base = 0; base < uint32_t(a.B); base += kWave) {
        const uint32_t b = base + lane;
        double t = 0.0;
        bool filled = false;
        if (b < uint32_t(a.B)) {
            unsigned long long x[8], v = 0;
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k)
                x[k] = __hip_atomic_load(&hist_acc[size_t(k) * kMaxBins + b], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                if (x[k]) hist_acc[size_t(k) * kMaxBins + b] = 0ull;
                v += x[k];
            }
            M[b] = v;
            filled = v > 0 && int(b) >= a.left_pad;
            if (filled) {
                const double m = double(v) * 0x1p-32 / double(a.R);
                const double dd = double(obs[b]) - m;
                t = dd * dd / m;
            }
        }
        effN += __popcll(__ballot(filled));
#pragma unroll 8
        for (int l = 0; l < kWave; ++l) c += lane_value(t, l);
    }
    if (lane == 0) {
        res->chi2 = c / double(effN - a.nstates * (a.nstates + 1));
        res->effN = effN;
        res->B = a.B;
        if (times) stamp(&times->end);
    }
}

hipError_t rb_walk_occupancy(bool scores, int n, int* per_cu) {
#define PDA_RB_OCC(SC, N) \
    hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_walk_kernel<SC, N>, kWave, 0)
    if (scores) return n == 2 ? PDA_RB_OCC(true, 2) : n == 3 ? PDA_RB_OCC(true, 3) : PDA_RB_OCC(true, 4);
    return n == 2 ? PDA_RB_OCC(false, 2) : n == 3 ? PDA_RB_OCC(false, 3) : PDA_RB_OCC(false, 4);
#undef PDA_RB_OCC
}

template <int kMode, bool kTurn>
static hipError_t rb_unit_occupancy_m(int n, size_t l, int* per_cu) {
    const int tu = rb_unit_threads_of(kMode);
    if (n == 2) return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_unit_kernel<kMode, 2, kTurn>, tu, l);
    if (n == 3) return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_unit_kernel<kMode, 3, kTurn>, tu, l);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_unit_kernel<kMode, 4, kTurn>, tu, l);
}

hipError_t rb_unit_occupancy(int mode, int n, bool turn, int dyn_lds, int* per_cu) {
    const size_t l = size_t(dyn_lds);
    if (mode == kRbGrad) return rb_unit_occupancy_m<kRbGrad, false>(n, l, per_cu);
    if (mode == kRbJac)
        return turn ? rb_unit_occupancy_m<kRbJac, true>(n, l, per_cu)
                    : rb_unit_occupancy_m<kRbJac, false>(n, l, per_cu);
    return rb_unit_occupancy_m<kRbFwd, false>(n, l, per_cu);
}

hipError_t rb_big_occupancy(int mode, bool wide, int dyn_lds, int* per_cu) {
    const size_t l = size_t(dyn_lds);
    if (mode == kRbGrad)
        return wide ? hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_big_kernel<kRbGrad, true>, kWave, l)
                    : hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_big_kernel<kRbGrad, false>, kWave, l);
    if (mode == kRbJac)
        return wide ? hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_big_kernel<kRbJac, true>, kWave, l)
                    : hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_big_kernel<kRbJac, false>, kWave, l);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rb_big_kernel<kRbFwd, false>, kWave, l);
}

template <bool kScores, int kN>
static void launch_rb_walk_n(uint32_t grid, uint32_t replay_grid, const BurstDesc* bursts,
                             const WalkBurst* order, const uint32_t* ticks, const uint2* links, const Model* model,
                             const RbModel* rbm, const RunArgs& a, const FastArgs& fa, uint2* cnt,
                             float* F, float* S, uint32_t* work, uint32_t* big, uint32_t* huge, uint32_t* big_count,
                             uint32_t* replay, uint32_t* replay_count, hipStream_t stream) {
    hipLaunchKernelGGL((rb_walk_kernel<kScores, kN>), dim3(grid), dim3(kWave), 0, stream, order,
                       ticks, links, model, rbm, a, fa, cnt, F, S, work, big, huge, big_count,
                       replay, replay_count);
    hipLaunchKernelGGL((rb_replay_kernel<kScores, kN>), dim3(replay_grid), dim3(kWave), 0, stream,
                       bursts, ticks, links, model, rbm, a, cnt, F, S, big, huge, big_count, replay,
                       replay_count);
}

hipError_t launch_rb_walk(bool scores, int n, uint32_t grid, uint32_t replay_grid,
                          const BurstDesc* bursts, const WalkBurst* order, const uint32_t* ticks,
                          const uint2* links, const Model* model, const RbModel* rbm,
                          const RunArgs& a, const FastArgs& fa, uint2* cnt, float* F, float* S, uint32_t* work,
                          uint32_t* big, uint32_t* huge, uint32_t* big_count,
                          uint32_t* replay, uint32_t* replay_count, hipStream_t stream) {
#define PDA_RB_WALK(SC, N)                                                                    \
    launch_rb_walk_n<SC, N>(grid, replay_grid, bursts, order, ticks, links, model, rbm, a, fa, \
                            cnt, F, S, work, big, huge, big_count, replay, replay_count, stream)
    if (n < 2 || n > kRbMaxStates) return hipErrorInvalidValue;
    if (scores) {
        if (n == 2) PDA_RB_WALK(true, 2);
        else if (n == 3) PDA_RB_WALK(true, 3);
        else PDA_RB_WALK(true, 4);
    } else {
        if (n == 2) PDA_RB_WALK(false, 2);
        else if (n == 3) PDA_RB_WALK(false, 3);
        else PDA_RB_WALK(false, 4);
    }
#undef PDA_RB_WALK
    return hipGetLastError();
}

int rb_unit_threads(int mode) { return rb_unit_threads_of(mode); }
size_t rb_unit_lds_bytes(int B, int mode, int n, bool turn, int copies, bool pool) {
    return rb_unit_lds(B, mode, n, turn, copies, rb_unit_threads_of(mode), pool);
}
size_t rb_big_lds_bytes(int B, int cap, int mode, bool wide) { return rb_big_lds(B, cap, mode, wide); }

hipError_t launch_rb_table(const RbModel& R, const Model& M, RbModel* rbm, Model* model,
                           const double* lf, float* pmf_tab, uint32_t* work, uint32_t* big_count,
                           uint32_t* replay_count, RunTimes* times, hipStream_t stream) {
    hipLaunchKernelGGL(rb_table_kernel, dim3(uint32_t((kRbPmfStride + 255) / 256), uint32_t(R.n)),
                       dim3(256), 0, stream, R, M, rbm, model, lf, pmf_tab, work, big_count,
                       replay_count, times);
    return hipGetLastError();
}

hipError_t launch_rb_begin(double* rows, uint32_t n, uint32_t* work, const double* g_host,
                           double* g, int B, RunTimes* times, hipStream_t stream) {
    const uint32_t most = std::max<uint32_t>(std::max<uint32_t>(n, uint32_t(B)),
                                             kMaxQueues + kAuxQueues + 1u);
    hipLaunchKernelGGL(rb_begin_kernel, dim3((most + 255u) / 256u), dim3(256), 0, stream, rows, n,
                       work, g_host, g, B, times);
    return hipGetLastError();
}

hipError_t launch_rb_memo(int n, const float* pmf_tab, const uint4* items, uint32_t nitems,
                          const uint32_t* rank_offP, float* poolP, hipStream_t stream) {
    const dim3 grid((nitems + kRbMemoWaves - 1) / kRbMemoWaves), threads(kWave * kRbMemoWaves);
    if (n == 2)
        hipLaunchKernelGGL(rb_memo_kernel<2>, grid, threads, 0, stream, pmf_tab, items, nitems,
                           rank_offP, poolP);
    else if (n == 3)
        hipLaunchKernelGGL(rb_memo_kernel<3>, grid, threads, 0, stream, pmf_tab, items, nitems,
                           rank_offP, poolP);
    else
        hipLaunchKernelGGL(rb_memo_kernel<4>, grid, threads, 0, stream, pmf_tab, items, nitems,
                           rank_offP, poolP);
    return hipGetLastError();
}

template <int kMode, int kN, bool kTurn>
static void launch_rb_unit_n(uint32_t grid, const RunArgs& a, const RbUnitArgs& p,
                             hipStream_t stream) {
    const int threads = rb_unit_threads_of(kMode);
    hipLaunchKernelGGL((rb_unit_kernel<kMode, kN, kTurn>), dim3(grid), dim3(uint32_t(threads)),
                       rb_unit_lds(a.B, kMode, kN, kTurn, p.copies, threads, p.pool != 0),
                       stream, a, p);
}

hipError_t launch_rb_unit(int mode, int n, uint32_t grid, int copies, bool turn, int tile,
                          bool pool, const RunArgs& a, const uint2* cnt, const float* F, const float* S,
                          const double* Sbar, const double* g, const uint32_t* rank_offP,
                          const uint4* rank_offD, const float* poolP,
                          unsigned long long* hist_acc, double* grad, uint32_t* work,
                          RunTimes* times, hipStream_t stream) {
    if (n < 2 || n > kRbMaxStates) return hipErrorInvalidValue;
    const RbUnitArgs p{cnt,      F,    S,    Sbar,   g,    rank_offP, rank_offD, poolP,
                       hist_acc, grad, work, copies, tile, pool ? 1 : 0, times};
#define PDA_RB_UNIT_M(M, T)                                         \
    if (n == 2) launch_rb_unit_n<M, 2, T>(grid, a, p, stream);      \
    else if (n == 3) launch_rb_unit_n<M, 3, T>(grid, a, p, stream); \
    else launch_rb_unit_n<M, 4, T>(grid, a, p, stream)
    if (mode == kRbGrad) {
        PDA_RB_UNIT_M(kRbGrad, false);
    } else if (mode == kRbJac && turn) {
        PDA_RB_UNIT_M(kRbJac, true);
    } else if (mode == kRbJac) {
        PDA_RB_UNIT_M(kRbJac, false);
    } else {
        PDA_RB_UNIT_M(kRbFwd, false);
    }
#undef PDA_RB_UNIT_M
    return hipGetLastError();
}

template <int kMode, bool kWide>
static void launch_rb_big_m(uint32_t grid, int cap, const RbModel* rbm, const double* lf,
                            const float* pmf_tab, const RunArgs& a, const uint2* cnt,
                            const float* F, const float* S, const double* Sbar, const double* g,
                            const uint32_t* big, const uint32_t* big_count,
                            unsigned long long* hist_acc, double* grad, hipStream_t stream) {
    hipLaunchKernelGGL((rb_big_kernel<kMode, kWide>), dim3(grid), dim3(kWave),
                       rb_big_lds(a.B, cap, kMode, kWide), stream, rbm, lf, pmf_tab, a, cnt, F, S,
                       Sbar, g, big, big_count, hist_acc, grad, cap);
}

hipError_t launch_rb_big(int mode, bool wide, uint32_t grid, int cap, const RbModel* rbm,
                         const double* lf, const float* pmf_tab, const RunArgs& a,
                         const uint2* cnt, const float* F, const float* S, const double* Sbar,
                         const double* g, const uint32_t* big, const uint32_t* big_count,
                         unsigned long long* hist_acc, double* grad, hipStream_t stream) {
#define PDA_RB_BIG(M, W)                                                                      \
    launch_rb_big_m<M, W>(grid, cap, rbm, lf, pmf_tab, a, cnt, F, S, Sbar, g, big, big_count, \
                          hist_acc, grad, stream)
    if (mode == kRbGrad) {
        if (wide) PDA_RB_BIG(kRbGrad, true);
        else PDA_RB_BIG(kRbGrad, false);
    } else if (mode == kRbJac) {
        if (wide) PDA_RB_BIG(kRbJac, true);
        else PDA_RB_BIG(kRbJac, false);
    } else {
        PDA_RB_BIG(kRbFwd, false);
    }
#undef PDA_RB_BIG
    return hipGetLastError();
}

hipError_t launch_rb_score_mean(const RunArgs& a, int K, const float* S, double* Sbar,
                                int num_cu, hipStream_t stream) {
    const uint64_t nb = a.nunits / a.R;
    const uint64_t per = uint64_t(a.R) * uint64_t(K);
    const uint64_t bpb = per <= kRbSbarStage ? kRbSbarStage / per : 1;
    const uint64_t want = (nb + bpb - 1) / bpb;
    // a few workgroups per CU, each looping over its share
    const uint64_t cap = uint64_t(num_cu > 0 ? num_cu : 1) * 8u;
    const uint32_t grid = uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(want, cap)));
    hipLaunchKernelGGL(rb_score_mean_kernel, dim3(grid), dim3(256), 0, stream, a, K, S, Sbar);
    return hipGetLastError();
}

hipError_t launch_rb_rows(const double* rows, int n, int nrows, double* out, RunTimes* times,
                          hipStream_t stream) {
    if (nrows >= kWave)
        hipLaunchKernelGGL(rb_rows_kernel<kWave>, dim3(uint32_t((n * kWave + 255) / 256)),
                           dim3(256), 0, stream, rows, n, nrows, n, out, times);
    else
        hipLaunchKernelGGL(rb_rows_kernel<8>, dim3(uint32_t((n * 8 + 255) / 256)), dim3(256), 0,
                           stream, rows, n, nrows, n, out, times);
    return hipGetLastError();
}

hipError_t launch_rb_finish(const RunArgs& a, const float* obs, unsigned long long* hist_acc,
                            void* res, RunTimes* times, hipStream_t stream) {
    hipLaunchKernelGGL(rb_finish_kernel, dim3(1), dim3(kWave), 0, stream, a, obs, hist_acc,
                       static_cast<RbResultHeader*>(res), times);
    return hipGetLastError();
}

}  // namespace pda
