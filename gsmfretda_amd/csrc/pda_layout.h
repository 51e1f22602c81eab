// pda_layout.h -- host-side construction of the resident device layout:
// burst re-encoding (src/loadHdf5.cpp:101-128 -> pda_types.h) and the model
// tables of one parameter set (src/eigenhelper.cpp:4-54, src/mc.cu:790-800).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "pda_types.h"

namespace pda {

// Photon channel of the reference's masks: bit 0 donor (mask_dd), bit 1
// acceptor (mask_ad) -- the photons burst_data encodes as "time or 0"
// (src/loadHdf5.cpp:120-121).
struct PhotonSrc {
    const int64_t* times;      // absolute ticks (or null: use ad/dd arrays)
    const uint8_t* mask_ad;
    const uint8_t* mask_dd;
    const int64_t* burst_ad;   // reference encoding (or null)
    const int64_t* burst_dd;
    uint32_t colour(int64_t i) const {
        if (times) return (mask_dd[i] ? 1u : 0u) | (mask_ad[i] ? 2u : 0u);
        return (burst_dd[i] != 0 ? 1u : 0u) | (burst_ad[i] != 0 ? 2u : 0u);
    }
    int64_t tick(int64_t i) const {
        if (times) return times[i];
        return burst_dd[i] != 0 ? burst_dd[i] : burst_ad[i];
    }
};


struct Photophysics {
    float gamma = 0.34f, dexdir = 0.08f, crosstalk = 0.07f, r0 = 52.0f;  // src/mc.cu:89-91
};

// What of the bursts takes a window's draws beyond the fast form's: of every
// kEvery-th photon of each burst, from its first, how much of a run -- the
// photons of one colour that a window starting there counts at most -- is to
// come.  (In a pass of its own over the links, 4.5 million photons took 6 ms.)
struct LongRuns {
    static constexpr uint32_t kEvery = 16;
    static constexpr uint32_t kMaxRun = 1u << 16;  // longer ones count as that
    int64_t starts = 0;                            // photons looked at
    // [0] donors, [1] acceptors: those with at least k photons to come
    std::vector<uint64_t> at_least[2];
    int64_t long_bursts = 0;  // bursts whose background mean may pass 64
};

// Validates the reference's burst arrays and re-encodes them.  Returns 0 or a
// negative PDA_E_* code with a message in err.  runs, where given, is empty on
// entry.
int encode_bursts(const int64_t* start, const int64_t* stop, const int64_t* istart,
                  const int32_t* phcount, int64_t nbursts, const PhotonSrc& src, int64_t nphotons,
                  const float* T, float clk_p, float bg_ad, float bg_dd,
                  std::vector<BurstDesc>& bursts, std::vector<uint32_t>& ticks,
                  std::vector<uint2>& links, std::string& err, LongRuns* runs = nullptr);

// Builds the kernel's model tables.  Returns 0 or PDA_E_ARG with err set.
int build_model(const Photophysics& ph, int n, const float* args, int nargs, Model& M,
                std::string& err);

// Whether a run of models with broadening over `range` of the nbursts bursts
// makes the draws beyond the fast form's in place (kPassBroadAll) rather than
// abandon their units (kPassBroad).
bool draws_in_place(const LongRuns& r, int64_t nbursts, int64_t nphotons, int64_t range,
                    const Photophysics& ph, bool bg_on, bool population);

// The bursts in the order in which a walk over all of them starts them: by
// falling duration (in 256 steps of the longest, a step's bursts in their order)
// within each of equal parts, four to a default queue's share.
std::vector<uint32_t> burst_order(const std::vector<BurstDesc>& bursts);
// Tabulated inversion constants for the fast walk (needs M from build_model).
void build_binom_table(const Model& M, BinomTable& T);

}  // namespace pda
