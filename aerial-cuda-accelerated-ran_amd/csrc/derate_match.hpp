// Host/device interface of the PUSCH de-rate-match kernel (derate_match.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "cuphy_hip.h"

namespace nrldpc {

// Device descriptor built by cuphySetupPuschRxRateMatch (the reference's
// puschRxRateMatchDescr, rate_matching.hpp:23-31).
struct rm_descriptor {
    const void* llr_in[MAX_N_TBS_SUPPORTED];  // input LLRs of scheduled TB slot i
    uint16_t sch_user_idxs[MAX_N_TBS_SUPPORTED];
    void** out;                               // HARQ buffer of each UE index
    const PerTbParams* tb_prms;               // device copy, indexed by UE index
    int descrambling_on;
};

// Kernel of a FP configuration (0: fp32->fp32, 1: fp16->fp32, 2: fp32->fp16,
// 3: fp16->fp16), with or without descrambling; nullptr otherwise.
void* rm_kernel(int fpconfig, bool descrambling);
void* rm_noop_kernel();

constexpr unsigned RM_BLOCK = 256;
// Descrambling sequence words per CB that fit in LDS (48 KB): E up to
// 32 * (RM_SEQ_WORDS - 1) = 393,184 rate-matched bits per CB (a CB's bits
// may start anywhere in a word).
constexpr int RM_SEQ_WORDS = 12288;
constexpr int RM_MAX_DESCR_E = 32 * (RM_SEQ_WORDS - 1);

// Dynamic LDS of a launch whose TBs have at most max_e[i] bits per CB: each
// CB's descrambling words and, up to RM_LDS_LIMIT bytes in all (the size a
// kernel gets without asking for more), its LLRs.  The kernel looks at the
// size its launch really has; with less it makes the sequence in parts, at
// least RM_SEQ_PART_WORDS words each.
constexpr int RM_LDS_LIMIT = 64 * 1024;
constexpr int RM_SEQ_PART_WORDS = 256;
int rm_lds_bytes(int fpconfig, const uint32_t* max_e, int n, bool descrambling);

// Whether a CB of E LLRs of `elem` bytes fits after seq_words words.
__host__ __device__ inline bool rm_staged_fits(int E, int elem, uint32_t seq_words, uint32_t lds_words)
{
    return (uint64_t)seq_words + ((uint64_t)(uint32_t)E * (uint32_t)elem + 3u) / 4u <= lds_words;
}

}  // namespace nrldpc
