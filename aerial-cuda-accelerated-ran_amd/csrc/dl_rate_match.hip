// DL rate matching of LDPC-encoded code blocks (TS 38.212 5.4.2) for gfx950:
// bit selection from k0 around the circular buffer of Ncb bits, skipping
// the filler bits, then bit interleaving, then (optionally) scrambling with
// the TS 38.211 7.3.1.1 Gold sequence of the TB's c_init.  The reference's
// PDSCH kernel (cuPHY/src/cuphy/dl_rate_matching/dl_rate_matching.cu:1951-2260)
// does the same with enable_layer_mapping = 0 and enable_modulation = 0 and
// writes CB r of TB t at bit (t * cmax + r) * emax of the output; so does
// this kernel.
//
// Output bit i of CB r (i < E_r) is bit (i mod Qm) of symbol i / Qm, i.e.
// selected bit m = (i mod Qm) * E_r / Qm + i / Qm; selected bit m sits at
// circle position c = (c0 + m) mod (Ncb - F) of the filler-free circular
// buffer, buffer position c < Kd ? c : c + F (the same closed form as the
// uplink de-rate-matcher).  Scrambling XORs c(start_r + i), start_r the
// CB's first bit in the TB.
//
// So the output interleaves Qm contiguous runs of the circular buffer.  A
// thread takes 32 symbols: 32 bits of each run (one funnel shift of two
// words read straight from the encoder's output: consecutive lanes read
// consecutive words, nothing is staged) and Qm output words, each a
// compile-time pattern of single-bit inserts.  One bit at a time, with a
// division, a modulo and an LDS read each, 2,800 code blocks of 9,088 bits
// (R = 0.93, 256QAM, scrambled) took 47 us (81 us with the earlier
// sequence generator); this takes 13 us, 6.4 MB in and out being 1.3 us: the
// sequence, the selection and one wave per code block bound it.
#include <hip/hip_runtime.h>

#include "derate_core.hpp"
#include "dl_rate_match.hpp"
#include "gold_core.hpp"

namespace nrldpc {

constexpr int DL_RM_MAX_N = 66 * 384;  // encoded bits of a BG1 Zc = 384 code block

// Where a code block's selected bits come from.
struct dl_source {
    const uint32_t* __restrict__ src;  // encoded bits
    int words, L, Kd, F;
};

// 32 selected bits from circle position c (< L) on, of which the first
// `want` (1 .. 32) are used.
__device__ __forceinline__ uint32_t circle_bits(const dl_source& s, int c, int want)
{
    uint32_t v = 0;
    for (int got = 0;;) {
        const bool head = c < s.Kd;
        const int p = head ? c : c + s.F, end = head ? min(s.Kd, s.L) : s.L;
        const int i = p >> 5;
        const uint32_t hi = (i + 1 < s.words) ? s.src[i + 1] : 0u;
        const uint32_t x = __builtin_amdgcn_alignbit(hi, s.src[i], (uint32_t)p & 31u);
        v |= (x & low_bits(end - c)) << got;
        got += end - c;
        if (got >= want) return v;
        c = (end == s.L) ? 0 : end;
    }
}

// Output words of a code block: thread t builds words QM * t .. QM * t + QM - 1.
template <int QM>
__device__ __forceinline__ void dl_words(const dl_source& s, const rm_geometry& g, const uint32_t* seq, int emax_words,
                                         uint32_t* __restrict__ dst)
{
    const uint32_t soff = (uint32_t)g.start & 31u;
    const int groups = (g.EQ + 31) >> 5;
    const int run_step = g.EQ % g.L;
    for (int t = threadIdx.x; t < groups; t += blockDim.x) {
        const int j0 = 32 * t, want = min(32, g.EQ - j0);
        uint32_t run[QM];
        int c = (g.c0 + j0) % g.L;
#pragma unroll
        for (int k = 0; k < QM; ++k) {
            run[k] = circle_bits(s, c, want);
            c += run_step;
            if (c >= g.L) c -= g.L;
        }
#pragma unroll
        for (int q = 0; q < QM; ++q) {
            const int at = QM * t + q;
            uint32_t w = 0;
#pragma unroll
            for (int b = 0; b < 32; ++b) w |= ((run[(32 * q + b) % QM] >> ((32 * q + b) / QM)) & 1u) << b;
            // (the word after the last with output bits exists too)
            if (seq && 32 * at < g.E) w ^= __builtin_amdgcn_alignbit(seq[at + 1], seq[at], soff);
            if (at < emax_words) dst[at] = w & low_bits(max(0, g.E - 32 * at));
        }
    }
    for (int w = QM * groups + (int)threadIdx.x; w < emax_words; w += blockDim.x) dst[w] = 0u;
}

__global__ __launch_bounds__(256) void dl_rate_match_kernel(const PerTbParams* __restrict__ prms,
                                                            const uint32_t* const* __restrict__ cw, int max_cbs,
                                                            int emax_words, int scrambling,
                                                            uint32_t* __restrict__ out)
{
    extern __shared__ uint32_t dl_seq[];  // scrambling words of the code block, one more than its E bits reach
    const int t = blockIdx.y, r = blockIdx.x;
    const PerTbParams& p = prms[t];
    const int C = __builtin_amdgcn_readfirstlane((int)p.num_CBs);
    if (r >= C || r >= max_cbs) return;
    const int Qm = __builtin_amdgcn_readfirstlane((int)p.Qm), Nl = __builtin_amdgcn_readfirstlane((int)p.Nl);
    const bool prm_ok = (Qm == 1 || Qm == 2 || Qm == 4 || Qm == 6 || Qm == 8) && Nl >= 1 && Nl <= 8;
    rm_geometry g{};
    if (prm_ok) {
        g = rm_geometry_of(p, r);
        rm_make_uniform(g);
    }
    const int N = __builtin_amdgcn_readfirstlane((int)p.N);
    uint32_t* dst = out + ((size_t)t * max_cbs + r) * emax_words;
    // a CB that does not fit its slot or the kernel's buffers stays zero
    const bool ok = prm_ok && g.E > 0 && g.E <= 32 * emax_words && g.Ncb <= N && N <= DL_RM_MAX_N && g.L > 0 &&
                    g.Kd >= 0 && g.c0 >= 0 && g.c0 < g.L;
    if (!ok) {
        for (int w = threadIdx.x; w < emax_words; w += blockDim.x) dst[w] = 0u;
        return;
    }
    const int words_in = (N + 31) >> 5;
    const dl_source s{cw[t] + (size_t)r * words_in, words_in, g.L, g.Kd, g.F};
    if (scrambling) {
        const uint32_t w_base = (uint32_t)g.start >> 5;
        const int nw = (int)(((uint32_t)(g.start + g.E - 1) >> 5) - w_base + 1u);
        if (threadIdx.x < 64) {
            gold_words_wave((uint32_t)__builtin_amdgcn_readfirstlane((int)p.cinit), w_base, nw, dl_seq);
            if (threadIdx.x == 0) dl_seq[nw] = 0u;
        }
        __syncthreads();
    }
    const uint32_t* seq = scrambling ? dl_seq : nullptr;
    switch (Qm) {  // (uniform)
    case 8: dl_words<8>(s, g, seq, emax_words, dst); break;
    case 6: dl_words<6>(s, g, seq, emax_words, dst); break;
    case 4: dl_words<4>(s, g, seq, emax_words, dst); break;
    case 2: dl_words<2>(s, g, seq, emax_words, dst); break;
    default: dl_words<1>(s, g, seq, emax_words, dst);
    }
}

cuphyStatus_t dl_rate_match(const PerTbParams* d_prms, int num_tbs, const uint32_t* const* d_cw, int max_cbs,
                            int emax, bool scrambling, uint32_t* d_out, hipStream_t strm)
{
    if (num_tbs < 0 || num_tbs > 65535 || max_cbs < 1 || max_cbs > 65535 || emax <= 0 || emax % 32 ||
        emax > DL_RM_MAX_EMAX)
        return CUPHY_STATUS_INVALID_ARGUMENT;
    if (num_tbs == 0) return CUPHY_STATUS_SUCCESS;
    if (!d_prms || !d_cw || !d_out) return CUPHY_STATUS_INVALID_ARGUMENT;
    const int emax_words = emax / 32;
    // the words of E <= emax scrambling bits from any bit of a word on, and one more
    const size_t lds = scrambling ? ((size_t)emax_words + 2) * sizeof(uint32_t) : 0;
    // a thread per 32 symbols: one wave holds 16,384 bits at 8 bits per symbol (at 2
    // it takes up to four turns: 2,800 blocks of 16,000 bits, whole call 24 us, the
    // host's time, as with 8)
    const unsigned block = emax_words <= 512 ? 64u : 256u;
    hipLaunchKernelGGL(dl_rate_match_kernel, dim3((unsigned)max_cbs, (unsigned)num_tbs), dim3(block), lds, strm, d_prms,
                       d_cw, max_cbs, emax_words, scrambling ? 1 : 0, d_out);
    return hipGetLastError() == hipSuccess ? CUPHY_STATUS_SUCCESS : CUPHY_STATUS_INTERNAL_ERROR;
}

}  // namespace nrldpc
