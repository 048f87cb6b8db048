// PUSCH de-rate-matching with HARQ soft combining (gfx950).
//
// Drop-in for the reference's puschRxRateMatch (cuPHY/src/cuphy/rate_matching/
// rate_matching.cu:239-1097); the per-CB arithmetic is in derate_core.hpp.
//   * descrambling (descramblingOn, not for UCI on PUSCH, as
//     rate_matching.cu:276): LLR n of the TB's rate-matched sequence is
//     negated where the Gold sequence c(n) of the TB's c_init is 1
//     (rate_matching.cu:378-387, 530-535); the CB's words of c are generated
//     into LDS first (gold_core.hpp);
//   * ndi = 1: write; ndi = 0: add to the HARQ buffer; clamp to +-10000;
//     untouched positions 0, filler +10000, the 2Zc punctured positions 0
//     (rate_matching.cu:622-683), HARQ layout [2Zc | Ncb] with stride
//     Ncb_padded per CB.
// Design difference (deterministic, atomics-free): one workgroup per CB.
// Its E LLRs come in symbol by symbol (one 16- or 32-byte load of a symbol's
// slots) and go, clamped and descrambled, to LDS in de-interleaved order
// (E * sizeof(TO) bytes); after one barrier every output position takes its
// LLRs from there -- positions that repeat (E > L = Ncb - F) in transmission
// order with a clamp after every addition -- so that the HARQ buffer is
// written once, in 16-byte stores, and read once when combining.  The
// reference uses atomicAdd in the wrap-around window plus a separate clamp
// pass.  A CB whose LLRs do not fit the launch's LDS walks the selected bits in
// passes of L with a barrier between passes, straight from and to memory
// (RM_LDS_LIMIT: E above 32,768 in binary16 and 16,384 in binary32; the
// sequence's words beside them: above 30,352 and 15,636 with descrambling).
// Bound by HBM: 2,800 BG1 Zc = 384 CBs of 9,088 bits in binary16 move 197 MB in
// a first transmission (39 us at the rate of a large copy) and 153 MB in a
// retransmission.  Measured 37 us on average of the two, against 69 us for the passes with a
// division and a 2-byte load and store per LLR.
#include "derate_core.hpp"
#include "derate_match.hpp"
#include "gold_core.hpp"

#include <algorithm>

namespace nrldpc {

template <typename TO, typename TI> __device__ __forceinline__ TO cvt_llr(TI v) { return (TO)v; }

template <typename T> struct rm_vec;  // the QAM_STRIDE slots of a symbol; 16 bytes of the output
template <> struct rm_vec<_Float16> {
    typedef _Float16 slots __attribute__((ext_vector_type(QAM_STRIDE)));
    typedef _Float16 out __attribute__((ext_vector_type(8)));
    static constexpr int N = 8;
};
template <> struct rm_vec<float> {
    typedef float slots __attribute__((ext_vector_type(QAM_STRIDE)));
    typedef float out __attribute__((ext_vector_type(4)));
    static constexpr int N = 4;
};

// Index in the input buffer of bit 0 of the CB's symbol j (bit k follows k
// further on), as rm_input_index.
__device__ __forceinline__ int rm_symbol_index(const rm_geometry& g, const PerTbParams& p, int j)
{
    if (g.uci) return g.start + j * g.Qm;
    if (g.Nl < g.nbbu) {
        const int jl = j / g.Nl;
        return g.adj * g.nbbu / g.Nl + (jl * g.nbbu + (int)p.layer_map_array[j - jl * g.Nl]) * QAM_STRIDE;
    }
    return g.adj + j * QAM_STRIDE;
}

// The CB's LLRs, clamped and descrambled, into llr[i], i = k * EQ + j.  seq:
// the words of c from word start / 32 on (seq_words of them).
template <typename TI, typename TO, bool DESCR>
__device__ __forceinline__ void rm_stage(TO* __restrict__ llr, const TI* __restrict__ in, const rm_geometry& g,
                                         const PerTbParams& p, bool descr, const uint32_t* __restrict__ seq)
{
    typedef typename rm_vec<TI>::slots slots_t;
    constexpr int NB = 4;  // symbols in flight per thread
    const int nthr = blockDim.x;
    const uint32_t soff = (uint32_t)g.start & 31u;
    // whole symbols by vector loads where every symbol starts at an aligned address
    const bool vec = !g.uci && ((uintptr_t)(in + rm_symbol_index(g, p, 0)) % sizeof(slots_t)) == 0;
    for (int j0 = threadIdx.x; j0 < g.EQ; j0 += NB * nthr) {
        slots_t v[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int j = min(j0 + u * nthr, g.EQ - 1);  // (past the end: the last symbol again, not stored)
            const TI* const src = in + rm_symbol_index(g, p, j);
            if (vec) {
                v[u] = *reinterpret_cast<const slots_t*>(src);
            } else {
#pragma unroll
                for (int k = 0; k < QAM_STRIDE; ++k) v[u][k] = (k < g.Qm) ? src[k] : (TI)0;
            }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int j = j0 + u * nthr;
            if (j >= g.EQ) break;
            uint32_t bits = 0;
            if (DESCR && descr) {  // bits n0 .. n0 + Qm - 1 (word n0 / 32 + 1 exists)
                const uint32_t n0 = soff + (uint32_t)(j * g.Qm);
                bits = __builtin_amdgcn_alignbit(seq[(n0 >> 5) + 1], seq[n0 >> 5], n0 & 31u);
            }
#pragma unroll
            for (int k = 0; k < QAM_STRIDE; ++k) {
                if (k < g.Qm) {
                    TO x = rm_num<TO>::clamp(cvt_llr<TO, TI>(v[u][k]));
                    if (DESCR && ((bits >> k) & 1u)) x = -x;
                    llr[k * g.EQ + j] = x;
                }
            }
        }
    }
}

// Whether c = c0 + d mod L of rm_position can be turned round to the d of a
// circle position (rm_combine).  A limited buffer that ends inside a long filler
// can have its start position past the circle's end (c0 > L); the passes
// over memory take it as it is.
__device__ __forceinline__ bool circle_inverts(const rm_geometry& g)
{
    return g.L <= 0 || (g.Kd >= 0 && g.c0 >= 0 && g.c0 <= g.L);
}

// Output positions from the staged LLRs: out[0, 2Zc) punctured, the circular
// buffer after it.  Circle position c holds LLRs d, d + L, ... < E, d = (c -
// c0) mod L.  A group of 16 bytes that is a run of consecutive d, all
// transmitted or none, is handled as a whole, any other value by value.
template <typename TO>
__device__ __forceinline__ void rm_combine(TO* __restrict__ out, const TO* __restrict__ llr, const rm_geometry& g)
{
    typedef typename rm_vec<TO>::out out_t;
    constexpr int G = rm_vec<TO>::N;
    const int head = 2 * g.Zc, E = g.L > 0 ? g.E : 0;
    // the filler is written whole, also where a limited buffer ends inside it
    const int total = head + max(g.Ncb, g.Kd + g.F);
    // value of position n after this transmission; false: not touched
    const auto one = [&](int n, TO& v) -> bool {
        const int q = n - head;
        if (q < 0 || (q >= g.Kd && q < g.Kd + g.F)) {
            v = (q < 0) ? (TO)0.0f : (TO)LLR_MAX_ABS;
            return g.ndi;
        }
        const int c = q < g.Kd ? q : q - g.F;
        if (c >= g.L) return false;
        const int d = c >= g.c0 ? c - g.c0 : c - g.c0 + g.L;
        if (d >= E && !g.ndi) return false;
        v = g.ndi ? (TO)0.0f : out[n];
        for (int i = d; i < E; i += g.L) v = rm_num<TO>::clamp(v + llr[i]);
        return true;
    };
    const bool aligned = ((uintptr_t)out & 15u) == 0;
    for (int n0 = (int)threadIdx.x * G; n0 < total; n0 += (int)blockDim.x * G) {
        if (aligned && n0 + G <= total) {
            const int q = n0 - head;
            if (g.ndi && (q + G <= 0)) {
                *reinterpret_cast<out_t*>(out + n0) = (out_t)((TO)0.0f);
                continue;
            }
            if (q >= 0 && (q + G <= g.Kd || q >= g.Kd + g.F)) {
                const int c = q < g.Kd ? q : q - g.F;
                const int d = c >= g.c0 ? c - g.c0 : c - g.c0 + g.L;
                if (c + G <= g.L && d + G <= g.L) {  // c .. c + G - 1 are d .. d + G - 1
                    if (d >= E) {
                        if (g.ndi) *reinterpret_cast<out_t*>(out + n0) = (out_t)((TO)0.0f);
                        continue;
                    }
                    if (d + G <= E) {
                        out_t v = (out_t)((TO)0.0f);
                        if (!g.ndi) v = *reinterpret_cast<const out_t*>(out + n0);
                        for (int i = d; i < E; i += g.L) {
#pragma unroll
                            for (int e = 0; e < G; ++e)
                                if (i + e < E) v[e] = rm_num<TO>::clamp(v[e] + llr[i + e]);
                        }
                        *reinterpret_cast<out_t*>(out + n0) = v;
                        continue;
                    }
                }
            }
        }
        for (int n = n0; n < min(n0 + G, total); ++n) {
            TO v;
            if (one(n, v)) out[n] = v;
        }
    }
}

// Bytes of dynamic LDS that this launch got: hidden_dynamic_lds_size of the
// implicit kernel arguments (code object version 5 and later).  Not taken from
// the descriptor, which a caller may set up again for other TBs under a
// kernel node that keeps the size of its own setup.
__device__ __forceinline__ uint32_t launch_lds_bytes()
{
    constexpr int OFFSET = 120;
    typedef const __attribute__((address_space(4))) uint32_t* arg_words;
    return ((arg_words)__builtin_amdgcn_implicitarg_ptr())[OFFSET / 4];
}

template <typename TI, typename TO, bool DESCR>
__global__ __launch_bounds__(RM_BLOCK) void derate_match_kernel(const rm_descriptor* __restrict__ desc)
{
    extern __shared__ __align__(16) unsigned char rm_lds[];
    __shared__ uint32_t seq_part[DESCR ? RM_SEQ_PART_WORDS : 1];
    const int cb_in_tb = blockIdx.x;
    const int tb_slot = blockIdx.y;
    const uint16_t ue = desc->sch_user_idxs[tb_slot];
    const PerTbParams& p = desc->tb_prms[ue];
    if (cb_in_tb >= (int)p.num_CBs) return;
    const int r = cb_in_tb + (int)p.firstCodeBlockIndex;
    TO* out = static_cast<TO*>(desc->out[ue]) + (size_t)r * p.Ncb_padded;
    const TI* in = static_cast<const TI*>(desc->llr_in[tb_slot]);
    const rm_geometry g = rm_geometry_of(p, cb_in_tb);

    // descrambling: nw words of c, from w_first on, cover the CB's bits [start, start + E)
    const uint32_t lds_words = launch_lds_bytes() / 4u;
    uint32_t* seq = reinterpret_cast<uint32_t*>(rm_lds);
    const bool descr = DESCR && !g.uci;
    const uint32_t w_first = (uint32_t)g.start >> 5;
    const uint32_t nw = (descr && g.E > 0) ? ((uint32_t)(g.start + g.E - 1) >> 5) - w_first + 1u : 0u;
    // (by one wave)
    const auto make_words = [&](uint32_t w, uint32_t n) {
        if (threadIdx.x < 64) gold_words_wave((uint32_t)__builtin_amdgcn_readfirstlane((int)p.cinit), w, (int)n, seq);
    };
    const uint32_t seq_words = descr ? (nw + 1u + 3u) & ~3u : 0u;  // one more word; the LLRs follow, 16-byte aligned
    if (rm_staged_fits(g.E, (int)sizeof(TO), seq_words, lds_words) && circle_inverts(g)) {
        if (descr) {
            make_words(w_first, nw);
            if (threadIdx.x == 0) seq[nw] = 0u;
            __syncthreads();
        }
        TO* const llr = reinterpret_cast<TO*>(seq + seq_words);
        rm_stage<TI, TO, DESCR>(llr, in, g, p, descr, seq);
        __syncthreads();
        rm_combine<TO>(out, llr, g);
        return;
    }

    // LLRs beyond the LDS: passes of distinct positions over memory, each in as
    // many parts as the sequence takes to fit (one with the setup's own LDS)
    TO* cbuf = out + 2 * g.Zc;
    uint32_t part_words = lds_words;
    if (DESCR && lds_words < (uint32_t)RM_SEQ_PART_WORDS) {
        seq = seq_part;
        part_words = RM_SEQ_PART_WORDS;
    }
    const uint32_t nparts = DESCR && nw > part_words ? (nw + part_words - 1u) / part_words : 1u;
    const int npass = rm_num_passes(g);
    for (int pass = 0; pass < npass; ++pass) {
        const int i0 = pass * g.L;
        const int span = g.ndi && pass == 0 ? g.L : min(g.L, g.E - i0);
        for (uint32_t part = 0; part < nparts; ++part) {
            const uint32_t w0 = part * part_words;
            if (descr && (nparts > 1u || pass == 0)) {  // (after the barrier that ends the part before)
                make_words(w_first + w0, min(part_words, nw - w0));
                __syncthreads();
            }
            for (int d = threadIdx.x; d < span; d += blockDim.x) {
                const int i = i0 + d;  // index in the de-interleaved sequence
                const int o = rm_position(g, d);
                if (i >= g.E) {  // ndi = 1, first pass: selected-bit positions not transmitted
                    if (part == 0) cbuf[o] = (TO)0.0f;
                    continue;
                }
                bool flip = false;
                if (descr) {
                    const uint32_t n = (uint32_t)rm_tx_position(g, i) - (w_first << 5);
                    const uint32_t w = (n >> 5) - w0;
                    if (w >= part_words) continue;  // in another part
                    flip = ((seq[w] >> (n & 31u)) & 1u) != 0;
                }
                TO v = rm_num<TO>::clamp(cvt_llr<TO, TI>(in[rm_input_index(g, p, i)]));
                if (flip) v = -v;
                const TO prev = (g.ndi && pass == 0) ? (TO)0.0f : cbuf[o];
                cbuf[o] = rm_num<TO>::clamp(prev + v);
            }
            __syncthreads();
        }
    }
    if (g.ndi) {
        for (int n = threadIdx.x; n < g.F; n += blockDim.x) cbuf[g.Kd + n] = (TO)LLR_MAX_ABS;
        for (int n = threadIdx.x; n < 2 * g.Zc; n += blockDim.x) out[n] = (TO)0.0f;
    }
}

// The reference launches separate reset and clamp kernels around the main
// one; this design needs neither, so their launch-configuration slots point
// at this empty kernel (grid 1) for callers that launch all three nodes.
__global__ void derate_match_noop_kernel(const rm_descriptor* desc) { (void)desc; }

template <bool DESCR>
void* rm_kernel_of(int fpconfig)
{
    switch (fpconfig) {
    case 0: return (void*)&derate_match_kernel<float, float, DESCR>;
    case 1: return (void*)&derate_match_kernel<_Float16, float, DESCR>;
    case 2: return (void*)&derate_match_kernel<float, _Float16, DESCR>;
    case 3: return (void*)&derate_match_kernel<_Float16, _Float16, DESCR>;
    default: return nullptr;
    }
}

void* rm_kernel(int fpconfig, bool descrambling)
{
    return descrambling ? rm_kernel_of<true>(fpconfig) : rm_kernel_of<false>(fpconfig);
}

int rm_lds_bytes(int fpconfig, const uint32_t* max_e, int n, bool descrambling)
{
    const int elem = (fpconfig == 2 || fpconfig == 3) ? 2 : 4;
    int words = 0;
    for (int i = 0; i < n; ++i) {
        const uint32_t e = std::min(max_e[i], (uint32_t)RM_MAX_DESCR_E);
        // a CB's bits start anywhere in a word; one more word; 16-byte units
        const int seq = descrambling ? (int)(((31u + e) / 32u + 2u + 3u) & ~3u) : 0;
        const int limit = (RM_LDS_LIMIT - (descrambling ? 4 * RM_SEQ_PART_WORDS : 0)) / 4;
        const int need = rm_staged_fits((int)e, elem, (uint32_t)seq, (uint32_t)limit)
                             ? seq + ((int)e * elem + 3) / 4
                             : seq;
        words = std::max(words, need);
    }
    return words * 4;
}

void* rm_noop_kernel() { return (void*)&derate_match_noop_kernel; }

}  // namespace nrldpc
