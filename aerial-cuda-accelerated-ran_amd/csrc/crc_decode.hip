// PUSCH code-block and transport-block CRC check with TB assembly (gfx950).
//
// Drop-in for the reference's puschRxCrcDecode (cuPHY/src/cuphy/crc/crc.cu:
// 55-237, setup :1174-1254):
//   CB kernel -- per code block: CRC over the ceil(K'/32) decoded words
//     (K' = K - F bits incl. the CB CRC; with C > 1 CRC24B, with C = 1 the
//     TB CRC itself: CRC16 when ceil(K'/8) <= 480 bytes else CRC24A);
//     remainder 0 = pass, stored at [sum of previous TBs' CBs + CB index];
//     the CB's data bytes (K' - 24 bits when C > 1, K' bits when C = 1) are
//     copied into the TB byte buffer, MSB-first per byte when reverseBytes
//     (bit 32w + i of the decoder output = bit i of word w);
//   TB kernel -- CRC24A over the assembled TB bytes (zero-padded to whole
//     words), remainder 0 = pass (C = 1: the CB kernel's remainder).
// Layouts as in the reference: CBs of TB y start at word sum_{i<y} C_i*264;
// TB y's bytes start at sum_{i<y} roundup4(C_i * data_bytes_i).
// CRC arithmetic (TS 38.212 5.1, zero initial value): thread t of S takes
// every S-th word (strided_crc in crc_core.hpp), the shares are XOR-combined.
// Pass/fail equals the reference's; a failing remainder's value is this
// definition's (the reference's depends on its LUT frame size).
//
// One wave per code block, four to a workgroup (they share the TB's step
// table in LDS); the TB's bytes go out as aligned words, each assembled from
// two decoded words, with single bytes only at a block's ends.  The offsets
// of a TB are sums over the TBs before it, taken by the lanes of the wave.
// The TB kernel gives each TB one workgroup, so that launches share no state
// and a setup's nodes may run on several streams at once (16 workgroups per
// TB, whose remainders met in the descriptor, took 10 us, but only one launch at
// a time was right).  16 waves: 147 KB in L2 take 18 us with 4, 13.6 with 8, 8.3
// with 16; bound by the four table reads per word (copies of the table against
// bank conflicts, 8 to 32: 8.7 to 9.3) and, on bytes that the CB kernel just
// wrote, by their way from other XCDs (more loads in flight: no change).
// Measured on 20 TBs of 140 BG1 Zc = 384 code blocks, against contiguous chunks
// per thread with byte tables in global memory, one loop over the TBs before and
// byte stores: CB kernel 30 -> 9 us, TB kernel 73 -> 18 us (both with about 4 us
// that an empty kernel measures the same way).
#include "crc_core.hpp"
#include "crc_decode.hpp"

namespace nrldpc {

// Step tables of the TB kernel's threads.
static __device__ const crc_stride_table<CRC_TB_BLOCK> g_tb_stride = make_crc_stride_table<CRC_TB_BLOCK>(CRC24A_P);

struct tb_layout {
    int cb_word_base, cb_count_base, tb_byte_base;
};

// Sums over the slots before `slot`, by the lanes of a wave (all active).
__device__ __forceinline__ tb_layout layout_of(const crc_descriptor& d, int slot)
{
    uint32_t cbs = 0, bytes = 0;
    for (int i = (int)(threadIdx.x & 63u); i < slot; i += 64) {
        const PerTbParams& q = d.tb_prms[d.sch_user_idxs[i]];
        const int data_bytes = ((int)(q.K - q.F) - cb_crc_bits(q) + 7) / 8;
        cbs += q.num_CBs;
        bytes += (uint32_t)(((int)q.num_CBs * data_bytes + 3) / 4 * 4);
    }
    const auto add = [](uint32_t a, uint32_t b) { return a + b; };
    if (slot > 0) {
        cbs = wave_reduce(cbs, add);
        bytes = wave_reduce(bytes, add);
    }
    return {(int)cbs * MAX_WORDS_PER_CB, (int)cbs, (int)bytes};
}

// The wave's code block: remainder of nw words (kind's polynomial).
template <typename Word>
__device__ __forceinline__ uint32_t wave_crc(int nw, int kind, Word word, const uint32_t (*table)[256])
{
    const uint32_t t = threadIdx.x & 63u;
    const uint32_t last = g_wave_stride[kind].last[t], fold = g_crc_fold.k[kind][t];
    const uint32_t v = strided_crc<64>(nw, (int)t, word, [&](int b, uint32_t x) { return table[b][x]; });
    return kind == K_CRC16 ? wave_sum_products<16>(t, v, last, fold) : wave_sum_products<24>(t, v, last, fold);
}

__global__ __launch_bounds__(CRC_CB_BLOCK) void crc_cb_kernel(const crc_descriptor* __restrict__ desc)
{
    __shared__ uint32_t step[4][256];
    const crc_descriptor& d = *desc;
    const int slot = blockIdx.y;
    const PerTbParams& p = d.tb_prms[d.sch_user_idxs[slot]];
    const int C = (int)p.num_CBs;
    if ((int)blockIdx.x * CRC_CBS_PER_BLOCK >= C) return;
    const int kind = cb_crc_kind(p);
    for (int i = threadIdx.x; i < 4 * 256; i += blockDim.x) (&step[0][0])[i] = (&g_wave_stride[kind].step[0][0])[i];
    const tb_layout l = layout_of(d, slot);
    __syncthreads();
    const int cb_in_tb = (int)blockIdx.x * CRC_CBS_PER_BLOCK + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (cb_in_tb >= C) return;  // (the whole wave)
    const int lane = (int)(threadIdx.x & 63u);
    const int cb = cb_in_tb + (int)p.firstCodeBlockIndex;
    const int nw = ((int)(p.K - p.F) + 31) / 32;
    const uint32_t* words = d.cb_in + l.cb_word_base + (size_t)cb * MAX_WORDS_PER_CB;
    const bool rev = d.reverse_bytes;
    const int data_bytes = cb_data_bytes(p);
    // message bytes in memory order; the message's first bit is the top bit of byte 0
    const auto bytes4 = [&](int w) { return rev ? rbit8x4(words[w]) : words[w]; };
    const uint32_t crc = wave_crc(nw, kind, [&](int w) { return __builtin_bswap32(bytes4(w)); }, step);
    uint8_t* const tb = d.tb_out + l.tb_byte_base;
    put_bytes(tb + (size_t)cb * data_bytes, data_bytes, bytes4, lane, 64);
    if (lane == 0) {
        d.cb_crc_out[l.cb_count_base + cb] = crc;
        if (cb_in_tb == 0) {
            if (C == 1) d.tb_crc_out[slot] = crc;
            const int bytes = C * data_bytes;
            for (int n = bytes; n < (bytes + 3) / 4 * 4; ++n) tb[n] = 0;
        }
    }
}

__global__ __launch_bounds__(CRC_TB_BLOCK) void crc_tb_kernel(const crc_descriptor* __restrict__ desc)
{
    __shared__ uint32_t table[4][256];
    __shared__ uint32_t red[CRC_TB_BLOCK / 64];
    const crc_descriptor& d = *desc;
    const int slot = blockIdx.x;
    const PerTbParams& p = d.tb_prms[d.sch_user_idxs[slot]];
    if (p.num_CBs <= 1) return;
    const int t = threadIdx.x;
    for (int i = t; i < 4 * 256; i += CRC_TB_BLOCK) (&table[0][0])[i] = (&g_tb_stride.step[0][0])[i];
    const uint32_t last = g_tb_stride.last[t], fold = g_crc_fold.k[K_CRC24A][t & 63];
    const tb_layout l = layout_of(d, slot);
    const int Kp = (int)(p.K - p.F);
    const int data_bytes = (Kp - 24 + 7) / 8;
    const int nw = ((int)p.num_CBs * data_bytes + 3) / 4;
    const uint32_t* tbw = reinterpret_cast<const uint32_t*>(d.tb_out + l.tb_byte_base);
    __syncthreads();
    const uint32_t v = wave_sum_products<24>(
        (uint32_t)t & 63u,
        strided_crc<CRC_TB_BLOCK>(
            nw, t, [&](int w) { return __builtin_bswap32(tbw[w]); },
            [&](int b, uint32_t x) { return table[b][x]; }),
        last, fold);
    if ((t & 63) == 0) red[t >> 6] = v;
    __syncthreads();
    if (t != 0) return;
    uint32_t crc = 0;
    for (int i = 0; i < (int)(CRC_TB_BLOCK / 64); ++i) crc ^= red[i];
    d.tb_crc_out[slot] = crc;
}

void* crc_cb_kernel_ptr() { return (void*)&crc_cb_kernel; }
void* crc_tb_kernel_ptr() { return (void*)&crc_tb_kernel; }

}  // namespace nrldpc
