// Device core of the CRC checks (TS 38.212 5.1, zero initial value), shared
// by the PUSCH CRC-decode kernels and the fused slot kernel.  Every thread
// computes the remainder of every S-th word of the message, shifted by the bits
// after it (strided_crc), and the shares are XOR-combined (CRC linearity).  All
// tables are built at compile time.
#pragma once

#include "nr_ldpc_common.hpp"

namespace nrldpc {

struct crc_poly {
    uint32_t g;     // polynomial without the leading term
    int L;          // degree
};

constexpr crc_poly CRC24A_P{0x864CFBu, 24};
constexpr crc_poly CRC24B_P{0x800063u, 24};
constexpr crc_poly CRC16_P{0x1021u, 16};
enum { K_CRC24A = 0, K_CRC24B = 1, K_CRC16 = 2 };

// a*b mod g (both < 2^L), carry-less
constexpr uint32_t gf2_mulmod(uint32_t a, uint32_t b, crc_poly p)
{
    const uint32_t mask = (p.L == 32) ? 0xFFFFFFFFu : ((1u << p.L) - 1u);
    uint32_t r = 0;
    for (int i = p.L - 1; i >= 0; --i) {
        const bool top = (r >> (p.L - 1)) & 1u;
        r = (r << 1) & mask;
        if (top) r ^= p.g;
        if ((b >> i) & 1u) r ^= a;
    }
    return r;
}

constexpr uint32_t byte_entry(uint32_t v, crc_poly p)
{
    const uint32_t mask = (1u << p.L) - 1u;
    uint32_t r = v << (p.L - 8);
    for (int i = 0; i < 8; ++i) r = ((r << 1) & mask) ^ (((r >> (p.L - 1)) & 1u) ? p.g : 0u);
    return r;
}

// The bits inside each byte reversed (byte order kept).
__device__ __forceinline__ uint32_t rbit8x4(uint32_t w) { return __builtin_bswap32(__builtin_bitreverse32(w)); }

// Multiplication of a 32-bit (unreduced) value by x^(32 * S) mod g, by
// bytes: v * x^(32 S) = XOR over b of step[b][byte b of v]; and the factors
// x^(32 t + L) of the last word of thread t of S.
template <int S> struct crc_stride_table {
    uint32_t step[4][256];
    uint32_t last[S];
};
template <int S> constexpr crc_stride_table<S> make_crc_stride_table(crc_poly p)
{
    crc_stride_table<S> t{};
    const uint32_t mask = (1u << p.L) - 1u;
    uint32_t x32 = 1, xs = 1;  // x^32, x^(32 S)
    for (int i = 0; i < 32; ++i) x32 = gf2_mulmod(x32, 2u, p);
    for (int i = S; i > 1; i >>= 1) xs = (i == S) ? gf2_mulmod(x32, x32, p) : gf2_mulmod(xs, xs, p);
    uint32_t v = xs;
    for (int b = 0; b < 4; ++b)
        for (int i = 0; i < 8; ++i) {
            for (int n = 0; n < (1 << i); ++n) t.step[b][(1 << i) + n] = t.step[b][n] ^ v;
            v = ((v << 1) & mask) ^ (((v >> (p.L - 1)) & 1u) ? p.g : 0u);
        }
    v = 1;
    for (int i = 0; i < p.L; ++i) v = ((v << 1) & mask) ^ (((v >> (p.L - 1)) & 1u) ? p.g : 0u);
    for (int n = 0; n < S; ++n) {
        t.last[n] = v;
        for (int b = 0; b < 4; ++b) v = ((v << 8) & mask) ^ byte_entry((v >> (p.L - 8)) & 0xFFu, p);
    }
    return t;
}

// Reduction of x over the wave, returned in every lane: within each row of
// 16 lanes by DPP (lane pairs, quads, half rows, rows: register-to-register,
// no LDS round trip), then across the four rows by readlane.  Every lane
// of the wave must be active (workgroups of whole waves, called in uniform
// control flow).
template <typename Op> __device__ __forceinline__ uint32_t wave_reduce(uint32_t x, Op op)
{
    x = op(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
    x = op(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
    x = op(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, false));  // row_half_mirror
    x = op(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x140, 0xF, 0xF, false));  // row_mirror
    const auto at = [&](int l) { return (uint32_t)__builtin_amdgcn_readlane((int)x, l); };
    return op(op(at(0), at(16)), op(at(32), at(48)));
}
__device__ __forceinline__ uint32_t wave_xor(uint32_t x)
{
    return wave_reduce(x, [](uint32_t a, uint32_t b) { return a ^ b; });
}

// Lane index, opaque: what depends on it alone (table loads, addresses) is then
// computed where it is used instead of being hoisted out of a persistent
// kernel's item loop into registers held across the decode.
__device__ __forceinline__ uint32_t opaque_lane()
{
    uint32_t t = threadIdx.x & 63u;
    asm volatile("" : "+v"(t));
    return t;
}

// Remainder of carry-less products, on a wave: the products' XOR over the
// lanes is reduced once, lane i contributing x^(L + i) mod g where bit L + i
// of it is set.
struct crc_fold_table {
    uint32_t k[3][64];  // x^(L + i) mod g of CRC24A, CRC24B, CRC16
};
constexpr crc_fold_table make_crc_fold_table()
{
    crc_fold_table t{};
    const crc_poly ps[3] = {CRC24A_P, CRC24B_P, CRC16_P};
    for (int q = 0; q < 3; ++q) {
        const uint32_t mask = (1u << ps[q].L) - 1u;
        uint32_t v = ps[q].g;  // x^L mod g
        for (int i = 0; i < 64; ++i) {
            t.k[q][i] = v;
            v = ((v << 1) & mask) ^ (((v >> (ps[q].L - 1)) & 1u) ? ps[q].g : 0u);
        }
    }
    return t;
}
static __device__ const crc_fold_table g_crc_fold = make_crc_fold_table();

// XOR over the wave of the 64-bit p, mod g (degree L, p < 2^(L + 64)), the
// same value in every lane; fold: the lane's entry of the polynomial's fold
// table.
template <int L> __device__ __forceinline__ uint32_t wave_fold(uint32_t lane, uint32_t lo, uint32_t hi, uint32_t fold)
{
    const uint64_t c = ((uint64_t)wave_xor(hi) << 32) | wave_xor(lo);
    const uint32_t bit = (lane < 64u - (uint32_t)L) ? (uint32_t)(c >> (lane + (uint32_t)L)) & 1u : 0u;
    return ((uint32_t)c & ((1u << L) - 1u)) ^ wave_xor((0u - bit) & fold);
}

// XOR over the lanes of v * f mod g (v any 32-bit value, f < 2^24): 32
// independent masked shifts per lane, one reduction.
template <int L>
__device__ __forceinline__ uint32_t wave_sum_products(uint32_t lane, uint32_t v, uint32_t f, uint32_t fold)
{
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const uint32_t m = (uint32_t)((int32_t)(v << (31 - i)) >> 31);
        lo ^= m & (f << i);
        if (i > 8) hi ^= m & (f >> (32 - i));
    }
    return wave_fold<L>(lane, lo, hi, fold);
}

// a * b mod g for uniform a, b < 2^24 and a polynomial of degree 24: lane i
// takes bit i of a.
__device__ __forceinline__ uint32_t wave_mulmod24(uint32_t lane, uint32_t a, uint32_t b, uint32_t fold)
{
    const uint64_t p = (lane < 24u && ((a >> lane) & 1u)) ? (uint64_t)b << lane : 0u;
    return wave_fold<24>(lane, (uint32_t)p, (uint32_t)(p >> 32), fold);
}

// Step tables of a wave (thread t of 64), by CRC kind.
static __device__ const crc_stride_table<64> g_wave_stride[3] = {
    make_crc_stride_table<64>(CRC24A_P), make_crc_stride_table<64>(CRC24B_P), make_crc_stride_table<64>(CRC16_P)};

// Share of the remainder of nw message words (`word(i)` = message word i,
// its first bit the most significant) that thread t of S holds: the words
// nw - 1 - t - S * i, by Horner's rule from the first, step(b, x) =
// x * x^(8 b + 32 S) mod g from the stride table.  Multiplied by
// x^(32 t + L) (the table's `last`) and XORed over the threads it gives the
// remainder.  The S threads read consecutive words; a step is four
// independent table reads.
template <int S, typename Word, typename Step>
__device__ __forceinline__ uint32_t strided_crc(int nw, int t, Word word, Step step)
{
    constexpr int U = 4;  // words in flight
    int i = (nw + S - 1) / S - 1;
    // (the first word needs no step; only it can be missing)
    uint32_t v = (i >= 0 && i * S + t < nw) ? word(nw - 1 - i * S - t) : 0u;
    for (--i; i >= 0; i -= U) {
        uint32_t w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = (i >= u) ? word(nw - 1 - (i - u) * S - t) : 0u;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i >= u) v = step(0, v & 255u) ^ step(1, (v >> 8) & 255u) ^ step(2, (v >> 16) & 255u) ^ step(3, v >> 24) ^ w[u];
    }
    return v;
}

// Byte-granular shift factors of CRC24A: x^(8m) and x^(8 * 1024 * m) mod g, for
// shifts inside a TB of up to 256 KiB (x^(8n) = x^(8 (n mod 1024)) *
// x^(8 * 1024 * (n / 1024))).  Built at compile time.
struct crc_shift_tables {
    uint32_t lo[1024];
    uint32_t hi[256];
};

constexpr crc_shift_tables make_crc_shift_tables()
{
    crc_shift_tables t{};
    uint32_t v = 1;  // x^0, advanced by x^8: one byte-wise step with a zero input byte
    const auto step8 = [&] { v = ((v << 8) & 0xFFFFFFu) ^ byte_entry(v >> 16, CRC24A_P); };
    for (int m = 0; m < 1024; ++m, step8()) t.lo[m] = v;
    const uint32_t step = v;  // x^(8 * 1024)
    v = 1;
    for (int m = 0; m < 256; ++m, v = gf2_mulmod(v, step, CRC24A_P)) t.hi[m] = v;
    return t;
}

static __device__ const crc_shift_tables g_crc_shift = make_crc_shift_tables();

// Bytes 0 .. nbytes - 1 of a message (bytes4(w): its word w, bytes in memory
// order) to dst, by thread t of n: whole aligned words of the destination, each
// from two message words, single bytes only at both ends.
template <typename Bytes4> __device__ __forceinline__ void put_bytes(uint8_t* dst, int nbytes, Bytes4 bytes4, int t, int n)
{
    const int head = min(nbytes, (int)((0u - (uint32_t)(uintptr_t)dst) & 3u));
    const int nfull = (nbytes - head) >> 2, tail = head + 4 * nfull;
    for (int i = t; i < nfull; i += n) {
        const uint32_t lo = bytes4(i), hi = (head != 0) ? bytes4(i + 1) : 0u;  // (byte 4 i + 3 + head < nbytes)
        *reinterpret_cast<uint32_t*>(dst + head + 4 * i) = __builtin_amdgcn_alignbyte(hi, lo, (uint32_t)head);
    }
    const int b = t < head ? t : tail + t - head;
    if (t < head + nbytes - tail) dst[b] = (uint8_t)(bytes4(b >> 2) >> (8 * (b & 3)));
}

// CRC bits attached to each CB: 24 (CRC24B) when the TB is segmented.
__device__ __forceinline__ int cb_crc_bits(const PerTbParams& p)
{
    return p.num_CBs > 1 ? 24 : 0;
}

// Payload bytes one CB contributes to the TB byte buffer.
__device__ __forceinline__ int cb_data_bytes(const PerTbParams& p)
{
    return ((int)(p.K - p.F) - cb_crc_bits(p) + 7) / 8;
}

// CRC checked over a CB's K' bits: CRC24B when the TB is segmented, else
// the TB CRC itself (CRC16 up to 480 bytes incl. the CRC, i.e. A <= 3824).
__device__ __forceinline__ int cb_crc_kind(const PerTbParams& p)
{
    return p.num_CBs > 1 ? K_CRC24B : (cb_data_bytes(p) <= 480 ? K_CRC16 : K_CRC24A);
}

}  // namespace nrldpc
