// Device core of the TS 38.211 5.2.1 Gold sequence (PUSCH descrambling) for
// gfx950: c(n) = x1(n + 1600) ^ x2(n + 1600), x1(n+31) = x1(n+3) ^ x1(n)
// (x1(0) = 1, x1(1..30) = 0), x2(n+31) = x2(n+3) ^ x2(n+2) ^ x2(n+1) ^ x2(n)
// (x2(0..30) = bits of c_init); the reference generates it with gold32n
// (cuPHY/src/cuphy/descrambling/descrambling.cuh:384) from lookup tables.
//
// Here one wave makes a run of 32-bit words, 64 at a time:
//   * the LFSR states at the run's first word: the word index in radix 16,
//     one 31x31 GF(2) matrix A^(32 * 16^d * v) per digit (compile-time
//     tables; the lowest digit's include the 1600 skipped steps).  A wave
//     applies a matrix in one step: lane i < 31 takes the parity of row i &
//     state, a ballot gathers the new state.  The rows of all five digits
//     are loaded together, before the first is used.
//   * lane t's word, 32 t steps on: with x^(32 t) mod f = sum of x^j over j
//     in J(t) (f the sequence's polynomial), x(n + 32 t) is the XOR of
//     x(n + j) over J(t): the XOR of shifted copies of the 62 bits that
//     follow from the state.
//   * the next 64 words from the last: x(n + 2048) likewise, where x^2048
//     mod f has 3 and 5 terms: about 20 operations for 64 words.
// Bound by its dependent chain (about 200 operations to the first 64 words).
// Measured against two matrix applications per word, each wave jumping to its
// share with a dependent table load per set bit: de-rate-match kernel of 200
// code blocks of 10,808 bits 41.5 -> 24.1 us, DL rate-match kernel of 2,800
// blocks of 9,088 bits 81 -> 47 us.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nrldpc {

constexpr int GOLD_NC = 1600;
constexpr int GOLD_DIGITS = 5;  // word indices below 16^5

constexpr uint32_t GOLD_MASK31 = 0x7FFFFFFFu;
// f without its leading x^31
constexpr uint32_t gold_poly(int q) { return q == 0 ? 0x9u : 0xFu; }

struct gold_matrix {
    uint32_t row[32];  // row i: mask of the state bits that sum to new bit i; row 31 unused
};
constexpr gold_matrix gold_mul(const gold_matrix& a, const gold_matrix& b)
{
    gold_matrix r{};
    for (int i = 0; i < 31; ++i) {
        uint32_t v = 0;
        for (int j = 0; j < 31; ++j)
            if ((a.row[i] >> j) & 1u) v ^= b.row[j];
        r.row[i] = v;
    }
    return r;
}
constexpr gold_matrix gold_step(int q)  // one step
{
    gold_matrix m{};
    for (int i = 0; i < 30; ++i) m.row[i] = 1u << (i + 1);
    m.row[30] = gold_poly(q);
    return m;
}
constexpr gold_matrix gold_power(const gold_matrix& m, int n)
{
    gold_matrix r{};
    for (int i = 0; i < 31; ++i) r.row[i] = 1u << i;
    gold_matrix s = m;
    for (; n; n >>= 1) {
        if (n & 1) r = gold_mul(r, s);
        if (n > 1) s = gold_mul(s, s);
    }
    return r;
}

struct gold_digit_table {
    gold_matrix m[16];  // A^(32 * 16^d * v), v = 0 .. 15 (d = 0: times A^1600)
};
constexpr gold_digit_table make_gold_digit(int q, int d)
{
    gold_digit_table t{};
    gold_matrix b = gold_power(gold_step(q), 32);
    for (int i = 0; i < 4 * d; ++i) b = gold_mul(b, b);
    t.m[0] = gold_power(gold_step(q), d == 0 ? GOLD_NC : 0);
    for (int v = 1; v < 16; ++v) t.m[v] = gold_mul(t.m[v - 1], b);
    return t;
}

// a * b mod f, polynomials as bit masks
constexpr uint32_t gold_poly_mul(uint32_t a, uint32_t b, int q)
{
    uint32_t r = 0;
    for (int i = 30; i >= 0; --i) {
        r = ((r << 1) & GOLD_MASK31) ^ (((r >> 30) & 1u) ? gold_poly(q) : 0u);
        if ((b >> i) & 1u) r ^= a;
    }
    return r;
}
constexpr uint32_t gold_x_pow(int n, int q)
{
    uint32_t r = 1, s = 2;
    for (; n; n >>= 1) {
        if (n & 1) r = gold_poly_mul(r, s, q);
        s = gold_poly_mul(s, s, q);
    }
    return r;
}
struct gold_lane_table {
    uint32_t j[2][64];  // x^(32 t) mod f
};
constexpr gold_lane_table make_gold_lanes()
{
    gold_lane_table t{};
    for (int q = 0; q < 2; ++q) {
        uint32_t v = 1;
        for (int i = 0; i < 64; ++i) {
            t.j[q][i] = v;
            v = gold_poly_mul(v, gold_x_pow(32, q), q);
        }
    }
    return t;
}

static __device__ const gold_digit_table g_gold_digits[2][GOLD_DIGITS] = {
    {make_gold_digit(0, 0), make_gold_digit(0, 1), make_gold_digit(0, 2), make_gold_digit(0, 3), make_gold_digit(0, 4)},
    {make_gold_digit(1, 0), make_gold_digit(1, 1), make_gold_digit(1, 2), make_gold_digit(1, 3), make_gold_digit(1, 4)}};
static __device__ const gold_lane_table g_gold_lanes = make_gold_lanes();

// Bits 31 .. of a sequence from its bits 0 .. 30 (or 31): bit i of the
// result is x(n + 31 + i), valid for i < 28.
template <int Q> __device__ __forceinline__ uint32_t gold_next(uint32_t s)
{
    return Q == 0 ? s ^ (s >> 3) : s ^ (s >> 1) ^ (s >> 2) ^ (s >> 3);
}

// The 62 bits x(n) .. x(n + 61) that follow from a state (31 bits).
template <int Q> __device__ __forceinline__ uint64_t gold_window(uint32_t s)
{
    uint64_t v = (uint64_t)s | ((uint64_t)(gold_next<Q>(s) & 0x0FFFFFFFu) << 31);
    return v | ((uint64_t)(gold_next<Q>((uint32_t)(v >> 28)) & 7u) << 59);
}

// Words 64 further on: lane t's word w -> word w + 64.
template <int Q> __device__ __forceinline__ uint32_t gold_advance64(uint32_t w)
{
    constexpr uint32_t J = gold_x_pow(2048, Q);
    static_assert((J >> 23) == 0, "the window of a word and its continuation holds 59 bits");
    const uint32_t hi = gold_next<Q>(w) >> 1;  // x(n + 32 + i), valid for i < 27
    uint32_t r = 0;
#pragma unroll
    for (int j = 0; j < 23; ++j)
        if ((J >> j) & 1u) r ^= __builtin_amdgcn_alignbit(hi, w, (uint32_t)j);
    return r;
}

// Words w0 .. w0 + nw - 1 of c for c_init into seq[0 .. nw) (bit b of word w
// = c(32 w + b)), generated by one wave (every lane active; arguments
// uniform).
__device__ __forceinline__ void gold_words_wave(uint32_t cinit, uint32_t w0, int nw, uint32_t* seq)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t rows[2][GOLD_DIGITS];
#pragma unroll
    for (int d = 0; d < GOLD_DIGITS; ++d) {
        const uint32_t v = (w0 >> (4 * d)) & 15u;
        rows[0][d] = g_gold_digits[0][d].m[v].row[lane & 31u];
        rows[1][d] = g_gold_digits[1][d].m[v].row[lane & 31u];
    }
    const uint32_t j1 = g_gold_lanes.j[0][lane], j2 = g_gold_lanes.j[1][lane];
    uint32_t s1 = 1u, s2 = cinit & GOLD_MASK31;
#pragma unroll
    for (int d = 0; d < GOLD_DIGITS; ++d) {
        s1 = (uint32_t)__ballot((__builtin_popcount(rows[0][d] & s1) & 1) != 0) & GOLD_MASK31;
        s2 = (uint32_t)__ballot((__builtin_popcount(rows[1][d] & s2) & 1) != 0) & GOLD_MASK31;
    }
    const uint64_t v1 = gold_window<0>(s1), v2 = gold_window<1>(s2);
    uint32_t x1 = 0, x2 = 0;
#pragma unroll
    for (int j = 0; j < 31; ++j) {
        x1 ^= (uint32_t)((int32_t)(j1 << (31 - j)) >> 31) & (uint32_t)(v1 >> j);
        x2 ^= (uint32_t)((int32_t)(j2 << (31 - j)) >> 31) & (uint32_t)(v2 >> j);
    }
    for (int w = (int)lane; w - (int)lane < nw; w += 64) {
        if (w < nw) seq[w] = x1 ^ x2;
        x1 = gold_advance64<0>(x1);
        x2 = gold_advance64<1>(x2);
    }
}

}  // namespace nrldpc
