// Systematic LDPC encoder for TS 38.212 BG1/BG2 (gfx950).
//
// Two entry kernels over one core: the decode path's test-signal source
// (bits as bytes, cuphyHipLDPCEncodeCodeBlocks: bench and serving workloads
// build their code blocks with it on the device) and the bit-packed encoder
// behind the reference's encoder API (cuphySetupLDPCEncode).  One workgroup
// encodes one code block in LDS, 32 bits per word and lane.  Check row z of
// block row r involves bit (z + s) mod Z of each connected column (circulant
// shifted right s times, TS 38.212 5.3.2).  Encoding uses the double-diagonal
// core of both base graphs (rows 0..3, parity columns p0..p3 = columns
// nsys..nsys+3):
//   lambda_i = sum of the systematic terms of core row i
//   BG1: row0 P^a p0 + p1,  row1 P^b p0 + p1 + p2,  row2 p2 + p3,  row3 P^a p0 + p3
//   BG2: row0 P^a p0 + p1,  row1 p1 + p2,  row2 P^b p0 + p2 + p3,  row3 P^a p0 + p3
// Summing the four rows leaves P^b p0 = sum_i lambda_i, so
// p0[y] = sum_i lambda_i[(y - b) mod Z]; p1, p3 follow from rows 0 and 3 and
// p2 from row 1.  Every extension column (nsys + r, r >= 4) has degree 1 and
// is the parity of its own row.  The result is checked against H*c = 0 and
// against the oracle's (independent, Gaussian-elimination) encoder.
//
// Layout: a column that check rows read (systematic and core parity) is kept
// twice over, bits [0, 64 * ceil(Z / 32)) of its periodic continuation, so
// that word w of the column rotated by any s is one funnel shift of the two
// words at bit 32 w + s, with no wrap to test: two LDS reads, a funnel shift
// and an XOR per edge and 32 check rows.  The edges' bit offsets (column *
// words + shift) are built in LDS once per code block.  The work is
// 316 * 12 edge words per BG1 Zc = 384 code block, so the launch is bound by
// its short dependent steps (eight barriers per code block), not by
// arithmetic or HBM.  2,800 such code blocks: 345 -> 18.6 us against one byte
// per bit and one check row per lane and step (12 MB in and out: 2.3 us).
#include "nr_ldpc_common.hpp"
#include "ldpc_encode.hpp"

#include <algorithm>

namespace nrldpc {

__device__ const reduced_shift_tables g_enc_shift_tables = make_reduced_shift_tables();
__device__ const graph_tables g_enc_graph = make_graph_tables();

// The last edge of every extension row is its own parity column, unshifted
// in every lifting set: the row's sum over the others is that column.
template <typename Tr> constexpr bool extension_rows_end_with_identity()
{
    for (int r = 4; r < Tr::NROWS; ++r) {
        const int e = Tr::row_start(r + 1) - 1;
        if (Tr::col(e) != Tr::NSYS + r || !Tr::identity_edge(e)) return false;
    }
    return true;
}
static_assert(extension_rows_end_with_identity<bg_traits<1>>() && extension_rows_end_with_identity<bg_traits<2>>(),
              "extension parity columns");

// Edge of row r at the first core parity column.
template <typename Tr> constexpr int core_edge(int r)
{
    for (int e = Tr::row_start(r); e < Tr::row_start(r + 1); ++e)
        if (Tr::col(e) == Tr::NSYS) return e;
    return -1;
}
static_assert(core_edge<bg_traits<1>>(0) >= 0 && core_edge<bg_traits<1>>(1) >= 0 && core_edge<bg_traits<2>>(0) >= 0 &&
                  core_edge<bg_traits<2>>(2) >= 0,
              "core parity column");

constexpr int ENC_PARTS = 4;         // lanes that share one word of a core row's sum (17..18 edges)
constexpr int ENC_MAX_EDGES = 320;

// LDS words of one code block: input words, edge offsets, row starts,
// columns, partial core sums, their total and the core parity columns.
__host__ __device__ inline int enc_col_words(int Z) { return 2 * ((Z + 31) / 32); }
__host__ __device__ inline int enc_raw_words(int nsys, int Z) { return (nsys * Z + 31) / 32 + 1; }
__host__ __device__ inline int enc_lds_words(int nsys, int nrows, int Z)
{
    const int nw = (Z + 31) / 32;
    return enc_raw_words(nsys, Z) + ENC_MAX_EDGES + 48 + (nsys + (nrows > 4 ? nrows : 4)) * enc_col_words(Z) +
           (4 * ENC_PARTS + 5) * nw;
}

// Threads of a workgroup: about one per (extension row, word) up to four
// waves; a code block of at most two words per column is one wave, whose
// barriers cost nothing.
static unsigned enc_block(int Z) { return Z <= 64 ? 64u : Z <= 160 ? 128u : 256u; }

struct enc_lds {
    uint32_t *raw, *edge, *rs, *x, *lam, *sum, *par;
    int nw, dw;
};
__device__ __forceinline__ enc_lds enc_carve(uint32_t* lds, int nsys, int nrows, int Z)
{
    enc_lds l;
    l.nw = (Z + 31) / 32;
    l.dw = enc_col_words(Z);
    l.raw = lds;
    l.edge = l.raw + enc_raw_words(nsys, Z);
    l.rs = l.edge + ENC_MAX_EDGES;
    l.x = l.rs + 48;
    l.lam = l.x + (nsys + max(nrows, 4)) * l.dw;
    l.sum = l.lam + 4 * ENC_PARTS * l.nw;
    l.par = l.sum + l.nw;
    return l;
}

// Bits [p, p + 32) of an LDS bit string (word (p >> 5) + 1 exists).
__device__ __forceinline__ uint32_t bits_at(const uint32_t* v, uint32_t p)
{
    return __builtin_amdgcn_alignbit(v[(p >> 5) + 1], v[p >> 5], p & 31u);
}

// Bits a .. a + 31 (a < Z) of the periodic continuation of the Z bits in
// v[0 .. nw), bits past Z zero.
__device__ __forceinline__ uint32_t cyclic_bits(const uint32_t* v, int nw, int Z, int a)
{
    const int i = a >> 5;
    const uint32_t hi = (i + 1 < nw) ? v[i + 1] : 0u;
    uint32_t r = __builtin_amdgcn_alignbit(hi, v[i], (uint32_t)a & 31u);
    for (int n = Z - a; n < 32; n += Z) r |= v[0] << n;
    return r;
}
__device__ __forceinline__ int wrap(int p, int Z) { return p >= Z ? p - Z : p; }
__device__ __forceinline__ int wrap_any(int p, int Z)
{
    while (p >= Z) p -= Z;
    return p;
}

// Encode one code block in LDS: l.raw holds its nsys * Z systematic bits on
// entry (bits past them zero), l.x the columns on return, column c's Z bits
// at l.x + c * l.dw (parity rows from nrows on are not computed, the core
// ones always).  Every thread of the workgroup calls it, after a barrier;
// ends with a barrier.
__device__ void encode_core(int bg, int Z, int nrows, const enc_lds& l)
{
    const int nsys = (bg == 1) ? 22 : 10;
    const int nw = l.nw, dw = l.dw;
    const int tid = threadIdx.x, nt = blockDim.x;
    // systematic columns, twice over
    for (int n = tid; n < nsys * dw; n += nt) {
        const int c = n / dw;
        const int a = wrap_any(32 * (n - c * dw), Z);
        uint32_t v = bits_at(l.raw, (uint32_t)(c * Z + a));
        if (Z - a < 32) {
            const uint32_t head = bits_at(l.raw, (uint32_t)(c * Z)) & low_bits(Z);
            v &= low_bits(Z - a);
            for (int k = Z - a; k < 32; k += Z) v |= head << k;
        }
        l.x[n] = v;
    }
    __syncthreads();
    // the core shifts a (row 0) and b (row 1 / 2) of column nsys
    const int base = nsys * dw * 32;
    const int a = (int)l.edge[bg == 1 ? core_edge<bg_traits<1>>(0) : core_edge<bg_traits<2>>(0)] - base;
    const int b = (int)l.edge[bg == 1 ? core_edge<bg_traits<1>>(1) : core_edge<bg_traits<2>>(2)] - base;
    // partial sums of the core rows' systematic terms
    for (int n = tid; n < 4 * ENC_PARTS * nw; n += nt) {
        const int w = n % nw, q = n / nw;
        const int r = q / ENC_PARTS, part = q % ENC_PARTS;
        uint32_t acc = 0;
        for (int e = (int)l.rs[r] + part; e < (int)l.rs[r + 1]; e += ENC_PARTS)
            if ((int)l.edge[e] < base) acc ^= bits_at(l.x, l.edge[e] + 32u * (uint32_t)w);
        l.lam[n] = acc;
    }
    __syncthreads();
    for (int w = tid; w < nw; w += nt) {
        uint32_t acc = 0;
        for (int r = 0; r < 4; ++r) {
            uint32_t v = 0;
            for (int p = 0; p < ENC_PARTS; ++p) v ^= l.lam[(r * ENC_PARTS + p) * nw + w];
            v &= low_bits(Z - 32 * w);
            l.lam[r * ENC_PARTS * nw + w] = v;  // (read by this thread only)
            acc ^= v;
        }
        l.sum[w] = acc;
    }
    __syncthreads();
    uint32_t* const p0 = l.par;
    for (int w = tid; w < nw; w += nt)
        p0[w] = cyclic_bits(l.sum, nw, Z, wrap_any(32 * w + Z - b, Z)) & low_bits(Z - 32 * w);
    __syncthreads();
    for (int w = tid; w < nw; w += nt) {
        const uint32_t m = low_bits(Z - 32 * w);
        const uint32_t pa = cyclic_bits(p0, nw, Z, wrap(32 * w + a, Z));
        const uint32_t p1 = (l.lam[w] ^ pa) & m;
        uint32_t p2 = l.lam[ENC_PARTS * nw + w] ^ p1;
        if (bg == 1) p2 ^= cyclic_bits(p0, nw, Z, wrap(32 * w + b, Z));
        l.par[nw + w] = p1;
        l.par[2 * nw + w] = p2 & m;
        l.par[3 * nw + w] = (l.lam[3 * ENC_PARTS * nw + w] ^ pa) & m;
    }
    __syncthreads();
    // core parity columns, twice over
    for (int n = tid; n < 4 * dw; n += nt) {
        const int c = n / dw;
        l.x[nsys * dw + n] = cyclic_bits(l.par + c * nw, nw, Z, wrap_any(32 * (n - c * dw), Z));
    }
    __syncthreads();
    // extension rows: column nsys + r is the sum over row r's other edges
    for (int n = tid; n < (nrows - 4) * nw; n += nt) {
        const int r = 4 + n / nw, w = n % nw;
        uint32_t acc = 0;
        for (int e = (int)l.rs[r]; e < (int)l.rs[r + 1] - 1; ++e) acc ^= bits_at(l.x, l.edge[e] + 32u * (uint32_t)w);
        l.x[(nsys + r) * dw + w] = acc;
    }
    __syncthreads();
}

// Bits n .. n + 31 of the code word (column after column), 0 past ncols.
__device__ __forceinline__ uint32_t codeword_bits(const enc_lds& l, int Z, int ncols, int n)
{
    int c = n / Z, a = n - c * Z;
    uint32_t v = 0;
    for (int got = 0; got < 32 && c < ncols; ++c) {
        v |= (bits_at(l.x + c * l.dw, (uint32_t)a) & low_bits(Z - a)) << got;
        got += Z - a;
        a = 0;
    }
    return v;
}

// Edge offsets (as bit positions in l.x) and row starts of the base graph
// into LDS; zi: the lifting size's index.
__device__ __forceinline__ void load_graph(int bg, int zi, const enc_lds& l)
{
    const int nrows = (bg == 1) ? 46 : 42;
    const uint32_t* sh = g_enc_shift_tables.v[bg - 1][zi];
    const uint16_t* rs = g_enc_graph.row_start[bg - 1];
    const uint8_t* col = g_enc_graph.col[bg - 1];
    const int ne = (bg == 1) ? NR_BG1_NUM_EDGES : NR_BG2_NUM_EDGES;
    for (int e = threadIdx.x; e < ne; e += blockDim.x) l.edge[e] = (uint32_t)col[e] * (uint32_t)l.dw * 32u + sh[e];
    for (int r = threadIdx.x; r <= nrows; r += blockDim.x) l.rs[r] = rs[r];
}

__global__ __launch_bounds__(256) void ldpc_encode_kernel(int bg, int Z, int zi, const uint8_t* __restrict__ info, int info_stride,
                                                          uint8_t* __restrict__ cw, int cw_stride)
{
    extern __shared__ uint32_t enc_lds_raw[];
    const int nsys = (bg == 1) ? 22 : 10;
    const int nrows = (bg == 1) ? 46 : 42;
    const enc_lds l = enc_carve(enc_lds_raw, nsys, nrows, Z);
    const uint8_t* src = info + (size_t)blockIdx.x * info_stride;
    uint8_t* dst = cw + (size_t)blockIdx.x * cw_stride;
    const int tid = threadIdx.x, nt = blockDim.x;
    load_graph(bg, zi, l);
    // 64 bytes per wave and step, one ballot
    const int kbits = nsys * Z, nraw = enc_raw_words(nsys, Z);
    for (int n = tid; n - (tid & 63) < 32 * nraw; n += nt) {
        const uint64_t m = __ballot(n < kbits && (src[n < kbits ? n : 0] & 1u));
        if ((tid & 63) == 0) l.raw[n >> 5] = (uint32_t)m;
        if ((tid & 63) == 32 && (n >> 5) < nraw) l.raw[n >> 5] = (uint32_t)(m >> 32);
    }
    __syncthreads();
    encode_core(bg, Z, nrows, l);
    // four bits to four bytes (the code word is a multiple of 4 bits)
    for (int n = 4 * tid; n < (nsys + nrows) * Z; n += 4 * nt) {
        const uint32_t v = ((codeword_bits(l, Z, nsys + nrows, n) & 0xFu) * 0x00204081u) & 0x01010101u;
        __builtin_memcpy(dst + n, &v, 4);
    }
}

// Bit-packed encoder of cuphySetupLDPCEncode: block (c, t) encodes code word
// c of TB t.  Input: Kb * Z information bits (bit i of word w = bit 32 w + i,
// filler bits as the caller set them); output: codeword bits from column 2
// (puncture) or 0 up to column nsys + num_rows, packed the same way, the
// rest of the last word 0.
__global__ __launch_bounds__(256) void ldpc_encode_bits_kernel(enc_descr d)
{
    extern __shared__ uint32_t enc_lds_raw[];
    const int t = blockIdx.y, c = blockIdx.x;
    const enc_tensor in = d.input[t], out = d.output[t];
    if (c >= in.num_cw || c >= out.num_cw) return;
    const int Z = d.Z, bg = d.BG;
    const int nsys = (bg == 1) ? 22 : 10;
    const enc_lds l = enc_carve(enc_lds_raw, nsys, d.num_rows, Z);
    const uint32_t* src = in.addr + (size_t)c * in.stride_words;
    uint32_t* dst = out.addr + (size_t)c * out.stride_words;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int kbits = d.Kb * Z, nraw = enc_raw_words(nsys, Z);
    for (int w = tid; w < nraw; w += nt) l.raw[w] = (32 * w < kbits) ? src[w] & low_bits(kbits - 32 * w) : 0u;
    load_graph(bg, d.zi, l);
    __syncthreads();
    encode_core(bg, Z, d.num_rows, l);
    const int first = d.puncture ? 2 * Z : 0;
    const int ncols = nsys + d.num_rows;
    const int nbits = ncols * Z - first;
    for (int w = tid; w < (nbits + 31) / 32; w += nt) dst[w] = codeword_bits(l, Z, ncols, first + 32 * w);
}

cuphyStatus_t encode_cbs(int bg, int Z, const uint8_t* info, int info_stride, int ncb, uint8_t* cw, int cw_stride,
                         hipStream_t strm)
{
    if ((bg != 1 && bg != 2) || lifting_size_index(Z) < 0 || !info || !cw || ncb < 0) return CUPHY_STATUS_INVALID_ARGUMENT;
    const int nsys = (bg == 1) ? 22 : 10, nrows = (bg == 1) ? 46 : 42;
    if (info_stride < nsys * Z || cw_stride < (nsys + nrows) * Z) return CUPHY_STATUS_INVALID_ARGUMENT;
    if (ncb == 0) return CUPHY_STATUS_SUCCESS;
    const size_t lds = (size_t)enc_lds_words(nsys, nrows, Z) * sizeof(uint32_t);
    hipLaunchKernelGGL(ldpc_encode_kernel, dim3(ncb), dim3(enc_block(Z)), lds, strm, bg, Z,
                       lifting_size_index(Z), info, info_stride, cw, cw_stride);
    return hipGetLastError() == hipSuccess ? CUPHY_STATUS_SUCCESS : CUPHY_STATUS_INTERNAL_ERROR;
}

encode_geometry encode_bits_geometry(int bg, int Z, int num_rows)
{
    return {(void*)&ldpc_encode_bits_kernel, enc_block(Z),
            (unsigned)(enc_lds_words(bg == 1 ? 22 : 10, num_rows, Z) * (int)sizeof(uint32_t)),
            lifting_size_index(Z)};
}

}  // namespace nrldpc
