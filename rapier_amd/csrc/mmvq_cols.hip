// mmvq_cols.hip - GGUF-layout GEMV over several activation columns (prompt chunks) in one pass over the weights, on the
// int8 matrix cores: Q4_K, Q5_K, Q6_K and Q8_0, up to 16 columns, gfx950.
//
// Reference behaviour: the multi-column kernels of src/native_mmvq.cu (1261-1356 and the IL kernels 1625-2310).
//
// The one- to four-column kernels (mmvq_kquant.hip, mmvq_q6k.hip, mmvq_q8_0.hip) take 16 columns in four passes over
// the weights and form every dot product with v_dot4.  Here a wave holds 16 rows x 16 columns of outputs in one
// 16x16x32 MFMA tile: activations are the A operand (a lane's registers run over four columns), weights the B operand
// (a lane is a row, so its scales are lane values), K is one Q8_1 block.
//
// Every output has the single-column kernel's bits.  That kernel gives a row's unit u (a Q4_K / Q5_K block's 64-element
// pair, a Q6_K half-block, a Q8_0 block) to lane u % NL, adds a lane's units in order and ends with an xor butterfly
// over the NL lanes (NL 64; Q6_K 16, 32 or 64 by shape).  Here the eight waves of a workgroup share a tile's units by
// lane % 8 (K-quants: block % 8, with the four pairs of a block side by side), a wave walks its lanes in the
// butterfly's depth-first order with a stack of three partial sums, and the last three levels meet in LDS.
//  * Q4_K / Q5_K: the dot of a sub-block times its scale and the code sum times the min are whole numbers below 2^24,
//    formed in fp32 without rounding (kBias below; the sums from a table made with the scales).
//  * Q6_K: sub-scale * (code - 32) cut in two int8 digits, s = (hi . x << 8) + lo . x, as the ingest GEMM does.
// Bound: the vector unit and the LDS (a block of 16 rows: ~250 vector instructions per wave; one workgroup per CU, so a
// tile's load wait, unpacking and sum over the waves overlap little).  16 columns of 24576 x 4096: Q4_K 78 -> 25 us, Q5_K
// 82 -> 27, Q6_K 103 -> 30.5, Q8_0 151 -> 28; of 4096 x 12288: 56 -> 20, 64 -> 21, 53 -> 28, 81 -> 20.
#include "rmi_common.h"

#include <algorithm>

namespace rmi {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short i16x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;
constexpr int kMaxWgs = 256;   // one workgroup per CU
constexpr int kMaxLds = 160 * 1024;

__device__ __forceinline__ void lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

typedef uint32_t u32x4_b2 __attribute__((ext_vector_type(4), aligned(2)));   // 16 bytes at a 2-byte aligned address

__device__ __forceinline__ long as_long(uint2 v) { return __builtin_bit_cast(long, v); }
__device__ __forceinline__ i32x4 mfma(uint2 x, uint2 w, int c = 0) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(as_long(x), as_long(w), i32x4{c, c, c, c}, 0, 0, 0);
}
// An integer sum v, |v| < 2^22, started at the bits of 1.5 * 2^23 is the float 1.5 * 2^23 + v, and with a whole factor
// f < 2^8 (v f < 2^24) fma(that, f, -1.5 * 2^23 f) is float(v f): the product and the offset are exact, so no rounding.
constexpr float kBiasF = 12582912.0f;
constexpr int kBias = 0x4b400000;
__device__ __forceinline__ float4 lds4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float elem(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// 4 codes times the sub-scale as digits (ingest_gemm.hip): sc (code - 32) + 128 = 256 hi + (lo + 128)
__device__ __forceinline__ void digits4(uint32_t codes, i16x2 scv, i16x2 offs, uint32_t& hi, uint32_t& lo) {
    const i16x2 even = __builtin_bit_cast(i16x2, codes & 0x00ff00ffu);
    const i16x2 odd = __builtin_bit_cast(i16x2, (codes >> 8) & 0x00ff00ffu);
    const uint32_t we = __builtin_bit_cast(uint32_t, even * scv + offs);
    const uint32_t wo = __builtin_bit_cast(uint32_t, odd * scv + offs);
    hi = __builtin_amdgcn_perm(wo, we, 0x07030501u);
    lo = __builtin_amdgcn_perm(wo, we, 0x06020400u) ^ 0x80808080u;
}

// Per type: a unit is 256 elements of a row (a block, or eight Q8_0 blocks), kBytes long; P running sums per output (the
// pairs of a K-quant block, the halves of a Q6_K one, the eight Q8_0 blocks).
template <int TYPE>
struct Fmt;

template <>
struct Fmt<12> {
    static constexpr int P = 4, kBytes = 144;
};
template <>
struct Fmt<13> {
    static constexpr int P = 4, kBytes = 176;
};
template <>
struct Fmt<14> {
    static constexpr int P = 2, kBytes = kQ6KBytes;
};
template <>
struct Fmt<8> {
    static constexpr int P = 8, kBytes = 8 * kQ8_0Bytes;
};

// A wave's 16 rows of a unit: 16-byte pieces, consecutive lanes on consecutive pieces of a row (every cache line is
// requested once; a lane per row and field requests it once per field), parked in the wave's own LDS rows.  The last
// piece of a 210-byte block starts at byte 194.
template <int TYPE>
struct Tile {
    static constexpr int kPieces = (Fmt<TYPE>::kBytes + 15) / 16;
    static constexpr int kLoads = (16 * kPieces + 63) / 64;
    static constexpr int kRow = kPieces * 16;   // LDS bytes per row
    u32x4_b2 v[kLoads];
    __device__ __forceinline__ static int row(int i) { return i / kPieces; }
    // byte offset of piece i (of 16 kPieces) in the matrix relative to the tile's first row and unit
    __device__ __forceinline__ static uint32_t offset(int i, uint32_t rowbytes, int last_row) {
        const int r = row(i), c = i - r * kPieces;
        return static_cast<uint32_t>(min(r, last_row)) * rowbytes + min(16 * c, Fmt<TYPE>::kBytes - 16);
    }
    __device__ __forceinline__ void load(const uint8_t* base, const uint32_t (&off)[kLoads]) {
#pragma unroll
        for (int m = 0; m < kLoads; ++m) v[m] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_b2*>(base + off[m]));
    }
    __device__ __forceinline__ void park(uint8_t* lds, int lane) const {
#pragma unroll
        for (int m = 0; m < kLoads; ++m)
            *reinterpret_cast<uint4*>(lds + 16 * min(lane + 64 * m, 16 * kPieces - 1)) = make_uint4(v[m][0], v[m][1], v[m][2], v[m][3]);
    }
};

// add one unit to the running sums acc[P][4] (columns 4 g + i of the lane's row); d8: its Q8_1 scales
// [block][16], for the K-quants [block][scales 16 | code sums 16].
// SEQ: a Q6_K half-block's sub-blocks in order (the generic kernel), else 0, 2, 1, 3 (the tiled and stream kernels).
template <int TYPE, bool SEQ>
__device__ __forceinline__ void add_unit(const uint8_t* row, const uint2* x, const float* d8, int g,
                                         float (&acc)[Fmt<TYPE>::P][4]) {
    d8 += 4 * g;
    if constexpr (TYPE == 12 || TYPE == 13) {
        constexpr int kQs = TYPE == 13 ? 48 : 16;
        const uint4 h = *reinterpret_cast<const uint4*>(row);
        const float d = half_bits_to_float(h.x & 0xffffu), dmin = half_bits_to_float(h.x >> 16);
        // bytes: scales 0..3 | 4..7, mins 0..3 | 4..7 (ggml get_scale_min_k4)
        const uint32_t s0 = h.y, s1 = h.z, s2 = h.w;
        const uint32_t sc[2] = {s0 & 0x3f3f3f3fu, (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)};
        const uint32_t mn[2] = {s1 & 0x3f3f3f3fu, ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u)};
        uint2 qh = make_uint2(0, 0);
        if constexpr (TYPE == 13) qh = *reinterpret_cast<const uint2*>(row + 16 + 8 * g);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint2 q = *reinterpret_cast<const uint2*>(row + kQs + 32 * p + 8 * g);
            uint2 lo = make_uint2(q.x & 0x0f0f0f0fu, q.y & 0x0f0f0f0fu);
            uint2 hi = make_uint2((q.x >> 4) & 0x0f0f0f0fu, (q.y >> 4) & 0x0f0f0f0fu);
            if constexpr (TYPE == 13) {
                lo.x |= ((qh.x >> (2 * p)) & 0x01010101u) << 4;
                lo.y |= ((qh.y >> (2 * p)) & 0x01010101u) << 4;
                hi.x |= ((qh.x >> (2 * p + 1)) & 0x01010101u) << 4;
                hi.y |= ((qh.y >> (2 * p + 1)) & 0x01010101u) << 4;
            }
            const int j0 = (2 * p) & 3, j1 = j0 + 1;
            const float sc0 = static_cast<float>((sc[p >> 1] >> (8 * j0)) & 0xffu);
            const float sc1 = static_cast<float>((sc[p >> 1] >> (8 * j1)) & 0xffu);
            const float m0 = static_cast<float>((mn[p >> 1] >> (8 * j0)) & 0xffu);
            const float m1 = static_cast<float>((mn[p >> 1] >> (8 * j1)) & 0xffu);
            const i32x4 d0 = mfma(x[2 * p], lo, kBias), d1 = mfma(x[2 * p + 1], hi, kBias);
            const float o0 = -kBiasF * sc0, o1 = -kBiasF * sc1;
            const float* t = d8 + 32 * (2 * p);
            const float4 a = lds4(t), ua = lds4(t + 16), b = lds4(t + 32), ub = lds4(t + 48);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float sumf_d = elem(a, i) * __builtin_fmaf(__int_as_float(d0[i]), sc0, o0);
                sumf_d = __builtin_fmaf(elem(b, i), __builtin_fmaf(__int_as_float(d1[i]), sc1, o1), sumf_d);
                float sumf_m = elem(a, i) * (elem(ua, i) * m0);
                sumf_m = __builtin_fmaf(elem(b, i), elem(ub, i) * m1, sumf_m);
                acc[p][i] += __builtin_fmaf(d, sumf_d, -(dmin * sumf_m));
            }
        }
    } else if constexpr (TYPE == 14) {
        const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(row + 222));   // the last piece's last bytes
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            const uint2 qh = *reinterpret_cast<const uint2*>(row + 128 + 32 * n + 8 * g);
            const uint2 ql[2] = {*reinterpret_cast<const uint2*>(row + 64 * n + 8 * g),
                                 *reinterpret_cast<const uint2*>(row + 64 * n + 32 + 8 * g)};
            const uint2 sw = *reinterpret_cast<const uint2*>(row + 192 + 8 * n);
            const uint32_t scw[4] = {sw.x, sw.x >> 16, sw.y, sw.y >> 16};   // sub-scales 2 k, 2 k + 1 in the low bytes
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int k = SEQ ? kk : ((kk & 1) << 1) | (kk >> 1);
                const int sc = static_cast<int>(static_cast<int8_t>(g & 2 ? scw[k] >> 8 : scw[k]));   // elements 8 g ..
                const short scs = static_cast<short>(sc), ofs = static_cast<short>(128 - 32 * sc);
                const i16x2 scv = {scs, scs}, offs = {ofs, ofs};
                const uint32_t q0 = ((ql[k & 1].x >> (4 * (k >> 1))) & 0x0f0f0f0fu) | (((qh.x >> (2 * k)) & 0x03030303u) << 4);
                const uint32_t q1 = ((ql[k & 1].y >> (4 * (k >> 1))) & 0x0f0f0f0fu) | (((qh.y >> (2 * k)) & 0x03030303u) << 4);
                uint2 hi, lo;
                digits4(q0, scv, offs, hi.x, lo.x);
                digits4(q1, scv, offs, hi.y, lo.y);
                const i32x4 dh = mfma(x[4 * n + k], hi), dl = mfma(x[4 * n + k], lo);
                const float4 a = lds4(d8 + 16 * (4 * n + k));
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s[i] = __builtin_fmaf(elem(a, i), static_cast<float>((dh[i] << 8) + dl[i]), s[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[n][i] = __builtin_fmaf(d, s[i], acc[n][i]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint8_t* b = row + kQ8_0Bytes * j;
            const float dw = half_bits_to_float(*reinterpret_cast<const uint16_t*>(b));
            // the lane's 8 codes: 2-byte aligned, from whole dwords
            const int at = kQ8_0Bytes * j + 2;   // + 8 g
            const uint32_t* q = reinterpret_cast<const uint32_t*>(row + (at & ~3) + 8 * g);
            uint2 c;
            if (at & 2) {
                const uint32_t w0 = q[0], w1 = q[1], w2 = q[2];
                c = make_uint2(__builtin_amdgcn_alignbyte(w1, w0, 2), __builtin_amdgcn_alignbyte(w2, w1, 2));
            } else {
                c = make_uint2(q[0], q[1]);
            }
            const float4 dx = lds4(d8 + 16 * j);
            const i32x4 dd = mfma(x[j], c);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[j][i] = __builtin_fmaf(dw * elem(dx, i), static_cast<float>(dd[i]), acc[j][i]);
        }
    }
}

constexpr int table_row(int type) { return type == 12 || type == 13 ? 32 : 16; }

// units in flight: at most d, a divisor of a tile's n steps (the last units' buffers are free for the next tile's first)
constexpr int depth(int n, int d) { return n % d == 0 ? d : depth(n, d - 1); }

// Activations are staged a slab of 2048 elements (64 Q8_1 blocks) x 16 columns at a time: coalesced into LDS as they
// are, then each lane takes its MFMA operands of the wave's units into registers for the whole launch, and the scales
// go to a table [block][16].  (Operands loaded straight from the columns, 8 bytes per lane 36 bytes apart, cost more
// cache requests than the weights.)
constexpr int kSlabBlocks = 64;
constexpr int kSlabCol = 2 * kSlabBlocks * kQ8_1Bytes / 4 + 8;   // dwords per staged column of a slab pair: 8 banks apart

// NLU: the units that get running sums of their own (unit u adds to those of u % NLU); NS: slabs of 2048 elements (the row
// has at most NS).
template <int TYPE, int NLU, int NS, bool RES>
__global__ __launch_bounds__(64 * kWaves) void cols_gemv_kernel(const uint8_t* __restrict__ w,
                                                                const uint8_t* __restrict__ x, float* y,
                                                                const float* res, float* partials, int n_in, int n_out,
                                                                int ncols, int ntiles) {
    using TL = Tile<TYPE>;
    constexpr int P = Fmt<TYPE>::P, M = NLU / kWaves;
    constexpr int T = table_row(TYPE);             // floats of the scale table per Q8_1 block
    constexpr int kChain = (NS + M - 1) / M;       // units of a leaf, at most
    constexpr int kUnits = kChain * M;             // steps of a tile
    // units in flight per wave (Q6_K at six slabs: two, a third would spill: 4096 x 12288 33 -> 24 us)
    constexpr int D = depth(kUnits, NS == 6 && TYPE == 14 ? 2 : 3);
    static_assert(M == 1 || M == 2 || M == 4, "leaves of a wave");
    constexpr bool SEQ = TYPE == 14 && NLU == 32;
    extern __shared__ __attribute__((aligned(16))) float smem[];   // the scale table; then a slab pair, or sums and tiles
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int nu = n_in / 256, nbq = n_in / 32;
    const uint32_t rowbytes = static_cast<uint32_t>(n_in / 256) * Fmt<TYPE>::kBytes;   // the matrix is below 4 GiB
    float* const area = smem + NS * kSlabBlocks * T;
    uint8_t* const park = reinterpret_cast<uint8_t*>(area + kWaves * P * 256) + wv * 16 * TL::kRow;

    // the wave's i-th unit of a tile in the depth-first order of its leaves: number v of its units in row order (unit
    // 8 v + wv of the row, in leaf v % M), or one past them (an empty step)
    auto number = [](int i) {
        const int q = i / kChain;
        return (M <= 2 ? q : ((q & 1) << 1) | (q >> 1)) + M * (i % kChain);
    };
    const int G = static_cast<int>(gridDim.x);
    int tile = static_cast<int>(blockIdx.x);

    // the slabs (NS even: two at a time), 16-byte pieces, lanes on consecutive pieces of a column; pieces past the row's
    // end re-read its last one and go unused
    uint2 xq[NS * 8];
    uint32_t* slab = reinterpret_cast<uint32_t*>(area);
    constexpr int kColUnits = 2 * kSlabBlocks * kQ8_1Bytes / 16;   // 288 per column of a slab pair
    constexpr int kLoads = 16 * kColUnits / (64 * kWaves);         // 9 per thread
    static_assert(kLoads * 64 * kWaves == 16 * kColUnits && NS % 2 == 0, "whole passes over slab pairs");
    typedef uint32_t u32x4_b4 __attribute__((ext_vector_type(4), aligned(4)));
    u32x4_b4 sv[kLoads];
    const int coldw = nbq * 9;
    auto slab_load = [&](int s) {
#pragma unroll
        for (int m = 0; m < kLoads; ++m) {
            const int i = t + 64 * kWaves * m, c = i / kColUnits, dw = 4 * (s * (kColUnits / 2) + i - c * kColUnits);
            const uint32_t* p = reinterpret_cast<const uint32_t*>(x) + static_cast<size_t>(min(c, ncols - 1)) * coldw;
            sv[m] = *reinterpret_cast<const u32x4_b4*>(p + min(dw, coldw - 4));
        }
    };
    slab_load(0);
    TL wu[D];
    uint32_t off[TL::kLoads];   // of the tile being loaded
    auto set_off = [&](int tile) {
#pragma unroll
        for (int m = 0; m < TL::kLoads; ++m)
            off[m] = TL::offset(min(lane + 64 * m, 16 * TL::kPieces - 1), rowbytes, n_out - 1 - 16 * tile);
    };
    // unit v of the wave (past the row's end: the last whole unit, unused) of tile `tile` into buffer b
    auto fetch = [&](int b, int tile, int v) {
        const int u = min(kWaves * v + wv, nu - 1);
        wu[b].load(w + static_cast<size_t>(tile) * 16 * rowbytes + static_cast<uint32_t>(u) * Fmt<TYPE>::kBytes, off);
    };
    set_off(tile);
#pragma unroll
    for (int b = 0; b < D; ++b)
        if (number(b) < NS) fetch(b, tile, number(b));
#pragma unroll
    for (int s = 0; s < NS; s += 2) {
        if (s * kSlabBlocks < nbq) {   // uniform
            if (s > 0) __syncthreads();   // the previous pair has been read
#pragma unroll
            for (int m = 0; m < kLoads; ++m) {
                const int i = t + 64 * kWaves * m, c = i / kColUnits;
                *reinterpret_cast<uint4*>(slab + c * kSlabCol + 4 * (i - c * kColUnits)) =
                    make_uint4(sv[m][0], sv[m][1], sv[m][2], sv[m][3]);
            }
            if (s + 2 < NS && (s + 2) * kSlabBlocks < nbq) slab_load(s + 2);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint32_t* p = slab + l16 * kSlabCol + ((j * kWaves + wv) * 8 + b) * 9 + 1 + 2 * g;
                    xq[(s + j) * 8 + b] = make_uint2(p[0], p[1]);
                }
            for (int i = t; i < 2 * kSlabBlocks * 16; i += 64 * kWaves) {
                const uint32_t* p = slab + (i & 15) * kSlabCol + (i >> 4) * 9;
                float* row = smem + (s * kSlabBlocks + (i >> 4)) * T + (i & 15);
                row[0] = half_bits_to_float(p[0]);
                if constexpr (T == 32) {
                    int su = 0;
#pragma unroll
                    for (int k = 1; k <= 8; ++k) su = sdot4(static_cast<int>(p[k]), 0x01010101, su);
                    row[16] = static_cast<float>(su);
                }
            }
        }
    }
    __syncthreads();   // the table is complete, and the slabs' area is free

    for (int k = 0; tile < ntiles; ++k, tile += G) {
        const int nt = tile + G;
        // the outputs of this tile belong to 256 of the threads, the two halves taking turns
        const int o = t - 256 * (k & 1);
        const bool mine = o >= 0 && o < 256;
        const int oc = (o >> 4) & 15, orow = 16 * tile + (o & 15);
        const bool live = mine && orow < n_out && oc < ncols;
        const size_t at = static_cast<size_t>(min(oc, ncols - 1)) * n_out + min(orow, n_out - 1);
        float rv = 0.0f;
        if constexpr (RES) rv = res[at];

        float acc[P][4], s0[P][4], s1[P][4], tot[P][4];
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[p][i] = s0[p][i] = s1[p][i] = tot[p][i] = 0.0f;
#pragma unroll
        for (int i = 0; i < kUnits; ++i) {
            const int v = number(i), u = kWaves * v + wv;
            if (v < NS && u < nu) {   // uniform: the row has this unit
                wu[i % D].park(park, lane);
                lds_fence();
                add_unit<TYPE, SEQ>(park + l16 * TL::kRow, &xq[v * 8], smem + u * 8 * T, g, acc);
                asm volatile("" ::: "memory");   // the wave's LDS accesses stay in order
            }
            const int vn = number((i + D) % kUnits);
            if (i + D == kUnits && nt < ntiles) set_off(nt);
            if (vn < NS && (i + D < kUnits || nt < ntiles)) fetch(i % D, i + D < kUnits ? tile : nt, vn);
            if (i % kChain == kChain - 1) {   // a finished leaf joins the butterfly's stack
                const int q = i / kChain;
#pragma unroll
                for (int p = 0; p < P; ++p)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = acc[p][e];
                        acc[p][e] = 0.0f;
                        if (q & 1) {
                            v = s0[p][e] + v;
                            if (q & 2) v = s1[p][e] + v;
                            else s1[p][e] = v;
                        } else {
                            s0[p][e] = v;
                        }
                        if (q == M - 1) tot[p][e] = v;
                    }
            }
        }
        // the next three levels over the waves, then those over the running sums of a unit: [wave][P][lane][4]
        if (k > 0) __syncthreads();   // the previous tile's sums have been read
#pragma unroll
        for (int p = 0; p < P; ++p)
            *reinterpret_cast<float4*>(area + ((wv * P + p) * 64 + lane) * 4) =
                make_float4(tot[p][0], tot[p][1], tot[p][2], tot[p][3]);
        __syncthreads();
        if (mine) {   // whole waves
            float v[P];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                float a[kWaves];
#pragma unroll
                for (int i = 0; i < kWaves; ++i) a[i] = area[((i * P + p) * 64 + 16 * (oc >> 2) + (o & 15)) * 4 + (oc & 3)];
                v[p] = ((a[0] + a[4]) + (a[2] + a[6])) + ((a[1] + a[5]) + (a[3] + a[7]));
            }
#pragma unroll
            for (int h = P / 2; h >= 1; h >>= 1)
#pragma unroll
                for (int i = 0; i < h; ++i) v[i] = v[i] + v[i + h];
            float r = v[0];
            if constexpr (RES) r += rv;
            if (live) y[at] = r;
            if constexpr (RES) {   // squares of four rows in row order
                const float v0 = quad_lane<0>(r), v1 = quad_lane<1>(r), v2 = quad_lane<2>(r), v3 = quad_lane<3>(r);
                if (live && (orow & 3) == 0) {
                    float q = __builtin_fmaf(v0, v0, 0.0f);
                    if (orow + 1 < n_out) q = __builtin_fmaf(v1, v1, q);
                    if (orow + 2 < n_out) q = __builtin_fmaf(v2, v2, q);
                    if (orow + 3 < n_out) q = __builtin_fmaf(v3, v3, q);
                    partials[static_cast<size_t>(oc) * ((n_out + 3) / 4) + orow / 4] = q;
                }
            }
        }
    }
}

template <int TYPE, int NLU, int NS, bool RES>
int launch(const uint8_t* w, const uint8_t* x, float* y, const float* res, float* partials, int n_in, int n_out, int ncols,
           hipStream_t s) {
    constexpr int tiles_bytes = kWaves * (Fmt<TYPE>::P * 1024 + 16 * Tile<TYPE>::kRow);
    constexpr int lds = NS * kSlabBlocks * table_row(TYPE) * 4 + std::max(tiles_bytes, 16 * kSlabCol * 4);
    static_assert(lds <= kMaxLds, "LDS");
    auto k = cols_gemv_kernel<TYPE, NLU, NS, RES>;
    static OncePerDevice attr;
    if (!attr([&] { return lds_limit(k, kMaxLds); })) return fail(RMI_ERR_LAUNCH, "native MMVQ: LDS not available");
    const int tiles = (n_out + 15) / 16, per = (tiles + kMaxWgs - 1) / kMaxWgs;
    hipLaunchKernelGGL(k, dim3((tiles + per - 1) / per), dim3(64 * kWaves), lds, s, w, x, y, res, partials, n_in, n_out, ncols,
                       tiles);
    return launch_status("native_mmvq");
}

template <int TYPE, int NLU>
int pick(const uint8_t* w, const uint8_t* x, float* y, const float* res, float* partials, int n_in, int n_out, int ncols,
         hipStream_t s) {
    auto go = [&](auto plain, auto with_res) {
        return res ? with_res(w, x, y, res, partials, n_in, n_out, ncols, s) : plain(w, x, y, res, partials, n_in, n_out, ncols, s);
    };
    if (n_in <= 4096) return go(launch<TYPE, NLU, 2, false>, launch<TYPE, NLU, 2, true>);
    if (n_in <= 8192) return go(launch<TYPE, NLU, 4, false>, launch<TYPE, NLU, 4, true>);
    return go(launch<TYPE, NLU, 6, false>, launch<TYPE, NLU, 6, true>);
}

// The fewest rows from which this kernel beats passes of at most four columns over the weights.  A launch's time steps
// with its tiles per workgroup (one per 4096 rows) and hardly depends on its columns; a pass's grows with the rows from
// the first one on, so few columns, and few rows of a long row's prologue, stay with the passes.  From grids of 64 to
// 24576 rows (this kernel / the passes, us):
//   Q4_K 6144 wide, 5 columns: 2048 rows 12.6 / 8.9, 7168 17.1 / 17.9; 8 columns: 2048 12.8 / 11.0, 3072 12.9 / 13.5
//   Q4_K 12288 wide, 5 columns: 1024 rows 18.6 / 9.7, 4608 25.5 / 25.1; 12 columns: 1024 18.8 / 17.2, 1280 19.0 / 23.3
//   Q6_K off the streaming shapes, 3 columns: 11008 wide 1024 rows 23.2 / 7.9, 5632 36.3 / 38.2; 1024 wide 2048 rows
//     6.7 / 5.4, 2560 6.8 / 7.0; 8 columns: 11008 wide 1024 rows 23.4 / 19.5, 1280 23.7 / 29.0
//   Q6_K on them: 3 and 4 columns slower everywhere, 8 faster everywhere to 8192 wide
//   Q8_0 12288 wide, 5 columns: 1024 rows 16.5 / 12.8, 1280 16.6 / 19.6; 3 columns: 5120 26.8 / 26.4, 5632 27.0 / 30.3
constexpr int kNever = 1 << 30;
struct Line {
    int max_in;    // rows of at most this length
    int rows[8];   // at 3, 4, .., 9 and 10..12 columns; from 13 on any
};
constexpr Line kLinesK[] = {{1024, {kNever, kNever, 2560, 2560, 1280, 1280, 0, 0}},
                            {2048, {kNever, kNever, 5632, 5632, 2560, 2560, 0, 0}},
                            {4096, {kNever, kNever, 10240, 6144, 5120, 4608, 768, 0}},
                            {10240, {kNever, kNever, 7168, 5632, 3584, 2560, 1280, 1280}},
                            {12288, {kNever, kNever, 4608, 2560, 2560, 2560, 1280, 1280}}};
constexpr Line kLinesQ8[] = {{2048, {kNever, kNever, 5632, 5120, 2560, 2560, 0, 0}},
                             {4096, {10240, 5632, 1280, 1280, 1280, 1280, 0, 0}},
                             {8192, {10240, 5632, 2048, 1280, 1280, 1280, 0, 0}},
                             {12288, {5632, 3584, 1280, 1280, 1280, 1280, 768, 0}}};
constexpr Line kLinesQ6[] = {{1024, {2560, 1280, 0, 0, 0, 0, 0, 0}},   // 64 lanes
                             {2048, {5632, 2560, 0, 0, 0, 0, 0, 0}},
                             {4096, {5632, 2560, 1280, 1280, 0, 0, 0, 0}},
                             {8192, {10240, 4608, 2560, 1536, 1280, 1280, 0, 0}},
                             {12288, {5632, 3584, 1536, 1280, 1280, 1280, 256, 0}}};
constexpr Line kLinesQ6Stream[] = {{2048, {kNever, kNever, kNever, kNever, kNever, 0, 0, 0}},   // 16 lanes
                                   {6144, {kNever, kNever, 512, 0, 0, 0, 0, 0}},
                                   {8192, {kNever, kNever, 2048, 0, 0, 0, 0, 0}},
                                   {12288, {kNever, kNever, kNever, kNever, kNever, kNever, 0, 0}}};

template <int N>
int rows_min(const Line (&lines)[N], int n_in, int ncols) {
    for (const Line& l : lines)
        if (n_in <= l.max_in) return ncols >= 13 ? 0 : l.rows[std::min(ncols, 10) - 3];
    return kNever;
}

int rows_min(int type, int lanes, int n_in, int ncols) {
    if (type == 12 || type == 13) return rows_min(kLinesK, n_in, ncols);
    if (type == 8) return rows_min(kLinesQ8, n_in, ncols);
    return lanes == 16 ? rows_min(kLinesQ6Stream, n_in, ncols) : rows_min(kLinesQ6, n_in, ncols);
}

}  // namespace

int cols_gemv(int type, int lanes, const uint8_t* w, const uint8_t* x, float* y, const float* res, float* partials,
              int n_in, int n_out, int ncols, hipStream_t s) {
    if (ncols > 16 || n_in > 12288 || n_in % 256 ||
        static_cast<uint64_t>(n_out) * (n_in / 32) * kQ8_0Bytes >= (uint64_t(1) << 32))
        return -1;
    if (ncols < 3 || n_out < rows_min(type, lanes, n_in, ncols)) return -1;
    if (type == 12) return pick<12, 16>(w, x, y, res, partials, n_in, n_out, ncols, s);
    if (type == 13) return pick<13, 16>(w, x, y, res, partials, n_in, n_out, ncols, s);
    if (type == 8) return (reinterpret_cast<uintptr_t>(w) & 1) ? -1 : pick<8, 8>(w, x, y, res, partials, n_in, n_out, ncols, s);
    if (lanes == 16) return pick<14, 8>(w, x, y, res, partials, n_in, n_out, ncols, s);
    if (lanes == 64) return pick<14, 32>(w, x, y, res, partials, n_in, n_out, ncols, s);
    return -1;
}

}  // namespace rmi
