// ingest_gemm.hip - packed Q6_K x Q8_1 GEMM for whole prompts (17 columns and more) on the int8 matrix cores, gfx950.
//
// Reference behaviour: the row-batched ingest GEMMs (src/qwythos_ingest.cu; native_mmvq IL kernels, mmvq:1625-2310).
//
// Every output has the bits of the single-column packed GEMV (mmvq_q6k_packed.hip), so the order of its fp32 operations
// is the GEMV's: per half-block (128 elements, 16 of them in a 2048-element chunk) acc = fma(d8, float(s), acc) over the
// four Q8_1 blocks k = 0, 2, 1, 3 with s the exact integer sc_lo * dot_lo + sc_hi * dot_hi, then tot_p = fma(d, acc,
// tot_p) over the chunks for each half-block position p, then the xor butterfly over the 16 positions.
//  * The integer.  sc * (code - 32) fits 14 bits, so it is cut into two int8 digits (256 hi + lo) when a weight is
//    unpacked, and s = (hi . x << 8) + lo . x is two 32x32x32 int8 MFMAs (K = one Q8_1 block) and one shift-add per
//    output, where applying the sub-scales after the MFMA would take a K = 16 product per sub-block and per-row scale
//    operands on the vector unit.
//  * The order.  A workgroup walks the half-block positions in the butterfly's depth-first order (0, 8, 4, 12, ...) and
//    runs a position's chunks back to back, so one tot and a stack of three partial sums per output stand for the 16
//    running sums.  Two wave groups take the even and the odd positions (the butterfly's last addition joins them).
//  * Tile: 64 rows x 128 columns, 8 waves: group (even / odd positions) x 32 rows x 64 columns.  A weight is unpacked
//    once per 128 columns.  A step is one half-block of the tile: 64 rows' codes as digits (16 KB) and 128 columns'
//    codes (16 KB) per group, double-buffered in LDS; the next step's loads (the columns straight into LDS) fly during
//    the MFMAs.
//  * Bound: the vector unit, 71% busy (two waves per SIMD; they wait 35% of their cycles). Per 32x32x32 cell 85 vector
//    instructions (340 cycles of a SIMD) against 64 cycles of MFMA: a shift-add, a convert and an fma per output and Q8_1
//    block are 48 of them, the rest unpacks weights (once per 128 columns), folds and moves.  24576 x 4096 at 1024 columns:
//    642 us (0.32 Pop/s) where 64 passes of the 16-column kernel take 1690 us; 4096 x 12288: 300 us (64 x 22.4).
//  * A tile costs the same whatever its columns (24576 x 4096: 107 us at 1..128, four 16-column passes 104), and matrices
//    of 4096 rows fill 64 CUs per 128 columns.  Over all matrices of the 9B model it wins from 64 columns (15.1 ms for a
//    64-token prompt, 16.0 in 16-column passes; 128 tokens 16.1 / 31.2).
#include "rmi_common.h"
#include "ingest.h"

#include <algorithm>

namespace rmi {
namespace {

constexpr int kTileRows = 64;
constexpr int kTileCols = kIngestColTile;
constexpr int kGemmThreads = 512;
constexpr int kWaveTileBytes = 4 * 8 * kQ6KBytes;   // 6720: one (quad, chunk) of the packed layout

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef short i16x2 __attribute__((ext_vector_type(2)));

// one group's half-block step in LDS
struct Step {
    u32x4 a[4 * 2 * 2 * kTileRows];   // [block k][half o][digit hi | lo][row]: 16 digits
    u32x4 b[4 * 2 * kTileCols];       // [block k][half o][column]: 16 codes
    float d8[4 * kTileCols];          // [block k][column]
    float d[kTileRows];               // the rows' block scale
};

// a thread's weights of a step: 16 ql bytes (two sub-block halves), their 16 qh bytes, the 8 sub-scales, the block scale
struct WLoad {
    u32x4 ql, qh;
    uint2 sc;
    uint32_t d;
};

// 4 codes (bytes) times the sub-scale (both halves of scv; offs = 128 - 32 sc) as digits: w + 128 = 256 hi + (lo + 128)
__device__ __forceinline__ void digits4(uint32_t codes, i16x2 scv, i16x2 offs, uint32_t& hi, uint32_t& lo) {
    const i16x2 even = __builtin_bit_cast(i16x2, codes & 0x00ff00ffu);
    const i16x2 odd = __builtin_bit_cast(i16x2, (codes >> 8) & 0x00ff00ffu);
    const uint32_t we = __builtin_bit_cast(uint32_t, even * scv + offs);
    const uint32_t wo = __builtin_bit_cast(uint32_t, odd * scv + offs);
    hi = __builtin_amdgcn_perm(wo, we, 0x07030501u);                  // bytes we.1 wo.1 we.3 wo.3
    lo = __builtin_amdgcn_perm(wo, we, 0x06020400u) ^ 0x80808080u;
}

__device__ __forceinline__ i16x2 dup16(int v) { return i16x2{static_cast<short>(v), static_cast<short>(v)}; }

__device__ __forceinline__ int sub_scale(uint2 sc, int i) {
    const uint32_t w = i < 4 ? sc.x : sc.y;
    return static_cast<int>(static_cast<int8_t>(w >> (8 * (i & 3))));
}

__device__ __forceinline__ void load16_to_lds(const void* g, void* l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) g,
                                     (__attribute__((address_space(3))) void*) l, 16, 0, 0);
}
__device__ __forceinline__ void load4_to_lds(const void* g, void* l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) g,
                                     (__attribute__((address_space(3))) void*) l, 4, 0, 0);
}

template <bool RES>
__global__ __launch_bounds__(kGemmThreads) void q6k_ingest_gemm(const uint8_t* __restrict__ wp,
                                                                const u32x4* __restrict__ xc,
                                                                const float* __restrict__ xd, float* y,
                                                                const float* res, float* partials, int n_in, int n_out,
                                                                int ncols, int tpad, int ct) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int grp = wv >> 2, wr = wv & 1, wc = (wv >> 1) & 1;
    const int tg = t & 255;
    const int nch = n_in / 2048;
    const int nq = (n_out + 3) / 4;
    // tile of this workgroup: the XCDs (workgroups round robin) take contiguous ranges, columns innermost, so the
    // workgroups of an XCD share their rows' weights in its L2
    const int total = static_cast<int>(gridDim.x);
    const int per = (total + 7) / 8;
    const int b = static_cast<int>(blockIdx.x);
    const int full = total - (per - 1) * 8;   // XCDs with `per` workgroups (the others per - 1)
    const int xcd = b & 7;
    const int tile = xcd * (per - 1) + min(xcd, full) + (b >> 3);
    const int row0 = (tile / ct) * kTileRows, col0 = (tile % ct) * kTileCols;

    Step* const st = reinterpret_cast<Step*>(smem) + 2 * grp;

    const int ar = tg & 63, au = tg >> 6;   // row of the tile and 16-byte unit this thread unpacks
    const size_t qbase = static_cast<size_t>(min(row0 / 4 + (ar >> 2), nq - 1)) * nch;
    // half-block positions of this group in the butterfly's order: grp + {0, 8, 4, 12, 2, 10, 6, 14}
    auto position = [&](int leaf) { return grp + ((leaf & 1) << 3) + ((leaf & 2) << 1) + ((leaf & 4) >> 1); };

    auto load_w = [&](int p, int c, WLoad& w) {
        const uint8_t* base = wp + (qbase + c) * kWaveTileBytes;
        const int l = 4 * p + (ar & 3);
        w.ql = *reinterpret_cast<const u32x4*>(base + au * 1024 + 16 * l);
        w.qh = *reinterpret_cast<const u32x4*>(base + 4096 + (au & 1) * 1024 + 16 * l);
        w.sc = *reinterpret_cast<const uint2*>(base + 6144 + 8 * l);
        w.d = *reinterpret_cast<const uint16_t*>(base + 6656 + 2 * (4 * (p >> 1) + (ar & 3)));
    };
    auto load_x = [&](int p, int c, Step& s) {
        const int j0 = 64 * c + 4 * p, w4 = tg >> 6;
#pragma unroll
        for (int m = 0; m < 4; ++m) {   // 1024 16-byte units, 64 consecutive columns per wave and pass
            const int ko = 2 * m + (w4 >> 1), cc = 64 * (w4 & 1);
            load16_to_lds(xc + static_cast<size_t>(2 * j0 + ko) * tpad + col0 + cc + lane, s.b + ko * kTileCols + cc);
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int k = 2 * m + (w4 >> 1), cc = 64 * (w4 & 1);
            load4_to_lds(xd + static_cast<size_t>(j0 + k) * tpad + col0 + cc + lane, s.d8 + k * kTileCols + cc);
        }
    };
    auto unpack = [&](const WLoad& w, Step& s) {
        const int o = au & 1, k0 = au >> 1;   // low nibbles: sub-block k0, high nibbles: k0 + 2
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = k0 + 2 * h;
            const int sc = sub_scale(w.sc, 2 * k + o);
            const i16x2 scv = dup16(sc), offs = dup16(128 - 32 * sc);
            u32x4 hi, lo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t codes = ((w.ql[i] >> (4 * h)) & 0x0f0f0f0fu) | (((w.qh[i] >> (2 * k)) & 0x03030303u) << 4);
                uint32_t dh, dl;
                digits4(codes, scv, offs, dh, dl);
                hi[i] = dh;
                lo[i] = dl;
            }
            s.a[((2 * k + o) * 2 + 0) * kTileRows + ar] = hi;
            s.a[((2 * k + o) * 2 + 1) * kTileRows + ar] = lo;
        }
        if (au == 0) s.d[ar] = half_bits_to_float(w.d);
    };

    float tot[2][16], l0[2][16], l1[2][16], l2[2][16];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) tot[n][i] = l0[n][i] = l1[n][i] = l2[n][i] = 0.0f;

    const int lr = lane & 31, lh = lane >> 5;
    auto compute = [&](const Step& s) {
        float acc[2][16];
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][i] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const int k = ((kk & 1) << 1) | (kk >> 1);   // 0, 2, 1, 3: the GEMV's order
            const i32x4 ah = __builtin_bit_cast(i32x4, s.a[((2 * k + lh) * 2 + 0) * kTileRows + 32 * wr + lr]);
            const i32x4 al = __builtin_bit_cast(i32x4, s.a[((2 * k + lh) * 2 + 1) * kTileRows + 32 * wr + lr]);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int col = 64 * wc + 32 * n + lr;
                const i32x4 bx = __builtin_bit_cast(i32x4, s.b[(2 * k + lh) * kTileCols + col]);
                const float d8 = s.d8[k * kTileCols + col];
                i32x16 zero = {};
                const i32x16 dh = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah, bx, zero, 0, 0, 0);
                const i32x16 dl = __builtin_amdgcn_mfma_i32_32x32x32_i8(al, bx, zero, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    acc[n][i] = __builtin_fmaf(d8, static_cast<float>((dh[i] << 8) + dl[i]), acc[n][i]);
            }
        }
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            const float4 dv = *reinterpret_cast<const float4*>(s.d + 32 * wr + 8 * i4 + 4 * lh);
            const float dr[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) tot[n][4 * i4 + e] = __builtin_fmaf(dr[e], acc[n][4 * i4 + e], tot[n][4 * i4 + e]);
        }
    };
    // fold a finished position into the butterfly's stack (leaf odd: joins its partner; and so on up)
    auto fold = [&](int leaf) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float v = tot[n][i];
                if (!(leaf & 1)) {
                    l0[n][i] = v;
                } else {
                    v = l0[n][i] + v;
                    if (!(leaf & 2)) {
                        l1[n][i] = v;
                    } else {
                        v = l1[n][i] + v;
                        l2[n][i] = leaf & 4 ? l2[n][i] + v : v;
                    }
                }
                tot[n][i] = 0.0f;
            }
    };

    WLoad w;
    load_w(position(0), 0, w);
    load_x(position(0), 0, st[0]);
    unpack(w, st[0]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the columns' loads into LDS
    __syncthreads();

    const int nsteps = 8 * nch;
    int leaf = 0, c = 0;
    for (int s = 0; s < nsteps; ++s) {
        const bool more = s + 1 < nsteps;
        const bool last_chunk = c == nch - 1;
        const int nleaf = last_chunk ? leaf + 1 : leaf, nc = last_chunk ? 0 : c + 1;
        Step& nxt = st[(s + 1) & 1];
        if (more) {
            load_w(position(nleaf), nc, w);
            load_x(position(nleaf), nc, nxt);
        }
        compute(st[s & 1]);
        if (last_chunk) fold(leaf);
        if (more) {
            unpack(w, nxt);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();
        leaf = nleaf;
        c = nc;
    }

    // join the even and odd positions through LDS, [column][row] with four floats of pad per column
    constexpr int kPitch = kTileRows + 4;
    float* out = reinterpret_cast<float*>(smem);
    auto slot = [&](int n, int i4) { return out + (64 * wc + 32 * n + lr) * kPitch + 32 * wr + 8 * i4 + 4 * lh; };
    if (grp == 1) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
                *reinterpret_cast<float4*>(slot(n, i4)) =
                    make_float4(l2[n][4 * i4], l2[n][4 * i4 + 1], l2[n][4 * i4 + 2], l2[n][4 * i4 + 3]);
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                float4* p = reinterpret_cast<float4*>(slot(n, i4));
                const float4 o = *p;
                *p = make_float4(l2[n][4 * i4] + o.x, l2[n][4 * i4 + 1] + o.y, l2[n][4 * i4 + 2] + o.z,
                                 l2[n][4 * i4 + 3] + o.w);
            }
    }
    __syncthreads();
    // 16 threads per column, four rows each
    const int np = nq;
    const bool vec = n_out % 4 == 0;
    for (int i = t; i < kTileCols * (kTileRows / 4); i += kGemmThreads) {
        const int cc = i >> 4, rq = i & 15;
        const int col = col0 + cc, row = row0 + 4 * rq;
        if (col >= ncols || row >= n_out) continue;
        const float4 v4 = *reinterpret_cast<const float4*>(out + cc * kPitch + 4 * rq);
        float v[4] = {v4.x, v4.y, v4.z, v4.w};
        const size_t o = static_cast<size_t>(col) * n_out + row;
        if (vec) {
            if constexpr (RES) {
                const float4 r = *reinterpret_cast<const float4*>(res + o);
                v[0] += r.x;
                v[1] += r.y;
                v[2] += r.z;
                v[3] += r.w;
            }
            *reinterpret_cast<float4*>(y + o) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (row + e < n_out) {
                    if constexpr (RES) v[e] += res[o + e];
                    y[o + e] = v[e];
                }
        }
        if constexpr (RES) {   // squares of the quad's rows in row order
            float p = __builtin_fmaf(v[0], v[0], 0.0f);
#pragma unroll
            for (int e = 1; e < 4; ++e)
                if (row + e < n_out) p = __builtin_fmaf(v[e], v[e], p);
            partials[static_cast<size_t>(col) * np + row / 4] = p;
        }
    }
}

// Q8_1 columns as the GEMM's operand: codes [block][half][column] in 16-byte units and scales [block][column], columns
// padded with zeros to the column tile.  Four adjacent blocks of 64 columns per workgroup (a column's 144 bytes share
// cache lines).
__global__ __launch_bounds__(256) void ingest_operand_kernel(const uint8_t* __restrict__ x, u32x4* __restrict__ xc,
                                                             float* __restrict__ xd, int nbt, int ncols, int tpad) {
    const int col = static_cast<int>(blockIdx.x) * 64 + (threadIdx.x & 63);
    const int j = static_cast<int>(blockIdx.y) * 4 + (threadIdx.x >> 6);
    if (j >= nbt) return;
    uint32_t v[9];
    const uint32_t* p = reinterpret_cast<const uint32_t*>(x + (static_cast<size_t>(min(col, ncols - 1)) * nbt + j) * kQ8_1Bytes);
#pragma unroll
    for (int i = 0; i < 9; ++i) v[i] = col < ncols ? p[i] : 0u;
    xc[static_cast<size_t>(2 * j) * tpad + col] = u32x4{v[1], v[2], v[3], v[4]};
    xc[static_cast<size_t>(2 * j + 1) * tpad + col] = u32x4{v[5], v[6], v[7], v[8]};
    xd[static_cast<size_t>(j) * tpad + col] = half_bits_to_float(v[0]);
}

int padded(int ncols) { return (ncols + kTileCols - 1) / kTileCols * kTileCols; }

}  // namespace

size_t ingest_operand_bytes(int n_in, int ncols) { return static_cast<size_t>(n_in / 32) * padded(ncols) * 36; }

int q6k_packed_gemm(const void* w_packed, const void* x_q8_1, float* y, const float* res, float* partials, int n_in,
                    int n_out, int ncols, void* ws, hipStream_t s) {
    const int tpad = padded(ncols), nbt = n_in / 32;
    auto* xc = static_cast<u32x4*>(ws);
    auto* xd = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + static_cast<size_t>(nbt) * tpad * 32);
    hipLaunchKernelGGL(ingest_operand_kernel, dim3(tpad / 64, (nbt + 3) / 4), dim3(256), 0, s,
                       static_cast<const uint8_t*>(x_q8_1), xc, xd, nbt, ncols, tpad);
    RMI_TRY(launch_status("q6_k_gemm_packed"));
    constexpr int lds = 4 * static_cast<int>(sizeof(Step));
    static OncePerDevice attr;
    if (!attr([] { return lds_limit(q6k_ingest_gemm<true>, lds) && lds_limit(q6k_ingest_gemm<false>, lds); }))
        return fail(RMI_ERR_LAUNCH, "q6_k_gemm_packed: LDS not available");
    const int ct = tpad / kTileCols, rt = (n_out + kTileRows - 1) / kTileRows;
    const auto* wp = static_cast<const uint8_t*>(w_packed);
    if (res)
        hipLaunchKernelGGL(q6k_ingest_gemm<true>, dim3(rt * ct), dim3(kGemmThreads), lds, s, wp, xc, xd, y, res, partials,
                           n_in, n_out, ncols, tpad, ct);
    else
        hipLaunchKernelGGL(q6k_ingest_gemm<false>, dim3(rt * ct), dim3(kGemmThreads), lds, s, wp, xc, xd, y, nullptr,
                           nullptr, n_in, n_out, ncols, tpad, ct);
    return launch_status("q6_k_gemm_packed");
}

}  // namespace rmi

using namespace rmi;

extern "C" size_t rmi_q6_k_gemm_workspace_bytes(int n_in, int ncols) {
    if (n_in <= 0 || n_in % 2048 != 0 || ncols < 1) {
        set_error("q6_k_gemm_workspace_bytes: n_in must be a positive multiple of 2048, ncols positive");
        return 0;
    }
    return ingest_operand_bytes(n_in, ncols);
}

extern "C" int rmi_q6_k_gemm_packed(const void* w_packed, const void* x_q8_1, float* y, const float* res,
                                    float* partials, int n_in, int n_out, int ncols, void* ws, void* stream) {
    if (n_in <= 0 || n_in % 2048 != 0 || n_out <= 0 || ncols < 1 || ncols > kIngestMaxCols)
        return fail(RMI_ERR_SHAPE, "q6_k_gemm_packed: n_in must be a positive multiple of 2048, 1 <= ncols <= 4096");
    if (!aligned16(w_packed) || !aligned4(x_q8_1) || !aligned16(y) || !aligned16(ws) ||
        (res && (!aligned16(res) || !aligned4(partials))))
        return fail(RMI_ERR_POINTER, "q6_k_gemm_packed: null or misaligned pointer");
    if (!stream) return fail(RMI_ERR_STREAM, "native MMVQ requires an explicit non-null CUDA stream");
    return q6k_packed_gemm(w_packed, x_q8_1, y, res, partials, n_in, n_out, ncols, ws, static_cast<hipStream_t>(stream));
}
