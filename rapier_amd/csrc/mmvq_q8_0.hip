// mmvq_q8_0.hip - Q8_0 x Q8_1 GEMV (reference src/native_mmvq.cu: small_q8_dot 835-847, native_small_mmvq_kernel
// 865-900, residual variant 3142-3185) and the GGML-type dispatcher native_mmvq (3787-3818).
//
// One wave64 per output row (q8_0_gemv_kernel: four rows per workgroup); lane l owns Q8_0 blocks l, l + 64, ...  Per block:
// sumi = sum of 8 v_dot4 over the 32 int8 pairs (exact), then acc = fma(d_w * d_x, float(sumi), acc) - the
// reference's d0 * d1 * float(sumi).  Rows are reduced by a fixed 64-lane butterfly, so every column of an
// ncols >= 2 call is bitwise the ncols = 1 result and the residual variant is bitwise plain + res.
#include "rmi_common.h"

namespace rmi {
namespace {

__device__ __forceinline__ uint32_t ldg_u32_b2(const uint8_t* p) {
    const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
    return static_cast<uint32_t>(h[0]) | (static_cast<uint32_t>(h[1]) << 16);
}

// other lanes' LDS writes of this wave have landed
__device__ __forceinline__ void lds_wave_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
// the weights are streamed once
__device__ __forceinline__ uint4 ld_stream(const uint4* p) {
    const u32x4v v = __builtin_nontemporal_load(reinterpret_cast<const u32x4v*>(p));
    return make_uint4(v[0], v[1], v[2], v[3]);
}

template <int NCOLS, bool RES>
__global__ __launch_bounds__(256) void q8_0_gemv_kernel(const uint8_t* __restrict__ w, const uint8_t* __restrict__ x,
                                                        float* y, const float* res, float* partials, int n_in,
                                                        int n_out) {
    __shared__ float vout[NCOLS][4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row = blockIdx.x * 4 + wv;
    const int nb = n_in / 32;
    float acc[NCOLS];
#pragma unroll
    for (int c = 0; c < NCOLS; ++c) acc[c] = 0.0f;
    if (row < n_out) {
        for (int j = lane; j < nb; j += 64) {
            const uint8_t* blk = w + (static_cast<size_t>(row) * nb + j) * kQ8_0Bytes;
            const float dw = half_bits_to_float(*reinterpret_cast<const uint16_t*>(blk));
            int v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = static_cast<int>(ldg_u32_b2(blk + 2 + 4 * i));
#pragma unroll
            for (int c = 0; c < NCOLS; ++c) {
                const uint32_t* xb = reinterpret_cast<const uint32_t*>(x + (static_cast<size_t>(c) * nb + j) * kQ8_1Bytes);
                int sumi = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) sumi = sdot4(v[i], static_cast<int>(xb[1 + i]), sumi);
                acc[c] = __builtin_fmaf(dw * half_bits_to_float(xb[0]), static_cast<float>(sumi), acc[c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NCOLS; ++c) {
        float s = group_sum<64>(acc[c]);
        if (row < n_out) {
            if constexpr (RES) s += res[static_cast<size_t>(c) * n_out + row];
            if (lane == 0) {
                y[static_cast<size_t>(c) * n_out + row] = s;
                vout[c][wv] = s;
            }
        }
    }
    if constexpr (RES) {
        __syncthreads();
        if (threadIdx.x < NCOLS) {
            const int c = threadIdx.x;
            float p = 0.0f;
            for (int i = 0; i < 4; ++i)
                if (blockIdx.x * 4 + i < n_out) p = __builtin_fmaf(vout[c][i], vout[c][i], p);
            partials[static_cast<size_t>(c) * ((n_out + 3) / 4) + blockIdx.x] = p;
        }
    }
}

// One or two columns of larger matrices, rows and columns of whole 16-byte pieces (`staged` below): the same
// lanes, blocks and order as above, so the same bits.  Bound by the weight stream and the chain ahead of it.  A Q8_0
// block is 34 bytes, so the loads above are 17 of two bytes per block and every wave reads the columns again; here a
// wave fetches 128 blocks as 272 consecutive 16-byte pieces into its own LDS area and the columns are staged once per
// workgroup of W rows.  4096 x 4096 with two columns 6.5 -> 5.7 us,
// 4096 x 24576 36.9 -> 23.1 (4.6 TB/s).
constexpr int kStep = 128;                               // blocks of a row per step: two per lane
constexpr int kPieces = kStep * kQ8_0Bytes / 16;         // 272
constexpr int kStagedMax = 64 * 1024;                    // LDS of the staged columns

template <int NCOLS, bool RES, int W>
__global__ __launch_bounds__(64 * W) void q8_0_gemv_staged(const uint4* __restrict__ w, const uint4* __restrict__ x,
                                                           float* y, const float* res, float* partials, int n_in,
                                                           int n_out) {
    extern __shared__ uint4 smem[];   // [W][kPieces] row pieces, then the columns
    __shared__ float vout[NCOLS][W];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row = blockIdx.x * W + wv;
    const int nb = n_in / 32;
    const int rp = nb / 8 * (8 * kQ8_0Bytes / 16);        // pieces of a row
    const int xp = NCOLS * (nb / 8) * (8 * kQ8_1Bytes / 16);
    uint4* area = smem + wv * kPieces;
    uint4* xs = smem + W * kPieces;
    uint4 xin[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) xin[i] = x[min(static_cast<int>(threadIdx.x) + 64 * W * i, xp - 1)];
    const uint4* wrow = w + static_cast<size_t>(min(row, n_out - 1)) * rp;
    // pieces 64 i + lane of a step (the last 16 by four times 16 lanes), clamped to the row: no load under a branch
    uint4 p[5];
    auto fetch = [&](int b0) {
        const int base = b0 / 8 * 17;
#pragma unroll
        for (int i = 0; i < 5; ++i) p[i] = ld_stream(wrow + min(base + 64 * i + (i == 4 ? lane & 15 : lane), rp - 1));
    };
    auto park = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) area[64 * i + lane] = p[i];
        if (lane < 16) area[256 + lane] = p[4];
    };
    fetch(0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (static_cast<int>(threadIdx.x) + 64 * W * i < xp) xs[threadIdx.x + 64 * W * i] = xin[i];
    for (int t = threadIdx.x + 128 * W; t < xp; t += 64 * W) xs[t] = x[t];
    float r[NCOLS];
#pragma unroll
    for (int c = 0; c < NCOLS; ++c) {
        if constexpr (RES) r[c] = res[static_cast<size_t>(c) * n_out + min(row, n_out - 1)];
    }
    park();
    __syncthreads();
    float acc[NCOLS];
#pragma unroll
    for (int c = 0; c < NCOLS; ++c) acc[c] = 0.0f;
    for (int b0 = 0; b0 < nb; b0 += kStep) {
        const bool more = b0 + kStep < nb;   // uniform
        if (more) fetch(b0 + kStep);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = b0 + 64 * h + lane;
            if (j < nb) {
                // block at byte 34 (64 h + lane): nine aligned dwords hold it, shifted by half a dword where that is even
                const int blk = 64 * h + lane;
                const uint32_t* q = reinterpret_cast<const uint32_t*>(area) + (kQ8_0Bytes * blk >> 2);
                uint32_t dws[9];
#pragma unroll
                for (int i = 0; i < 9; ++i) dws[i] = q[i];
                const bool odd = blk & 1;
                const float dw = half_bits_to_float(odd ? dws[0] >> 16 : dws[0] & 0xffffu);
                int v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    v[i] = static_cast<int>(__builtin_amdgcn_alignbyte(dws[i + 1], odd ? dws[i + 1] : dws[i], odd ? 0 : 2));
#pragma unroll
                for (int c = 0; c < NCOLS; ++c) {
                    const uint32_t* xb = reinterpret_cast<const uint32_t*>(xs) + 9 * (c * nb + j);
                    int sumi = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) sumi = sdot4(v[i], static_cast<int>(xb[1 + i]), sumi);
                    acc[c] = __builtin_fmaf(dw * half_bits_to_float(xb[0]), static_cast<float>(sumi), acc[c]);
                }
            }
        }
        if (more) {
            lds_wave_sync();   // every lane has read this step's pieces
            park();
            lds_wave_sync();
        }
    }
#pragma unroll
    for (int c = 0; c < NCOLS; ++c) {
        float s = group_sum<64>(acc[c]);
        if constexpr (RES) s += r[c];
        if (row < n_out && lane == 0) {
            y[static_cast<size_t>(c) * n_out + row] = s;
            vout[c][wv] = s;
        }
    }
    if constexpr (RES) {
        __syncthreads();
        if (threadIdx.x < NCOLS * (W / 4)) {
            const int c = threadIdx.x / (W / 4), g = threadIdx.x - c * (W / 4), r0 = blockIdx.x * W + 4 * g;
            if (r0 < n_out) {
                float q = 0.0f;
                for (int i = 0; i < 4; ++i)
                    if (r0 + i < n_out) q = __builtin_fmaf(vout[c][4 * g + i], vout[c][4 * g + i], q);
                partials[static_cast<size_t>(c) * ((n_out + 3) / 4) + r0 / 4] = q;
            }
        }
    }
}

template <int NCOLS, bool RES, int W>
int launch_staged(const uint8_t* w, const uint8_t* x, float* y, const float* res, float* partials, int n_in, int n_out,
                  hipStream_t s) {
    // the columns' LDS limit and the row areas together exceed the default 64 KB
    static OncePerDevice attr;
    if (!attr([] { return lds_limit(q8_0_gemv_staged<NCOLS, RES, W>, W * kPieces * 16 + kStagedMax); }))
        return fail(RMI_ERR_LAUNCH, "native_q8_0_mmvq: LDS not available");
    const size_t lds = static_cast<size_t>(W) * kPieces * 16 + static_cast<size_t>(NCOLS) * (n_in / 32) * kQ8_1Bytes;
    hipLaunchKernelGGL((q8_0_gemv_staged<NCOLS, RES, W>), dim3((n_out + W - 1) / W), dim3(64 * W), lds, s,
                       reinterpret_cast<const uint4*>(w), reinterpret_cast<const uint4*>(x), y, res, partials, n_in, n_out);
    return launch_status("native_q8_0_mmvq");
}

// W: as many rows per workgroup as leave a workgroup for each of the 256 CUs
template <int NCOLS, bool RES>
int launch_staged(const uint8_t* w, const uint8_t* x, float* y, const float* res, float* partials, int n_in, int n_out,
                  hipStream_t s) {
    if (n_out >= 16 * 256) return launch_staged<NCOLS, RES, 16>(w, x, y, res, partials, n_in, n_out, s);
    if (n_out >= 8 * 256) return launch_staged<NCOLS, RES, 8>(w, x, y, res, partials, n_in, n_out, s);
    return launch_staged<NCOLS, RES, 4>(w, x, y, res, partials, n_in, n_out, s);
}

// Matrices the staged kernel takes: whole aligned pieces, the columns within their LDS, rows of half a step or more, and
// more than 10M elements.  Below that the two-byte loads are faster, their chain being shorter (no LDS behind the loads):
// 2048 x 4096 3.8 us against 4.3, 12288 x 512 4.6 / 5.1; above it 4096 x 3072 6.6 / 5.1, 12288 x 1024 6.6 / 5.8,
// 4096 x 24576 33.2 / 21.4 (one column; two columns alike).  Short rows leave its lanes idle: 512 x 16384 5.6 / 7.3.
// At 2048 wide the line is 11M: 4900 rows (10.0M) 4.9 / 5.1, 5632 (11.5M) 5.5 / 5.2.  As the last pass of a call of more
// columns (`behind`) it finds the weights in the caches, which the two-byte loads use better where workgroups or steps are
// few: the whole call of five columns 2048 x 4900 10.4 / 11.7, 10240 x 1024 11.3 / 11.7, 20480 x 1024 (six) 19.6 / 20.0,
// but 8192 x 1300 14.3 / 13.7, 12288 x 1279 19.8 / 18.6, 20480 x 4096 56.2 / 53.8.
bool staged(const uint8_t* w, const uint8_t* x, int n_in, int n_out, int ncols, bool behind) {
    return n_in >= 2048 && n_in % 256 == 0 && static_cast<int64_t>(n_in) * n_out > (n_in > 2048 ? 10000000 : 11000000) &&
           (!behind || (n_in >= 4096 && n_out >= 1280)) && aligned16(w) && aligned16(x) &&
           static_cast<int64_t>(ncols) * (n_in / 32) * kQ8_1Bytes <= kStagedMax;
}

template <bool RES>
int launch(const void* wv, const void* xv, float* y, const float* res, float* partials, int n_in, int n_out,
           int ncols, hipStream_t s, bool behind = false) {
    const auto* w = static_cast<const uint8_t*>(wv);
    const auto* x = static_cast<const uint8_t*>(xv);
    const dim3 grid((n_out + 3) / 4), block(256);
    if (ncols > 2)
        if (const int rc = cols_gemv(8, 64, w, x, y, res, partials, n_in, n_out, ncols, s); rc >= 0)
            return rc;
    if (ncols <= 2 && staged(w, x, n_in, n_out, ncols, behind))
        return ncols == 1 ? launch_staged<1, RES>(w, x, y, res, partials, n_in, n_out, s)
                          : launch_staged<2, RES>(w, x, y, res, partials, n_in, n_out, s);
    if (ncols > 4) {
        const size_t xcol = static_cast<size_t>(n_in / 32) * kQ8_1Bytes;
        const size_t pcol = static_cast<size_t>((n_out + 3) / 4);
        for (int j = 0; j < ncols; j += 4) {
            const int nj = ncols - j < 4 ? ncols - j : 4;
            const int rc = launch<RES>(w, x + j * xcol, y + static_cast<size_t>(j) * n_out,
                                       RES ? res + static_cast<size_t>(j) * n_out : nullptr,
                                       RES ? partials + j * pcol : nullptr, n_in, n_out, nj, s, j > 0);
            if (rc != RMI_OK) return rc;
        }
        return RMI_OK;
    }
    switch (ncols) {
        case 1: hipLaunchKernelGGL((q8_0_gemv_kernel<1, RES>), grid, block, 0, s, w, x, y, res, partials, n_in, n_out); break;
        case 2: hipLaunchKernelGGL((q8_0_gemv_kernel<2, RES>), grid, block, 0, s, w, x, y, res, partials, n_in, n_out); break;
        case 3: hipLaunchKernelGGL((q8_0_gemv_kernel<3, RES>), grid, block, 0, s, w, x, y, res, partials, n_in, n_out); break;
        default: hipLaunchKernelGGL((q8_0_gemv_kernel<4, RES>), grid, block, 0, s, w, x, y, res, partials, n_in, n_out); break;
    }
    return launch_status("native_q8_0_mmvq");
}

int validate(const void* w, const void* x, const float* y, int n_in, int n_out, int ncols, void* stream) {
    if (n_in <= 0 || n_in % 32 != 0)
        return fail(RMI_ERR_SHAPE, "native MMVQ requires n_in > 0 and divisible by its block element count");
    if (ncols < 1 || ncols > kMaxCols) return fail(RMI_ERR_SHAPE, "native MMVQ requires 1 <= ncols <= 16");
    if (n_out <= 0) return fail(RMI_ERR_SHAPE, "native MMVQ requires n_out > 0");
    if (!aligned4(w) || !aligned4(x) || !aligned4(y))
        return fail(RMI_ERR_POINTER, "native MMVQ requires non-null 4-byte aligned device pointers");
    if (!stream) return fail(RMI_ERR_STREAM, "native MMVQ requires an explicit non-null CUDA stream");
    return RMI_OK;
}

}  // namespace
}  // namespace rmi

using namespace rmi;

extern "C" int rmi_native_q8_0_mmvq(const void* w, const void* x_q8_1, float* y, int n_in, int n_out, int ncols,
                                    void* stream) {
    if (int rc = validate(w, x_q8_1, y, n_in, n_out, ncols, stream)) return rc;
    return launch<false>(w, x_q8_1, y, nullptr, nullptr, n_in, n_out, ncols, static_cast<hipStream_t>(stream));
}

extern "C" int rmi_native_q8_0_mmvq_res_n(const void* w, const void* x_q8_1, float* y, const float* res,
                                          float* partials, int n_in, int n_out, int ncols, void* stream) {
    if (int rc = validate(w, x_q8_1, y, n_in, n_out, ncols, stream)) return rc;
    if (!aligned4(res) || !aligned4(partials))
        return fail(RMI_ERR_POINTER, "native MMVQ requires non-null 4-byte aligned device pointers");
    return launch<true>(w, x_q8_1, y, res, partials, n_in, n_out, ncols, static_cast<hipStream_t>(stream));
}

extern "C" int rmi_native_q8_0_mmvq_res(const void* w, const void* x_q8_1, float* y, const float* res,
                                        float* partials, int n_in, int n_out, void* stream) {
    return rmi_native_q8_0_mmvq_res_n(w, x_q8_1, y, res, partials, n_in, n_out, 1, stream);
}

extern "C" int rmi_native_mmvq_supported(int ggml_type) {
    return ggml_type == 14 || ggml_type == 13 || ggml_type == 12 || ggml_type == 8;
}

extern "C" size_t rmi_native_mmvq_weight_bytes(int ggml_type, int n_in, int n_out) {
    int elems, bytes;
    if (ggml_type == 14) { elems = 256; bytes = kQ6KBytes; }
    else if (ggml_type == 13) { elems = 256; bytes = 176; }
    else if (ggml_type == 12) { elems = 256; bytes = 144; }
    else if (ggml_type == 8) { elems = 32; bytes = kQ8_0Bytes; }
    else { set_error("unsupported native MMVQ GGML type"); return 0; }
    if (n_in <= 0 || n_in % elems != 0 || n_out <= 0) {
        set_error("native MMVQ requires n_in > 0 and divisible by its block element count");
        return 0;
    }
    return static_cast<size_t>(n_in / elems) * bytes * static_cast<size_t>(n_out);
}

extern "C" int rmi_native_q6_k_mmvq(const void*, const void*, float*, int, int, int, void*);
extern "C" int rmi_native_q5_k_mmvq(const void*, const void*, float*, int, int, int, void*);
extern "C" int rmi_native_q4_k_mmvq(const void*, const void*, float*, int, int, int, void*);

extern "C" int rmi_native_mmvq(int ggml_type, const void* w, const void* x_q8_1, float* y, int n_in, int n_out,
                               int ncols, void* stream) {
    // more than 16 columns: passes of 16 over the same weights (each column unchanged), as the reference does
    if (ncols > kMaxCols) {
        const size_t xcol = static_cast<size_t>(n_in / 32) * kQ8_1Bytes;
        for (int j = 0; j < ncols; j += kMaxCols) {
            const int nj = ncols - j < kMaxCols ? ncols - j : kMaxCols;
            const int rc = rmi_native_mmvq(ggml_type, w, static_cast<const uint8_t*>(x_q8_1) + j * xcol,
                                           y + static_cast<size_t>(j) * n_out, n_in, n_out, nj, stream);
            if (rc != RMI_OK) return rc;
        }
        return RMI_OK;
    }
    if (ggml_type == 14) return rmi_native_q6_k_mmvq(w, x_q8_1, y, n_in, n_out, ncols, stream);
    if (ggml_type == 13) return rmi_native_q5_k_mmvq(w, x_q8_1, y, n_in, n_out, ncols, stream);
    if (ggml_type == 12) return rmi_native_q4_k_mmvq(w, x_q8_1, y, n_in, n_out, ncols, stream);
    if (ggml_type == 8) return rmi_native_q8_0_mmvq(w, x_q8_1, y, n_in, n_out, ncols, stream);
    return fail(RMI_ERR_UNSUPPORTED, "unsupported native MMVQ GGML type");
}
