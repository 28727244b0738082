// topk.hip - the k largest logits (k <= 64) with their token ids, on the device: the per-token list the serve protocol
// prints (reference qw:2513-2531, topk_out: a host scan over all n logits keeping the k largest in descending order; an
// incoming logit must be strictly greater than the current k-th to displace it, so among equal logits the lower id
// ranks first and is kept).  Here each logit becomes a 64-bit key (order-preserving float bits with -0 folded into +0,
// then the inverted id), all keys are distinct, and the list is the k largest keys in descending order: the same
// (logit descending, id ascending) order.
//
// Two launches.  The lists, from k = 17 on, come from bitonic networks whose lanes hold the keys (compile-time lane
// strides, VALU exchanges).  topk_lists: a wave takes 256 consecutive logits at a time, four keys per lane, sorts each of
// the four 64-key registers across its lanes (21 exchanges, the four independent of one another), and merges them and its
// list so far into the 64 largest; the eight waves of a workgroup then merge theirs.  Up to k = 16, topk_pop: each lane
// sorts its keys in registers and k rounds of a wave-wide maximum pop the wave's list, ~0.21 us a round.
// topk_merge: one workgroup of 16 waves; each loads eight workgroup lists and merges them in registers, and the 16 results
// meet in LDS four to a wave (topk_merge_few: up to eight lists in all, one wave).  Two sorted lists merge in one
// wave: lane l takes max(A[l], B[63 - l]), the top half of the bitonic sequence A | reverse(B), i.e. the 64 largest keys
// of both, and a bitonic half-cleaner network (lane strides 32 .. 1) sorts them; B is kept ascending, so no lane
// reversal is needed.
// All are bound by their chains of exchanges.  Both launches, networks / popping: 248320 logits k = 1 13.6 / 10.1 us, k = 16
// 13.6 / 13.2, k = 24 13.6 / 14.9, k = 40 13.7 / 18.3; 1000 logits k = 1 8.6 / 4.8, k = 16 8.5 / 8.0, k = 20 8.6 / 8.8.
// Merging the lists pair by pair through LDS took 12.4 us at 248320 logits (6.5 to 7.3 here).
#include "rmi_common.h"

#include <type_traits>

namespace rmi {
namespace {

constexpr int kTopkMax = 64;       // largest k
constexpr int kListStride = 64;    // keys per list in the workspace
constexpr int kListWaves = 8;      // waves of a list workgroup
constexpr int kMaxLists = 128;     // workgroup lists the merge takes: 8 per wave
constexpr int kMergeWaves = 16;
constexpr int kPopMax = 16;        // the popping list kernel's largest k

__device__ __forceinline__ uint64_t topk_key(float v, uint32_t idx) {
    uint32_t b = __float_as_uint(v);
    if (b == 0x80000000u) b = 0u;   // -0 compares equal to +0
    b ^= (b >> 31) ? 0xffffffffu : 0x80000000u;
    return (static_cast<uint64_t>(b) << 32) | (0xffffffffu - idx);   // > 0 for every real key; 0 = no entry
}

// key of lane l ^ K (the VALU lane exchange of rmi_common.h on both halves)
template <int K>
__device__ __forceinline__ uint64_t xor64(uint64_t v) {
    const uint32_t lo = xor_lane<K>(static_cast<uint32_t>(v)), hi = xor_lane<K>(static_cast<uint32_t>(v >> 32));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// one compare-exchange with lane l ^ K: the larger key where `larger` holds (equal keys are the same key, or both 0)
template <int K>
__device__ __forceinline__ uint64_t exchange(uint64_t v, bool larger) {
    const uint64_t o = xor64<K>(v);
    return (v > o) == larger ? v : o;
}

// the bitonic network's last stage: a bitonic sequence over the wave's lanes into descending (ASC: ascending) order
template <bool ASC, int K = 32>
__device__ __forceinline__ uint64_t half_clean(uint64_t v, int lane) {
    v = exchange<K>(v, ((lane & K) == 0) != ASC);
    if constexpr (K > 1) v = half_clean<ASC, K / 2>(v, lane);
    return v;
}

// The 64 largest keys of a (descending) and b (ascending), in descending (ASC: ascending) order.  Every lane active.
template <bool ASC>
__device__ __forceinline__ uint64_t merge_lists(uint64_t a, uint64_t b, int lane) {
    return half_clean<ASC>(a > b ? a : b, lane);
}

// one stage of the sort: runs of SIZE lanes, alternately descending and ascending (ASC: the other way round)
template <bool ASC, int SIZE, int K = SIZE / 2>
__device__ __forceinline__ uint64_t sort_stage(uint64_t v, int lane) {
    v = exchange<K>(v, (((lane & K) == 0) != ((lane & SIZE) != 0)) != ASC);
    if constexpr (K > 1) v = sort_stage<ASC, SIZE, K / 2>(v, lane);
    return v;
}
template <bool ASC>
__device__ __forceinline__ uint64_t sort64(uint64_t v, int lane) {
    v = sort_stage<ASC, 2>(v, lane);
    v = sort_stage<ASC, 4>(v, lane);
    v = sort_stage<ASC, 8>(v, lane);
    v = sort_stage<ASC, 16>(v, lane);
    v = sort_stage<ASC, 32>(v, lane);
    return sort_stage<ASC, 64>(v, lane);   // lane & 64 is 0
}

// `groups` slices of 256 logits per wave
__global__ __launch_bounds__(64 * kListWaves) void topk_lists_kernel(const float* __restrict__ x, int n, int groups,
                                                                     uint64_t* __restrict__ lists) {
    __shared__ uint64_t wl[kListWaves][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t base = (static_cast<int64_t>(blockIdx.x) * kListWaves + w) * groups * 256 + lane;
    const int64_t last = n - 1;
    float xv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xv[j] = x[min(base + 64 * j, last)];   // clamped: no load under a branch
    uint64_t mine = 0;   // the wave's list, descending
    for (int g = 0; g < groups; ++g) {
        const int64_t i0 = base + 256 * g;
        uint64_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t i = i0 + 64 * j;
            v[j] = i < n ? topk_key(xv[j], static_cast<uint32_t>(i)) : 0ull;
            xv[j] = x[min(i + 256, last)];   // the next slice's, in flight during this one's sort
        }
        v[0] = sort64<false>(v[0], lane);
        v[1] = sort64<true>(v[1], lane);
        v[2] = sort64<false>(v[2], lane);
        v[3] = sort64<true>(v[3], lane);
        const uint64_t a = merge_lists<false>(v[0], v[1], lane), b = merge_lists<true>(v[2], v[3], lane);
        if (g == 0) {
            mine = merge_lists<false>(a, b, lane);
        } else {
            mine = merge_lists<false>(mine, merge_lists<true>(a, b, lane), lane);
        }
    }
    // the workgroup's lists: odd waves' ascending
    wl[w][w & 1 ? 63 - lane : lane] = mine;
    __syncthreads();
    uint64_t m = 0;
    if (w < 2) {
        const uint64_t a = merge_lists<false>(wl[4 * w][lane], wl[4 * w + 1][lane], lane);
        m = merge_lists<false>(a, merge_lists<true>(wl[4 * w + 2][lane], wl[4 * w + 3][lane], lane), lane);
    }
    __syncthreads();
    if (w == 1) wl[1][63 - lane] = m;
    __syncthreads();
    if (w == 0) lists[static_cast<size_t>(blockIdx.x) * kListStride + lane] = merge_lists<false>(m, wl[1][lane], lane);
}

__global__ __launch_bounds__(64 * kMergeWaves) void topk_merge_kernel(const float* __restrict__ x,
                                                                      const uint64_t* __restrict__ lists, int nlists, int k,
                                                                      int* __restrict__ out_idx,
                                                                      float* __restrict__ out_val) {
    __shared__ uint64_t buf[kMergeWaves][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint64_t v[8];   // lists 8 w + j: odd ones read backwards, so ascending
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int l = 8 * w + j;
        const uint64_t e = lists[static_cast<size_t>(min(l, nlists - 1)) * kListStride + (j & 1 ? 63 - lane : lane)];
        v[j] = l < nlists ? e : 0ull;
    }
    uint64_t m = 0;
    if (8 * w < nlists) {   // uniform
        const uint64_t a = merge_lists<false>(v[0], v[1], lane), b = merge_lists<true>(v[2], v[3], lane);
        const uint64_t c = merge_lists<false>(v[4], v[5], lane), d = merge_lists<true>(v[6], v[7], lane);
        m = merge_lists<false>(merge_lists<false>(a, b, lane), merge_lists<true>(c, d, lane), lane);
    }
    buf[w][w & 1 ? 63 - lane : lane] = m;
    __syncthreads();
    if (w < 4) {
        const uint64_t a = merge_lists<false>(buf[4 * w][lane], buf[4 * w + 1][lane], lane);
        m = merge_lists<false>(a, merge_lists<true>(buf[4 * w + 2][lane], buf[4 * w + 3][lane], lane), lane);
    }
    __syncthreads();
    if (w < 4) buf[w][w & 1 ? 63 - lane : lane] = m;
    __syncthreads();
    if (w == 0) {
        const uint64_t a = merge_lists<false>(buf[0][lane], buf[1][lane], lane);
        m = merge_lists<false>(a, merge_lists<true>(buf[2][lane], buf[3][lane], lane), lane);
        if (lane < k) {
            const int idx = m ? static_cast<int>(0xffffffffu - static_cast<uint32_t>(m)) : -1;
            out_idx[lane] = idx;
            out_val[lane] = idx >= 0 ? x[idx] : 0.0f;
        }
    }
}

// up to eight lists: one wave (its own kernel: as a branch of the one above it slowed that one by 0.3 us)
__global__ __launch_bounds__(64) void topk_merge_few_kernel(const float* __restrict__ x, const uint64_t* __restrict__ lists,
                                                            int nlists, int k, int* __restrict__ out_idx,
                                                            float* __restrict__ out_val) {
    const int lane = threadIdx.x;
    uint64_t v[8];   // odd lists read backwards, so ascending
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint64_t e = lists[static_cast<size_t>(min(j, nlists - 1)) * kListStride + (j & 1 ? 63 - lane : lane)];
        v[j] = j < nlists ? e : 0ull;
    }
    uint64_t m = v[0];
    if (nlists > 4) {   // uniform
        const uint64_t a = merge_lists<false>(v[0], v[1], lane), b = merge_lists<true>(v[2], v[3], lane);
        const uint64_t c = merge_lists<false>(v[4], v[5], lane), d = merge_lists<true>(v[6], v[7], lane);
        m = merge_lists<false>(merge_lists<false>(a, b, lane), merge_lists<true>(c, d, lane), lane);
    } else if (nlists > 1) {
        m = merge_lists<false>(m, v[1], lane);
        if (nlists > 2) m = merge_lists<false>(m, merge_lists<true>(v[2], v[3], lane), lane);
    }
    if (lane < k) {
        const int idx = m ? static_cast<int>(0xffffffffu - static_cast<uint32_t>(m)) : -1;
        out_idx[lane] = idx;
        out_val[lane] = idx >= 0 ? x[idx] : 0.0f;
    }
}

// wave-uniform largest key: DPP within each row of 16 lanes (xor 1, xor 2, half-row mirror, row mirror; the maximum is
// symmetric, so a mirror partner serves as well as an xor one), then the four rows' maxima
__device__ __forceinline__ uint64_t wave_max64(uint64_t v) {
    auto larger = [](uint64_t a, uint64_t b) { return a > b ? a : b; };
    auto dpp = [](uint64_t u, auto ctrl) {
        const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), decltype(ctrl)::value, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), decltype(ctrl)::value, 0xf, 0xf, false);
        return (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo);
    };
    auto row = [&](int l) {
        const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(v), l);
        const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(v >> 32), l);
        return (static_cast<uint64_t>(hi) << 32) | lo;
    };
    v = larger(v, dpp(v, std::integral_constant<int, 0xb1>{}));
    v = larger(v, dpp(v, std::integral_constant<int, 0x4e>{}));
    v = larger(v, dpp(v, std::integral_constant<int, 0x141>{}));
    v = larger(v, dpp(v, std::integral_constant<int, 0x140>{}));
    return larger(larger(row(0), row(16)), larger(row(32), row(48)));
}

// Short lists: the lane's E keys sorted in registers, then the wave's k largest popped one by one
template <int E>
__global__ __launch_bounds__(256) void topk_pop_kernel(const float* __restrict__ x, int n, int k,
                                                       uint64_t* __restrict__ lists) {
    __shared__ uint64_t wl[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t base = (static_cast<int64_t>(blockIdx.x) * 4 + w) * 64 * E + lane;
    const int64_t last = n - 1;
    float xv[E];
#pragma unroll
    for (int j = 0; j < E; ++j) xv[j] = x[min(base + 64 * j, last)];   // clamped: no load under a branch
    uint64_t v[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int64_t i = base + 64 * j;
        v[j] = i < n ? topk_key(xv[j], static_cast<uint32_t>(i)) : 0ull;
    }
#pragma unroll
    for (int size = 2; size <= E; size <<= 1) {
#pragma unroll
        for (int stride = size / 2; stride > 0; stride >>= 1) {
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int j = i ^ stride;
                if (j > i) {
                    const uint64_t a = v[i], b = v[j];
                    const bool swap = (i & size) == 0 ? a < b : a > b;
                    v[i] = swap ? b : a;
                    v[j] = swap ? a : b;
                }
            }
        }
    }
    uint64_t mine = 0;
    for (int it = 0; it < k; ++it) {
        const uint64_t m = wave_max64(v[0]);
        if (m == 0) break;              // the slice has fewer than k logits (uniform across the wave)
        if (lane == it) mine = m;
        if (v[0] == m) {                // keys are distinct: exactly one lane pops
#pragma unroll
            for (int j = 0; j + 1 < E; ++j) v[j] = v[j + 1];
            v[E - 1] = 0;
        }
    }
    wl[w][w & 1 ? 63 - lane : lane] = mine;   // odd waves' ascending
    __syncthreads();
    if (w > 0) return;
    const uint64_t a = merge_lists<false>(wl[0][lane], wl[1][lane], lane);
    const uint64_t b = merge_lists<true>(wl[2][lane], wl[3][lane], lane);
    lists[static_cast<size_t>(blockIdx.x) * kListStride + lane] = merge_lists<false>(a, b, lane);
}

// a workgroup's logits / 256: the smallest of 8, 16, 32 that keeps the lists within one merge workgroup
int lane_elems(int n) {
    for (int e = 8; e <= 32; e *= 2)
        if ((static_cast<int64_t>(n) + 256 * e - 1) / (256 * e) <= kMaxLists) return e;
    return 0;
}

}  // namespace
}  // namespace rmi

using namespace rmi;

extern "C" size_t rmi_topk_workspace_bytes(int n) {
    const int e = lane_elems(n);
    if (n <= 0 || e == 0) return 0;
    // four lists a workgroup, one of which is used (the size callers have allocated before)
    const int64_t waves = (static_cast<int64_t>(n) + 64 * e - 1) / (64 * e);
    return static_cast<size_t>((waves + 3) / 4 * 4) * kListStride * sizeof(uint64_t);
}

extern "C" int rmi_topk(const float* logits, int n, int k, int* out_idx, float* out_val, void* workspace,
                        void* stream) {
    const int e = lane_elems(n);
    if (n <= 0 || e == 0) return fail(RMI_ERR_SHAPE, "topk: n must be 1..1048576");
    if (k < 1 || k > kTopkMax || k > n) return fail(RMI_ERR_SHAPE, "topk: k must be 1..min(64, n)");
    if (!aligned4(logits) || !aligned4(out_idx) || !aligned4(out_val) || !workspace ||
        (reinterpret_cast<uintptr_t>(workspace) & 7u) != 0)
        return fail(RMI_ERR_POINTER, "topk: null or misaligned pointer");
    const int blocks = static_cast<int>((static_cast<int64_t>(n) + 256 * e - 1) / (256 * e));
    auto* lists = static_cast<uint64_t*>(workspace);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (k > kPopMax)
        hipLaunchKernelGGL(topk_lists_kernel, dim3(blocks), dim3(64 * kListWaves), 0, s, logits, n, e / 8, lists);
    else if (e == 8)
        hipLaunchKernelGGL(topk_pop_kernel<8>, dim3(blocks), dim3(256), 0, s, logits, n, k, lists);
    else if (e == 16)
        hipLaunchKernelGGL(topk_pop_kernel<16>, dim3(blocks), dim3(256), 0, s, logits, n, k, lists);
    else
        hipLaunchKernelGGL(topk_pop_kernel<32>, dim3(blocks), dim3(256), 0, s, logits, n, k, lists);
    const int rc = launch_status("topk_lists");
    if (rc != RMI_OK) return rc;
    if (blocks <= 8)
        hipLaunchKernelGGL(topk_merge_few_kernel, dim3(1), dim3(64), 0, s, logits, lists, blocks, k, out_idx, out_val);
    else
        hipLaunchKernelGGL(topk_merge_kernel, dim3(1), dim3(64 * kMergeWaves), 0, s, logits, lists, blocks, k, out_idx, out_val);
    return launch_status("topk_merge");
}
