// rad_topk.h - sorted 64-key lists, one key per lane of a wavefront (lane 0
// largest): the sorting and merging networks of the top-K selections.
#pragma once

#include "rad_internal.h"

namespace rad {

// Lane exchanges of the top-K networks without ds_bpermute: lane i gets the
// value of lane i ^ M, from DPP lane moves (strides 1, 2, 4, 8 inside a row
// of 16 lanes) and the gfx950 row and half-wave swaps (16, 32).
template <int M> __device__ __forceinline__ uint32_t lane_xor(uint32_t x)
{
    const int lane = threadIdx.x & 63;
    const int xi = (int)x;
    if constexpr (M == 1) {
        return (uint32_t)__builtin_amdgcn_update_dpp(xi, xi, 0xB1, 0xF, 0xF, false); // quad_perm 1,0,3,2
    } else if constexpr (M == 2) {
        return (uint32_t)__builtin_amdgcn_update_dpp(xi, xi, 0x4E, 0xF, 0xF, false); // quad_perm 2,3,0,1
    } else if constexpr (M == 4) {
        const int up = __builtin_amdgcn_update_dpp(xi, xi, 0x104, 0xF, 0xF, false); // row_shl:4, lane i + 4
        const int dn = __builtin_amdgcn_update_dpp(xi, xi, 0x114, 0xF, 0xF, false); // row_shr:4, lane i - 4
        return (uint32_t)((lane & 4) ? dn : up);
    } else if constexpr (M == 8) {
        return (uint32_t)__builtin_amdgcn_update_dpp(xi, xi, 0x128, 0xF, 0xF, false); // row_ror:8
    } else if constexpr (M == 16) {
        // odd rows of the first operand swap with even rows of the second:
        // r[0] holds rows (0, 0, 2, 2) of x, r[1] rows (1, 1, 3, 3)
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return (lane & 16) ? r[0] : r[1];
    } else {
        static_assert(M == 32, "lane_xor strides 1 .. 32");
        // the upper half of the first operand swaps with the lower half of
        // the second: r[0] holds x's lower half twice, r[1] its upper half
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        return (lane & 32) ? r[0] : r[1];
    }
}

template <int M> __device__ __forceinline__ uint64_t lane_xor_u64(uint64_t v)
{
    return ((uint64_t)lane_xor<M>((uint32_t)(v >> 32)) << 32) | lane_xor<M>((uint32_t)v);
}

// The value of lane 63 - i: each row mirrored (row_mirror), then rows
// r and 3 - r exchanged.
__device__ __forceinline__ uint64_t lane_reverse_u64(uint64_t v)
{
    const int lo = __builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(v >> 32), (int)(v >> 32), 0x140, 0xF, 0xF, false);
    const uint64_t m = ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
    return lane_xor_u64<32>(lane_xor_u64<16>(m));
}

// A wave-uniform lane's value (lane src, a constant).
__device__ __forceinline__ uint64_t lane_read_u64(uint64_t v, int src)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

// One compare-exchange step of a bitonic network at lane stride M.
template <int M> __device__ __forceinline__ uint64_t bitonic_step(uint64_t v, bool take_max)
{
    const uint64_t o = lane_xor_u64<M>(v);
    return take_max ? (v > o ? v : o) : (v < o ? v : o);
}

__device__ __forceinline__ uint64_t wave_sort_desc(uint64_t v)
{
    const int lane = threadIdx.x & 63;
    // stage `size`: lanes in blocks of size sort descending where
    // lane & size == 0; a step at stride m keeps the max in the lower lane
    // of a pair when that block is descending
#define RAD_SORT_STEP(size_, m_) \
    v = bitonic_step<m_>(v, ((lane & (m_)) == 0) == ((lane & (size_)) == 0));
    RAD_SORT_STEP(2, 1)
    RAD_SORT_STEP(4, 2) RAD_SORT_STEP(4, 1)
    RAD_SORT_STEP(8, 4) RAD_SORT_STEP(8, 2) RAD_SORT_STEP(8, 1)
    RAD_SORT_STEP(16, 8) RAD_SORT_STEP(16, 4) RAD_SORT_STEP(16, 2) RAD_SORT_STEP(16, 1)
    RAD_SORT_STEP(32, 16) RAD_SORT_STEP(32, 8) RAD_SORT_STEP(32, 4) RAD_SORT_STEP(32, 2)
    RAD_SORT_STEP(32, 1)
    RAD_SORT_STEP(64, 32) RAD_SORT_STEP(64, 16) RAD_SORT_STEP(64, 8) RAD_SORT_STEP(64, 4)
    RAD_SORT_STEP(64, 2) RAD_SORT_STEP(64, 1)
#undef RAD_SORT_STEP
    return v;
}

// top and b sorted descending over the lanes: the top 64 of both, sorted.
__device__ __forceinline__ uint64_t wave_merge_desc(uint64_t top, uint64_t b)
{
    const int lane = threadIdx.x & 63;
    const uint64_t r = lane_reverse_u64(b);
    uint64_t v = top > r ? top : r;
    v = bitonic_step<32>(v, (lane & 32) == 0);
    v = bitonic_step<16>(v, (lane & 16) == 0);
    v = bitonic_step<8>(v, (lane & 8) == 0);
    v = bitonic_step<4>(v, (lane & 4) == 0);
    v = bitonic_step<2>(v, (lane & 2) == 0);
    v = bitonic_step<1>(v, (lane & 1) == 0);
    return v;
}

// The keys above thr = the k-th key of the sorted list top (k <= 64,
// wave-uniform) of a batch, one per lane, taken into the list; a few are
// inserted one by one (about 20 instructions each), more are sorted and
// merged (about 400).
__device__ __forceinline__ void wave_take_desc(uint64_t &top, uint64_t &thr, uint64_t key, int k)
{
    const int lane = threadIdx.x & 63;
    uint64_t m = __ballot(key > thr);
    if (__popcll(m) > 12) {
        top = wave_merge_desc(top, wave_sort_desc(key));
    } else {
        for (; m; m &= m - 1) {
            const uint64_t v = lane_read_u64(key, __ffsll((long long)m) - 1);
            const int at = __popcll(__ballot(top > v));
            // wave_shr:1: lane i - 1's key
            const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)top, 0x138,
                                                                      0xF, 0xF, true);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(
                0, (int)(uint32_t)(top >> 32), 0x138, 0xF, 0xF, true);
            const uint64_t below = ((uint64_t)hi << 32) | lo;
            top = lane < at ? top : lane == at ? v : below;
        }
    }
    thr = lane_read_u64(top, k - 1);
}

// The sorted 64-key lists of the workgroup's waves (top) merged pairwise
// through wl; wave 0 returns the 64 largest keys of all of them.  Every
// thread of the workgroup calls it.
__device__ static uint64_t merge_wave_lists(uint64_t top, uint64_t (*wl)[64])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    wl[w][lane] = top;
    for (int h = nw >> 1; h >= 1; h >>= 1) {
        __syncthreads();
        if (w < h)
            top = wave_merge_desc(wl[w][lane], wl[w + h][lane]);
        __syncthreads();
        if (w < h)
            wl[w][lane] = top;
    }
    return top;
}

} // namespace rad
