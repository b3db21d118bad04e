// Weights for the L2s ahead of the GEMM that reads them.
//
// A short launch spends much of its time on the way of its weights from memory: 17 x 4096 x 1024 in bf16 lasts 5.5 us, and 3.1 where
// they lie in the L2 of the XCD that reads them; 128 x 4096 x 1024 on split operands 14.0 and 9.5.  The LayerNorm and attention launches
// before it leave the memory and most CUs idle, so workgroups added to them touch every line of those weights once, on each XCD the
// eighth of the features whose tiles the skinny kernel gives it.  (Touched from another XCD a line comes from the Infinity Cache
// afterwards, which is worth a fifth of that.  The GEMMs themselves as launches that touch gain nothing: their own waves are in the way.)
// A wave takes one piece of 64 lines: with four a wave the added workgroups outlast the launch.
// The description is 16 bytes, since what it adds to the record of arguments is paid by every launch: 48 bytes, 0.18 us.
#pragma once
#include "kernels.h"

namespace cubert {

// A group of 32 features: pieces of 64 lines of 128 bytes (K a multiple of 32).
template <bool SPLIT>
__host__ __device__ constexpr int l2_lines(int K) { return SPLIT ? K / 2 * 3 : K / 2; }
template <bool SPLIT>
__host__ __device__ constexpr int l2_pieces(int K) { return (l2_lines<SPLIT>(K) + 63) / 64; }

// Byte offset of a line of group g.
template <bool SPLIT>
__host__ __device__ constexpr size_t l2_offset(int K, int g, int line) {
    return SPLIT ? (size_t)g * (K / 16 * 3072) + line * 128
                 : (size_t)(g >> 3) * (K / 32 * 16384) + (g & 7) * 2048 + (line >> 4) * 16384 + (line & 15) * 128;
}

#if defined(__HIPCC__)
// The index'th of `waves` waves on that XCD.
template <bool SPLIT>
__device__ __forceinline__ void l2_touch(const WeightsAhead& a, int xcd, int index, int waves, int lane) {
    const int pieces = l2_pieces<SPLIT>(a.K), lines = l2_lines<SPLIT>(a.K), first = a.groups * xcd / 8, end = a.groups * (xcd + 1) / 8;
    for (int u = index; u < (end - first) * pieces; u += waves) {
        const int rel = u / pieces, g = first + rel, line = (u - rel * pieces) * 64 + lane;
        unsigned t = 0;
        if (line < lines) t = *reinterpret_cast<const unsigned*>(static_cast<const unsigned char*>(a.w) + l2_offset<SPLIT>(a.K, g, line));
        asm volatile("" :: "v"(t));              // a use, or the load would not be there
    }
}
#endif

// Workgroups of four waves to add to a launch, a multiple of eight: a piece a wave, or a few.
template <bool SPLIT>
int l2_touch_workgroups(const WeightsAhead& a) {
    if (!a.w) return 0;
    const int per_xcd = ((a.groups + 7) / 8 * l2_pieces<SPLIT>(a.K) + 3) / 4;
    return 8 * (per_xcd < 32 ? per_xcd : 32);
}

}  // namespace cubert
