// Weights for the L2s ahead of the GEMM that reads them.
//
// A short launch spends much of its time on the way of its weights from memory: 17 x 4096 x 1024 in bf16 lasts 5.5 us, and 3.1 where
// they lie in the L2 of the XCD that reads them; 128 x 4096 x 1024 on split operands 14.0 and 9.5.  The LayerNorm and attention launches
// before it leave the memory and most CUs idle, so workgroups added to them touch every line of those weights once, on each XCD the
// eighth of the features whose tiles the skinny kernel gives it.  (Touched from another XCD a line comes from the Infinity Cache
// afterwards, which is worth a fifth of that.  The GEMMs themselves as launches that touch gain nothing: their own waves are in the way.)
// A wave takes a piece of 64 lines, and of weights with more pieces an XCD than 128 (BERT-large FFN-in in float32, 384) up to three one after
// the other: the workgroups added are 32 an XCD at most.  Many of them are not free: LayerNorm of 128 rows of BERT-large in float32 lasts 5.1 us
// without and 6.2 with them, of 17 rows of BERT-base in bf16 3.0 and 2.9.
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

// Which XCD's weights, and which share of them, an added wave takes: the index'th of `waves`.  Workgroups go round the XCDs in the order of their ids.
struct L2Share {
    int xcd, index, waves;
};
// Workgroup `block` of a grid of `rows` workgroups and the added ones.
__host__ __device__ __forceinline__ L2Share l2_share_after_rows(int block, int rows, int grid, int wave) {
    return {block & 7, ((block - rows) >> 3) * 4 + wave, (grid - rows) / 8 * 4};
}
// Workgroup (x, y, z) of a grid of gx x gy x (blocks + added planes); workgroups of `nw` waves.  The last few, where they are no multiple of eight, take
// nothing (an index past all pieces).
__host__ __device__ __forceinline__ L2Share l2_share_after_planes(int x, int y, int z, int gx, int gy, int gz, int blocks, int nw, int wave) {
    const int plane = gx * gy, id = x + gx * y + plane * z, e = id - plane * blocks, per_xcd = plane * (gz - blocks) / 8;
    return {id & 7, (e >> 3) < per_xcd ? (e >> 3) * nw + wave : 1 << 30, per_xcd * nw};
}

// Offsets that a lane of that wave touches.
template <bool SPLIT, class Touch>
__host__ __device__ __forceinline__ void l2_walk(const WeightsAhead& a, const L2Share& s, int lane, Touch touch) {
    const int pieces = l2_pieces<SPLIT>(a.K), lines = l2_lines<SPLIT>(a.K), first = a.groups * s.xcd / 8, end = a.groups * (s.xcd + 1) / 8;
    for (int u = s.index; u < (end - first) * pieces; u += s.waves) {
        const int rel = u / pieces, g = first + rel, line = (u - rel * pieces) * 64 + lane;
        if (line < lines) touch(l2_offset<SPLIT>(a.K, g, line));
    }
}

#if defined(__HIPCC__)
template <bool SPLIT>
__device__ __forceinline__ void l2_touch(const WeightsAhead& a, const L2Share& s, int lane) {
    l2_walk<SPLIT>(a, s, lane, [&](size_t at) {
        const unsigned t = *reinterpret_cast<const unsigned*>(static_cast<const unsigned char*>(a.w) + at);
        asm volatile("" :: "v"(t));              // a use, or the load would not be there
    });
}
#endif

// Workgroups of four waves to add to a launch, a multiple of eight.
template <bool SPLIT>
int l2_touch_workgroups(const WeightsAhead& a) {
    if (!a.w) return 0;
    const int per_xcd = ((a.groups + 7) / 8 * l2_pieces<SPLIT>(a.K) + 3) / 4;
    return 8 * (per_xcd < 32 ? per_xcd : 32);
}

}  // namespace cubert
