// Which tile and which part of K a workgroup of the skinny kernel (gemm_skinny.hip) takes.
#pragma once
#include "gemm_common.h"

namespace cubert {
namespace gemm_detail {

// Workgroup ids go round the XCDs.  Each of them owns a run of the tiles, all rows of a band of features before the next band, so
// that a weight row is fetched into one L2 (two at the ends of a run); the parts of K of a tile follow each other.
// An XCD has per_xcd tiles, one more on the first splits_more & 7; tiles_m: tiles in a band of features.
// cells = 2 or 4, taken where the grid divides: the XCDs own the cells of a partition into `cells` by 8 / cells of features by rows, as in tile_of_block;
// tiles_m is then a cell's.
// A grid of more than kSkinnyGridX workgroups goes on in y: x takes no more than 2^32 threads.
struct SkinnyMap {
    int per_xcd, tiles_m;
    unsigned m_magic, split_magic;      // divisors tiles_m, splits
    int splits_more;                    // 3 or log2(cells) << 16 | splits << 3 | tiles % 8
    unsigned shifts;                    // of the divisors, tiles_m's in the low byte
    unsigned grid_x, grid_y;
};
constexpr int kSkinnyGridXLog2 = 22;
constexpr unsigned kSkinnyGridX = 1u << kSkinnyGridXLog2;

// False: more workgroups than there are numbers for (no result of that many tiles fits the memory).
inline bool skinny_map(int tiles_n, int tiles_m, int splits, int cells, SkinnyMap* m) {
    const long tiles = (long)tiles_n * tiles_m;
    if (tiles > (1L << 31) / splits) return false;
    const long all = 8 * ((tiles + 7) / 8) * splits, rows = (all + kSkinnyGridX - 1) / kSkinnyGridX;
    if (rows * kSkinnyGridX >= (1L << 31)) return false;
    if (cells && (tiles_n % cells != 0 || tiles_m % (8 / cells) != 0)) cells = 0;
    if (cells) tiles_m /= 8 / cells;
    const Divisor dm = divisor_of(tiles_m), ds = divisor_of(splits);
    m->per_xcd = (int)(tiles / 8); m->tiles_m = tiles_m;
    m->m_magic = dm.magic; m->split_magic = ds.magic;
    m->splits_more = (cells ? cells / 2 : 3) << 16 | splits << 3 | (int)(tiles % 8);      // log2(2) = 1, log2(4) = 2
    m->shifts = dm.shift | ds.shift << 8;
    m->grid_x = rows > 1 ? kSkinnyGridX : (unsigned)all; m->grid_y = (unsigned)rows;
    return true;
}

// False: a workgroup without a tile.
__host__ __device__ __forceinline__ bool skinny_tile(unsigned block_x, unsigned block_y, int tiles_n, int per_xcd, int tiles_m, unsigned m_magic, unsigned split_magic,
                                                     int splits_more, unsigned shifts, int* tile_n, int* tile_m, int* split) {
    const int id = (int)(block_x + (block_y << kSkinnyGridXLog2)), splits = (splits_more >> 3) & 255, more = splits_more & 7, lg = splits_more >> 16;
    const int xcd = id & 7, is = id >> 3, idx = div_by(is, split_magic, shifts >> 8);
    if (idx >= per_xcd + (xcd < more ? 1 : 0)) return false;
    *split = is - idx * splits;
    // Runs: tile / tiles_m and what is left.  Cells: the quotient goes on through all cells, those of the next rows begin at its multiples of tiles_n.
    const int tile = xcd * per_xcd + (xcd < more ? xcd : more) + idx, q = div_by(tile, m_magic, shifts), rows = xcd >> lg;
    *tile_n = q - rows * tiles_n;
    *tile_m = tile - q * tiles_m + rows * tiles_m;
    return true;
}

}  // namespace gemm_detail
}  // namespace cubert
