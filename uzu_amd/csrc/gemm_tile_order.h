// gemm_tile_order.h -- workgroup id -> output tile of the large-tile products (k_gemm128.hip, k_gemm_dma.hip, k_linear_mfma.hip).
//
// Workgroups are dealt to the 8 XCDs round-robin, and the 64 or so that an XCD runs at a time should share row and column panels in its L2.  The tiles are put in one sequence --
// columns in blocks of 64 / TM, in those the rows in blocks of TM = 8 (all of them if there are fewer), in those column by column -- and XCD x takes the x-th eighth of it: whatever the
// counts, no XCD has more than one tile above another, and what it runs at a time is about 8 x 8 tiles.  Whole super-tiles dealt to the XCDs (gemm_tile_map.h) leave some with half
// as many tiles again: 2048 x 7712 x 2048 in bf16 (16 x 61 tiles) 126 -> 82 us, 517 x 8224 x 1024 in int4 (5 x 65) 33.8 -> 24.6.
// Plain C++ so that a test can compile it for the host.
#pragma once
#include <stdint.h>
#ifndef __HIPCC__
#define UZU_ORDER_HD
#else
#define UZU_ORDER_HD __host__ __device__
#endif

namespace uzu {
namespace k {

UZU_ORDER_HD inline uint32_t tile_order_grid(uint32_t m_tiles, uint32_t n_tiles) { return (m_tiles * n_tiles + 7) / 8 * 8; }
// false = padding workgroup (exits)
UZU_ORDER_HD inline bool tile_of_block(uint32_t block, uint32_t m_tiles, uint32_t n_tiles, uint32_t* m_t, uint32_t* n_t) {
    const uint32_t total = m_tiles * n_tiles, share = total / 8, more = total % 8, xcd = block & 7, slot = block >> 3;
    if (slot >= share + (xcd < more ? 1u : 0u)) return false;
    const uint32_t TM = m_tiles < 8 ? m_tiles : 8, TN = 64 / TM;
    uint32_t t = xcd * share + (xcd < more ? xcd : more) + slot;
    const uint32_t n_block = t / (m_tiles * TN), n0 = n_block * TN, width = n_tiles - n0 < TN ? n_tiles - n0 : TN;
    t -= n_block * (m_tiles * TN);
    const uint32_t m_block = t / (TM * width), m0 = m_block * TM, height = m_tiles - m0 < TM ? m_tiles - m0 : TM;
    t -= m_block * (TM * width);
    const uint32_t column = t / height;
    *m_t = m0 + t - column * height;
    *n_t = n0 + column;
    return true;
}

// Two variations for products whose weights are small beside the rows (linear_tile_order, k_linear_mfma.hip), with the same shares per XCD:
// row by row, where a row of tiles is short; and a last column that is mostly padding behind the whole tiles, so that what goes beyond a full round of workgroups is its cheap tiles.
enum TileOrder { kTileBlocks, kTileRows, kTileLastColumnBehind };
UZU_ORDER_HD inline bool tile_of_block(uint32_t block, uint32_t m_tiles, uint32_t n_tiles, TileOrder order, uint32_t* m_t, uint32_t* n_t) {
    const uint32_t xcd = block & 7, slot = block >> 3;
    if (order == kTileRows) {
        const uint32_t total = m_tiles * n_tiles, share = total / 8, more = total % 8, t = xcd * share + (xcd < more ? xcd : more) + slot;
        *m_t = t / n_tiles, *n_t = t - *m_t * n_tiles;
        return slot < share + (xcd < more ? 1u : 0u);
    }
    const uint32_t behind = order == kTileLastColumnBehind && n_tiles > 1 ? 1 : 0;
    if (tile_of_block(block, m_tiles, n_tiles - behind, m_t, n_t)) return true;
    if (!behind) return false;
    const uint32_t whole = m_tiles * (n_tiles - 1), more = whole % 8;
    *m_t = (slot - whole / 8 - (xcd < more ? 1u : 0u)) * 8 + ((xcd - more) & 7u), *n_t = n_tiles - 1;
    return *m_t < m_tiles;
}

} // namespace k
} // namespace uzu
