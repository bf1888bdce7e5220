// Host check of uzu_amd/csrc/gemm_tile_order.h: in each order every output tile is visited once and the XCDs' (block id mod 8) shares differ by one tile at most.
#include <stdio.h>
#include <vector>

#include "../../uzu_amd/csrc/gemm_tile_order.h"

using namespace uzu::k;

static bool check(uint32_t m_tiles, uint32_t n_tiles, TileOrder order) {
    std::vector<int> seen(m_tiles * n_tiles, 0);
    uint32_t share[8] = {0, 0, 0, 0, 0, 0, 0, 0}, least = ~0u, most = 0;
    for (uint32_t b = 0; b < tile_order_grid(m_tiles, n_tiles); ++b) {
        uint32_t m_t, n_t;
        if (!tile_of_block(b, m_tiles, n_tiles, order, &m_t, &n_t)) continue;
        if (m_t >= m_tiles || n_t >= n_tiles) return false;
        seen[m_t * n_tiles + n_t]++, share[b & 7]++;
    }
    for (int v : seen)
        if (v != 1) return false;
    for (uint32_t v : share) least = v < least ? v : least, most = v > most ? v : most;
    return most - least <= 1;
}

int main() {
    long checked = 0, bad = 0;
    for (uint32_t m_tiles = 1; m_tiles <= 48; ++m_tiles)
        for (uint32_t n_tiles = 1; n_tiles <= 160; ++n_tiles)
            for (TileOrder order : {kTileBlocks, kTileRows, kTileLastColumnBehind}) ++checked, bad += !check(m_tiles, n_tiles, order);
    printf("tile_order: %ld shapes, %ld bad\n", checked, bad);
    return bad != 0;
}
