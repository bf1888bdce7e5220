// Host check of uzu_amd/csrc/gemm_tile_order.h: every output tile is visited once and the XCDs' (block id mod 8) shares differ by one tile at most.
#include <stdio.h>
#include <vector>

#include "../../uzu_amd/csrc/gemm_tile_order.h"

int main() {
    using namespace uzu::k;
    long checked = 0, bad = 0;
    for (uint32_t m_tiles = 1; m_tiles <= 48; ++m_tiles)
        for (uint32_t n_tiles = 1; n_tiles <= 160; ++n_tiles) {
            std::vector<int> seen(m_tiles * n_tiles, 0);
            uint32_t share[8] = {0, 0, 0, 0, 0, 0, 0, 0}, least = ~0u, most = 0;
            bool ok = true;
            for (uint32_t b = 0; b < tile_order_grid(m_tiles, n_tiles); ++b) {
                uint32_t m_t, n_t;
                if (!tile_of_block(b, m_tiles, n_tiles, &m_t, &n_t)) continue;
                if (m_t >= m_tiles || n_t >= n_tiles) {
                    ok = false;
                    continue;
                }
                seen[m_t * n_tiles + n_t]++, share[b & 7]++;
            }
            for (int v : seen) ok = ok && v == 1;
            for (uint32_t v : share) least = v < least ? v : least, most = v > most ? v : most;
            ok = ok && most - least <= 1;
            ++checked, bad += !ok;
        }
    printf("tile_order: %ld shapes, %ld bad\n", checked, bad);
    return bad != 0;
}
