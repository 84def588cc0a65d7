// How the tiles of expert-routed rows are dealt to the XCDs: shared by the tile kernels and a host test.
#pragma once
#include <cstdint>

namespace mtq {

constexpr uint32_t QD_HEIGHTS = 4;   // classes of row tiles by their 32-row blocks: 5, 4, 3, up to 2

// Tile number `at` of XCD `xcd`, or 0xFFFFFFFF past its last one. The row tiles of height class h, the highest first, are
// [h * stride, h * stride + count[h]), `n_tiles` column tiles each. Every XCD gets an even share of consecutive tiles of each class (a
// class's odd tiles go to the XCDs after those that had the last class's), the highest first: with skewed routing too, no XCD has
// only high tiles and none of them starts at the end. An XCD has ceil(total / 8) tiles at most.
constexpr uint32_t routed_deal(const uint32_t (&count)[QD_HEIGHTS], uint32_t stride, uint32_t n_tiles, uint32_t xcd, uint32_t at) {
    uint32_t turn = 0;
    for (uint32_t h = 0; h < QD_HEIGHTS; h++) {
        const uint32_t total = count[h] * n_tiles, each = total / 8, odd = total % 8;
        const uint32_t x = (xcd - turn) & 7u, mine = each + (x < odd ? 1u : 0u);
        if (at < mine) return h * stride * n_tiles + x * each + (x < odd ? x : odd) + at;
        at -= mine;
        turn = (turn + odd) & 7u;
    }
    return 0xFFFFFFFFu;
}

}  // namespace mtq
