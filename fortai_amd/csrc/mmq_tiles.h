// The tile rules of the token products (mmq.hip): a time per chunk (four
// blocks of width) for each kernel from the workgroups on the busiest CU, the
// least of which is launched.  Host code; includes nothing but the standard
// library, so that a host-only checker can include it.
#pragma once
#include <algorithm>

namespace fortai_hip {

constexpr int kXcds = 8, kXcdCus = 32;  // dies of the chip, CUs of each; workgroup b runs on die b % 8

constexpr int kFewRows = 128, kFewTokens = 32;  // tile of q8_mmq_kernel_few
constexpr int kSmallRows = 32;                  // rows per workgroup of q8_mmq_exact_kernel_small

inline long long tiles_of(int n, int tile) { return (static_cast<long long>(n) + tile - 1) / tile; }

// The one-dimensional grids of the kernels for few tokens or rows: from eight
// row tiles on ("grouped") workgroup b takes row tile b / 8 / token_tiles * 8 +
// b % 8, so that all token tiles of a row tile are on one die, and the grid is
// padded to whole groups of eight row tiles; with fewer, workgroups in order.
inline bool few_grouped(long long row_tiles) { return row_tiles >= kXcds; }
inline long long few_grid(int rows, int tokens, int row_tile, int token_tile) {
    const long long r = tiles_of(rows, row_tile);
    return (few_grouped(r) ? tiles_of(static_cast<int>(r), kXcds) * kXcds : r) * tiles_of(tokens, token_tile);
}

// Workgroups on the busiest CU: of the whole chip where the tiles go round the
// dies one by one, of the die with the most row tiles where they are grouped.
inline double busiest_cu(int rows, int tokens, int row_tile, int token_tile, bool may_group) {
    const long long r = tiles_of(rows, row_tile), t = tiles_of(tokens, token_tile);
    const long long die = may_group && few_grouped(r) ? tiles_of(static_cast<int>(r), kXcds) * t : (r * t + kXcds - 1) / kXcds;
    return static_cast<double>((die + kXcdCus - 1) / kXcdCus);
}

// The exact product.  Measured over rows 16 .. 9216, widths 1024 .. 9216 and
// 1 .. 1200 tokens, us per chunk: 64 x 64 tiles 2.15 while each CU has at most
// one, then 3.1 for two and 1.6 for each more; 32 rows x 16 tokens 0.15 + 0.29
// each, x 32 tokens 0.25 + 0.47 each (a workgroup of either does 1/8 or 1/4 of
// the large one's work), and 0.05 + 0.85, 0.1 + 1.07 when block-major tokens
// crowd two L2 channels.  The busiest die counts: 777 rows x 257 tokens are
// 225 workgroups of 32 x 32, but 36 on the die that has four of the 25 row
// tiles, so two on some CUs there (width 3072: 62.4 us against 55.7 with 64 x
// 64 tiles, when they were counted over the whole chip).
enum class ExactTiles { LARGE, SMALL_16, SMALL_32 };
inline ExactTiles exact_tiles(int rows, int tokens, bool block_major) {
    const double n = busiest_cu(rows, tokens, 64, 64, false);
    const double large = n <= 1.0 ? 2.15 : std::max(3.1, 1.6 * n);
    const double n16 = busiest_cu(rows, tokens, kSmallRows, 16, true), n32 = busiest_cu(rows, tokens, kSmallRows, 32, true);
    const double t16 = block_major ? 0.05 + 0.85 * n16 : 0.15 + 0.29 * n16;
    const double t32 = block_major ? 0.1 + 1.07 * n32 : 0.25 + 0.47 * n32;
    if (std::min(t16, t32) >= large) return ExactTiles::LARGE;
    return t16 <= t32 ? ExactTiles::SMALL_16 : ExactTiles::SMALL_32;
}

// The whole-block product, measured likewise: 128 x 128 tiles 1.75 while each
// CU has at most one, then 1.65 each; 128 rows x 32 tokens (a quarter of the
// work) 0.2 + 0.66 each.
inline bool few_tiles(int rows, int tokens) {
    const double n = busiest_cu(rows, tokens, 128, 128, false);
    return 0.2 + 0.66 * busiest_cu(rows, tokens, kFewRows, kFewTokens, true) < (n <= 1.0 ? 1.75 : 1.65 * n);
}

}  // namespace fortai_hip
