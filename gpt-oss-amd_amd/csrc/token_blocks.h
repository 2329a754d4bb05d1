// How an expert's bucket of rows is cut into token blocks (the tiles of a TileMap), and the order in which a launch lists them.
#pragma once
#include <hip/hip_runtime.h>

namespace moe {

constexpr int kPrefillStep = 16;      // the MXFP4 kernel runs any number of MFMA tiles,
constexpr int kPrefillStepBf16 = 64;  // the bf16 kernel (full row blocks) multiples of four
// Rows of each but the last of an expert's tiles, cut evenly; as many tiles as tile_tokens (a multiple of step) would give.  step is
// what the kernel that takes the tiles rounds their rows up to: all but the last are multiples of it, so that a bucket's matrix work is
// ceil(count / step) steps, as few as there can be.  Of MXFP4 buckets only those of two tiles are cut evenly: from three on a remainder
// is a smaller part of the bucket, and short blocks at the end of a launch even out how its compute units finish.  Whole MoE block, us,
// 128-row tiles and a remainder : all cut evenly : those of two tiles, 32 experts: 1000 tokens 238 : 233 : 231, 1500 tokens 306 : 304 : 304, 1800
// tokens 349 : 365 : 348, 2000 tokens 382 : 394 : 380, 3000 tokens 542 : 551 : 541, 4096 tokens 712 : 707 : 713; skewed, 900 tokens 210 : 221 :
// 209, 1000 tokens 236 : 233 : 233, 4096 tokens 713 : 711 : 711; 8 experts, 600 tokens 145 : 155 : 145, 800 tokens 189 : 182 : 188; 128 experts,
// 6000 tokens 1233 : 1174 : 1172.  169 sizes together 1 : 1.001 : 0.997.
__host__ __device__ inline int even_tile_rows(int count, int tile_tokens, int step) {
    const int n = (count + tile_tokens - 1) / tile_tokens;
    if (n <= 1 || (n > 2 && step == kPrefillStep)) return tile_tokens;
    return ((count + n - 1) / n + step - 1) / step * step;
}

// An expert's token blocks: `full` ones of `rows` rows and a last one of `rem` (none if 0).  EVEN > 0: as many blocks as tile_tokens
// gives, cut evenly in steps of EVEN rows (even_tile_rows).  A remainder of a few rows streams the expert's weights once
// more for next to no matrix work, and takes more than half of a whole block's time for it.  (MXFP4: figures at even_tile_rows.)
// bf16, whole MoE block, us, whole token blocks and a remainder : even ones, 32 experts: 1500 tokens 433 : 434, 2048 tokens 599 : 575,
// 2400 tokens 667 : 591, 3400 tokens 726 : 727, 4096 tokens 868 : 855, 4864 tokens 1025 : 1017, 6656 tokens 1323 : 1327, 8192 tokens 1548 :
// 1548; 8 experts, 1100 tokens 335 : 309.  In steps of 16 rows, which the bf16 kernel rounds up to 64: 2400 tokens 600, 4096 tokens 859
// (skewed 878 against 869), 4864 tokens 1022 (1028), 6656 tokens 1363 (1357).
struct TokenBlocks {
    int rows, full, rem;
};
template <int EVEN>
__host__ __device__ inline TokenBlocks token_blocks(int tile_tokens, int count) {
    TokenBlocks b;
    b.rows = EVEN ? even_tile_rows(count, tile_tokens, EVEN) : tile_tokens;
    if constexpr (EVEN > 0) {  // all of ceil(count / tile_tokens) but perhaps the last are full: no division by rows
        const int n = (count + tile_tokens - 1) / tile_tokens;
        b.full = n > 0 && n * b.rows != count ? n - 1 : n;
    } else {
        b.full = count / b.rows;
    }
    b.rem = count - b.full * b.rows;
    return b;
}

// The order of a launch's tiles.  by_size: from the largest to the smallest, in steps of the cut (equal sizes: ascending expert).  An
// expert kernel that takes tiles in this order runs its shortest blocks last, next to compute units that have already run out of work.
// Otherwise: the tiles but every expert's last, ascending expert, and then the last ones by size.  (EVEN = 0: the two are the same.)
template <int EVEN>
struct TileOrder {
    int tile_tokens, by_size;
    __host__ __device__ int steps(int rows) const { return EVEN > 0 ? (rows + EVEN - 1) / (EVEN > 0 ? EVEN : 1) : rows; }
    __host__ __device__ int full_size(const TokenBlocks& b) const { return by_size ? steps(b.rows) : tile_tokens; }
    __host__ __device__ int last_size(const TokenBlocks& b) const { return steps(b.rem); }
    // tiles of expert i that are larger than `size`, or as large and i comes before e
    __host__ __device__ int ahead_of(const TokenBlocks& b, int i, int size, int e) const {
        const int least = i < e ? size : size + 1;
        return (full_size(b) >= least ? b.full : 0) + (b.rem > 0 && last_size(b) >= least ? 1 : 0);
    }
    // tiles of expert i listed ahead of expert e's full ones (which are consecutive), and of its last one
    __host__ __device__ int ahead_of_full(const TokenBlocks& b, int i, const TokenBlocks& mine, int e) const {
        return ahead_of(b, i, full_size(mine), e);
    }
    __host__ __device__ int ahead_of_last(const TokenBlocks& b, int i, const TokenBlocks& mine, int e) const {
        const int own = i == e && full_size(mine) == last_size(mine) ? mine.full : 0;
        return ahead_of(b, i, last_size(mine), e) + own;
    }
};

}  // namespace moe
