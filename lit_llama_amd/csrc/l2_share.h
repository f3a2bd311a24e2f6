// Internal: the order of a BF16 launch's blocks, and how the blocks of an XCD share out the weights of a row block that they all read (gemm_deep_kernel, csrc/gemm.hip).
#pragma once

constexpr int kSquare = 4;  // row blocks of a square

// Blocks of `waves` waves and `tokens` tokens that share out their weights (l2_share()).  Their place in the row is what their share goes by, so they keep to whole rows; blocks of 8 waves
// that share nothing may run in squares.  (Blocks of 64 tokens x 8 waves in squares, sharing by their place in the row: 550 tokens, N = 6656, K = 17920 187 us, row by row 160; 1344, N = 3072,
// K = 12288 131 / 113; 1600, N = 2560, K = 6912 78 / 67)
constexpr bool shares_weights(int waves, int tokens) { return tokens == 64 || (tokens > 64 && waves == 4); }
constexpr bool may_run_in_squares(int waves, int tokens) { return waves == 8 && !shares_weights(waves, tokens); }

// Block L of a launch of n_blocks row blocks x m_blocks token blocks: row block by row block, or in squares, kSquare row blocks (the last ones: what is left) by a token block each
struct BlockAt {
    int nb, mb;
};
__host__ __device__ inline BlockAt block_at(int L, int n_blocks, int m_blocks, bool squares) {
    int nb = L / m_blocks, mb = L - nb * m_blocks;
    if (squares) {
        const int first = nb / kSquare * kSquare, at = L - first * m_blocks, rows = n_blocks - first < kSquare ? n_blocks - first : kSquare;
        mb = rows == kSquare ? at / kSquare : at / rows;
        nb = first + at - mb * rows;
    }
    return {nb, mb};
}

// Workgroup L2 = L * ksplit + slice of a launch (row block by row block: L = nb * m_blocks + token block) is one of the per_xcd that run on an XCD.  Without K-slices the blocks
// of row block nb on that XCD, four at least, bring each up to `count` of its `lines` cache lines, from `first` on; fewer of them, or slices of K (whose blocks read
// different units): none.  (One division and no branch: an early return took launches of 5-15 us 0.2 us)
struct L2Share {
    int first, count;
};
__host__ __device__ inline L2Share l2_share(int lines, int L, int nb, int m_blocks, int ksplit, int xcd, int per_xcd) {
    const int begin = xcd * per_xcd, end = begin + per_xcd;
    const int lo = nb * m_blocks > begin ? nb * m_blocks : begin, hi = (nb + 1) * m_blocks < end ? (nb + 1) * m_blocks : end;
    const int n = hi - lo > 1 ? hi - lo : 1, share = (lines + n - 1) / n;  // (per_xcd counts slices: hi - lo may be 0 or less)
    return {(L - lo) * share, ksplit == 1 && n >= 4 ? share : 0};
}
