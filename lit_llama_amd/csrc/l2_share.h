// Internal: how the blocks of an XCD share out the weights of a row block that they all read (gemm_deep_kernel, csrc/gemm.hip).
#pragma once

// Workgroup L2 = L * ksplit + slice of a launch (row block major: L = nb * m_blocks + token block) is one of the per_xcd that run on an XCD.  Without K-slices the blocks
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
