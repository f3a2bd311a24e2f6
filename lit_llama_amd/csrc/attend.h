// Shared by the attention kernels that multiply f32 queries and weights on the bf16 matrix cores: an f32 as three bf16 (limbs), whose products with bf16 are exact in f32, and a plain loop for
// the rows that three limbs do not carry (not part of the C ABI).
#pragma once
#include "common.h"

// what is left of x behind its upper 16 bits
__device__ __forceinline__ float below_limb(float x) { return x - __uint_as_float(__float_as_uint(x) & 0xffff0000u); }
// the upper halves of eight dwords
__device__ __forceinline__ u32x4 upper_halves(const uint32_t (&t)[8]) {
    return u32x4{__builtin_amdgcn_perm(t[1], t[0], 0x07060302u), __builtin_amdgcn_perm(t[3], t[2], 0x07060302u), __builtin_amdgcn_perm(t[5], t[4], 0x07060302u),
                 __builtin_amdgcn_perm(t[7], t[6], 0x07060302u)};
}

// An infinite key or value times three limbs is a NaN wherever one of them is 0 (the largest score's weight is 1, 0 and 0), where its product with the f32 is an infinity, or a score of -inf.
// Sums that are not finite are therefore made again, here, in f32: THREADS threads, a key each, then a dimension each (vdim <= THREADS).  `score(k)` is the score of key k,
// `value(k, d)` its value; the maximum m, the sum of weights l and, in thread d, the sum o of weighted values of dimension d.  `lds`: THREADS + 32 floats.  Every thread of the block calls it
template <int THREADS, typename Score, typename Value>
__device__ __forceinline__ void attend_plain(int k_begin, int k_end, int vdim, float* lds, Score score, Value value, float& m, float& l, float& o) {
    const int tid = threadIdx.x;
    float* const red = lds + THREADS;
    m = -INFINITY, l = o = 0.f;
#pragma unroll 1
    for (int kb = k_begin; kb < k_end; kb += THREADS) {
        const int n = min(THREADS, k_end - kb);
        const float s = tid < n ? score(kb + tid) : -INFINITY;
        const float top = fmaxf(m, block_max(s, red)), base = top == -INFINITY ? 0.f : top, corr = expf(m - base), w = tid < n ? expf(s - base) : 0.f;
        lds[tid] = w;
        l = l * corr + block_sum(w, red);
        m = top;
        if (tid < vdim) {
            o *= corr;
#pragma unroll 4
            for (int i = 0; i < n; ++i) o += lds[i] * value(kb + i, tid);
        }
    }
    __syncthreads();
}
// sum over n dimensions (a multiple of 8) of f32 times a row of bf16 (16-B aligned)
__device__ __forceinline__ float dot_row(const float* q, const bf16_t* row, int n) {
    float s = 0.f;
#pragma unroll 2
    for (int d = 0; d < n; d += 8) {
        const u32x4 v = *(const u32x4*)(row + d);
#pragma unroll
        for (int i = 0; i < 4; ++i) s += q[d + 2 * i] * __uint_as_float(v[i] << 16), s += q[d + 2 * i + 1] * __uint_as_float(v[i] & 0xffff0000u);
    }
    return s;
}
