// Wide (M >= 32 tokens) LLM.int8 linear for gfx950: prompt prefill / no-cache evaluation of a `--quantize llm.int8` model.
//
// Replaces, for B * T >= 32 rows, bitsandbytes' MatMul8bitLt forward as Linear8bitLt reaches it
// (lit_llama/quantization.py:38-77; the algorithm is restated in oracle/oracle.py::llm_int8_linear — PARITY
// UNPINNED: bitsandbytes is not vendored).  The skinny kernel (int8.hip) feeds such inputs in chunks
// of <= 16 rows and determines the outlier COLUMN set per chunk; this path determines it over all rows of the call, as the
// algorithm does, and runs the int8 product on v_mfma_i32_16x16x64_i8 over 128-token blocks:
//   1. i8_stage_kernel   (one workgroup per row) — xh = f16(norm_scale * x * 1/rms) (or f16(x)), the row's absmax over its
//                        sub-threshold entries, and the column mask |xh| >= threshold OR-ed over all rows (atomicOr: order
//                        does not matter);
//   2. i8_quant_kernel   — CA = rint(xh * 127 / absmax) with the masked columns zeroed, int8; the ascending list of outlier columns; and those columns by
//                        themselves, f16: xo (rows) and so = f16(CB * SCB / 127) (weights; workgroups behind the rows');
//   3. i8_gemm_kernel    — the int8 weight stream of int8.hip ([tile][unit][r][piece e][lane][16 x int8], one piece = one
//                        MFMA A operand) against CA through LDS (128 or 64 tokens x 128 k, XOR-swizzled), two row tiles per
//                        wave, 8 or 4 waves; then so x xo in the same loop on the f16 MFMA (of a launch cut along K: a slice of its own); epilogue with the arithmetic
//                        of int8.hip, rounding for rounding:
//                            d = f16((acc * 6.200012e-05 * absmax[m]) * SCB[n]);   o = sum over outlier columns k (ascending) of
//                            xh[m, k] * f16(CB[n, k] * SCB[n] / 127);   y = f16(d + f16(o))   (the last step only with outliers)
//                        More outlier columns than `so` has room for are staged through LDS 64 at a time, as all of them once were.
// 512 tokens, 7B, two layers (2000 of mlp.c_proj's 11008 columns hold an outlier): 1950 -> 976 us.  A launch: quantise 30 -> 12 us, stage 16.4 -> 7.5, c_fc1/c_fc2
// 108 -> 83, attn.c_proj / mlp.c_proj slices 48 -> 35 and their sum 151 -> 15 us on average.
#include <type_traits>

#include <stdio.h>
#include <stdlib.h>

#include "common.h"
#include "int8_chain.h"

namespace {

constexpr int kBM = 128;      // tokens per block (64 in launches that leave CUs idle: i8_cut())
constexpr int kTPW = 2;       // 16-row tile slots per wave
constexpr int kOutChunk = 64;            // outlier columns staged per pass of the epilogue
constexpr int kDepth = 4;                // units of operands in LDS and registers
constexpr int kSoLd = kOutChunk + 8;     // row pitch of the staged outlier weights (halves): 144 B, so that 16 rows written side by side fall into 16 banks
template <int kWaves, int BM>
constexpr int kLdsEpi = (BM * kOutChunk + kWaves * kTPW * 16 * kSoLd) * 2;  // f16 [BM tokens][kOutChunk] + [rows][kSoLd]
template <int kWaves, int BM>
constexpr int kLds = kDepth * BM * 128 > kLdsEpi<kWaves, BM> ? kDepth * BM * 128 : kLdsEpi<kWaves, BM>;

__device__ __forceinline__ float f16r(float v) { return f16_to_f32(f32_to_f16(v)); }
// the same for a value that must be an f32 PRODUCT rounded to f32 first (MatMul8bitLt's dequantisation multiplies in f32 and converts): hipcc
// otherwise may contract the last multiply and the conversion into v_fma_mixlo_f16 — one rounding instead of two, a bf16 ulp in ~1e-5 of the
// outputs against the oracle (seen when the outlier side product moved to MFMA and the register allocation around it changed)
__device__ __forceinline__ float f16r_of_f32(float v) {
    asm volatile("" : "+v"(v));
    return f16r(v);
}
// 16 B per lane from `off` of a buffer to 1 KiB of LDS; out of range: zeros
__device__ __forceinline__ void i8_lds_from(__amdgpu_buffer_rsrc_t r, char* lds, unsigned off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, 0, 0, 0);
}
// 16-B chunk swizzle of a 128-B activation row in LDS: rows alternate bank halves (128-B pitch), pairs of rows rotate the
// 8 chunks — the 16 lanes a ds_read_b128 serves together (tokens {0-3, 12-15} with one k-group, {4-11} with the next)
// land in 16 different bank groups
__device__ __forceinline__ int swz8(int tok) { return (tok >> 1) & 7; }

struct I8GemmParams {
    const uint8_t* w;
    unsigned w_bytes;
    const int8_t* ca;      // [M, Kp]
    const f16_t* xh;       // [M, Kp]
    const float* sca;      // [M] row absmax
    const int* olist;      // [0] = n_out, [1 ..] ascending outlier columns
    const float* scb;
    const float* scb2;
    void* y;
    int64_t ldy;
    int M, N, K, Kp, units, n_tiles, n_blocks, per_xcd, total_blocks;
    int y_dtype;
    // split-K for short prompts (a 128-token prompt is ONE token block: 16 workgroups for N = 4096): MODE 1 launches
    // total_blocks x ksplit workgroups that store their int32 partial tiles to part[ks][M][ldp]; MODE 2 (total_blocks
    // workgroups) sums them — integer sums: exact in any order — and runs the epilogue.  Sums move four columns at a time: a row has ldn = N rounded up to four of
    // them, and a pair's c_fc2 starts at ldn
    int ksplit;
    int ldn;
    int64_t ldp;
    int* part;
    // the outlier columns by themselves (i8_quant_kernel): xo[m][ld], so[(tile R + r) 16 + row][ld] = f16(CB SCB / 127), ld = compact_ld(n_out) (whole units of 64), columns past
    // n_out zero.  They exist where so fits its region
    f16_t* xo;
    f16_t* so;
    unsigned* mask_next;  // what the next product of a chain ORs into, cleared here (int8_chain.h), or NULL
    int mask_words;
};
constexpr size_t kSplitBudget = (size_t)32 << 20;             // bytes of the int32 partial tiles of all K-slices,
constexpr size_t kPartBytes = kSplitBudget + kSplitBudget / 2;  // next to the f32 tiles of the outlier columns (2 slices at least)
constexpr size_t kOutlierBudget = (size_t)128 << 20;  // bytes of `so`
__device__ __forceinline__ int compact_ld(int n_out) { return (n_out + 63) & ~63; }
__device__ __forceinline__ bool is_compact(int n_out, int n_tiles, int R, int M) {
    return n_out > 0 && (size_t)n_tiles * R * 16 * compact_ld(n_out) * 2 <= kOutlierBudget && (size_t)M * compact_ld(n_out) * 2 < 0x7fffffffu;
}
constexpr int kMaxSplit = 8;

// ---- 1. rows: f16 operand, absmax over the sub-threshold entries, outlier column mask
__global__ void i8_clear_mask_kernel(unsigned* mask, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) mask[i] = 0u;
}

// (a thread's elements are 256 apart, kAhead of them requested at a time: one at a time behind a switch over the type, a row of 11008 took 25 us.  Of short rows as many
// as there are: 2000 rows of 512 7.8 us with 16 ahead, 5.9 one at a time, 5.1 with 4)
template <typename T>
__device__ __forceinline__ float i8_row_value(T v);
template <>
__device__ __forceinline__ float i8_row_value<float>(float v) { return v; }
template <>
__device__ __forceinline__ float i8_row_value<bf16_t>(bf16_t v) { return bf16_to_f32(v); }
struct f16_raw { f16_t v; };
template <>
__device__ __forceinline__ float i8_row_value<f16_raw>(f16_raw v) { return f16_to_f32(v.v); }

template <typename T, int kAhead>
__global__ __launch_bounds__(256) void i8_stage_kernel(const T* x, int64_t ldx, const void* norm_scale, int norm_dtype, float eps, float threshold, int K,
                                                       int Kp, f16_t* xh, float* sca, unsigned* mask) {
    __shared__ float red[32];
    const int m = blockIdx.x;
    const T* row = x + (int64_t)m * ldx;
    float rinv = 1.f;
    if (norm_scale != nullptr) {
        float ss = 0.f;
        for (int k0 = threadIdx.x; k0 < K; k0 += 256 * kAhead) {
            T raw[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) raw[i] = row[k0 + 256 * i < K ? k0 + 256 * i : k0];
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                if (k0 + 256 * i < K) {
                    const float v = i8_row_value(raw[i]);
                    ss += v * v;
                }
        }
        rinv = rsqrtf(block_sum(ss, red) / (float)K + eps);
    }
    float amax = 0.f;
    for (int k0 = threadIdx.x; k0 < Kp; k0 += 256 * kAhead) {
        T raw[kAhead];
        float ns[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) raw[i] = row[k0 + 256 * i < K ? k0 + 256 * i : 0];
        if (norm_scale != nullptr) {
            if (norm_dtype == MI355_BF16) {
#pragma unroll
                for (int i = 0; i < kAhead; ++i) ns[i] = bf16_to_f32(((const bf16_t*)norm_scale)[k0 + 256 * i < K ? k0 + 256 * i : 0]);
            } else {
#pragma unroll
                for (int i = 0; i < kAhead; ++i) ns[i] = ld_as_f32(norm_scale, k0 + 256 * i < K ? k0 + 256 * i : 0, norm_dtype);
            }
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int k = k0 + 256 * i;
            f16_t h = 0;
            if (k < K) {
                float v = i8_row_value(raw[i]);
                if (norm_scale != nullptr) v = ns[i] * (v * rinv);
                h = f32_to_f16(v);
                const float a = fabsf(f16_to_f32(h));
                if (threshold > 0.f && a >= threshold)
                    atomicOr(mask + (k >> 5), 1u << (k & 31));
                else
                    amax = fmaxf(amax, a);
            }
            if (k < Kp) xh[(int64_t)m * Kp + k] = h;
        }
    }
    amax = block_max(amax, red);
    if (threadIdx.x == 0) sca[m] = amax;
}

// The same for rows in whole aligned groups of four columns, up to kHeld groups a thread: read once, four columns to a request and a store, and the mask a word of 32 columns at a time.
// 512 rows: 11 008 columns of bf16, some 3000 with an outlier, 11.8 -> 8.9 us; 4096 of f32 with a norm 7.4 -> 6.6, 4096 of bf16 5.6 -> 4.4.  kHeld is the least that does: with more a thread
// requests and stores what its row has not (2048 rows of bf16, element by element / 4 or 24 groups / the least: 512 columns 4.5 / 6.3 / 4.1, 2048 7.5 / 7.9 / 6.4, 13 824 34 / 34 / 24, 17 920
// 45 / 38 / 34; 1024 rows of 13 824 16.3 / 19.4 / 15.1, of 17 920 19.5 / 20.8 / 19.6).
template <typename T>
__device__ __forceinline__ f32x4 i8_row_four(const T* p) {
    if constexpr (sizeof(T) == 4) {
        return *(const f32x4*)p;
    } else {
        const u32x2 w = *(const u32x2*)p;
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = i8_row_value(__builtin_bit_cast(T, (uint16_t)((j & 1) ? w[j >> 1] >> 16 : w[j >> 1] & 0xffffu)));
        return v;
    }
}
template <typename T, int kHeld>
__global__ __launch_bounds__(256) void i8_stage_fours_kernel(const T* x, int64_t ldx, const void* norm_scale, int norm_dtype, float eps, float threshold, int K,
                                                             int Kp, f16_t* xh, float* sca, unsigned* mask) {
    __shared__ float red[32];
    const int m = blockIdx.x;
    const T* row = x + (int64_t)m * ldx;
    f32x4 v[kHeld];
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        const int k = 4 * ((int)threadIdx.x + 256 * i);
        v[i] = i8_row_four(row + (k < K ? k : 0));
    }
    if (norm_scale != nullptr) {
        f32x4 ns[kHeld];  // (requested ahead of the sum over the row)
#pragma unroll
        for (int i = 0; i < kHeld; ++i) {
            const int k = 4 * ((int)threadIdx.x + 256 * i), at = k < K ? k : 0;
            ns[i] = norm_dtype == MI355_F32    ? *(const f32x4*)((const float*)norm_scale + at)
                    : norm_dtype == MI355_BF16 ? i8_row_four((const bf16_t*)norm_scale + at)
                                               : i8_row_four((const f16_raw*)norm_scale + at);
        }
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < kHeld; ++i)
            if (4 * ((int)threadIdx.x + 256 * i) < K) ss += (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
        const float rinv = rsqrtf(block_sum(ss, red) / (float)K + eps);
#pragma unroll
        for (int i = 0; i < kHeld; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = ns[i][j] * (v[i][j] * rinv);
    }
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        const int k = 4 * ((int)threadIdx.x + 256 * i);
        f16_t h[4];
        unsigned out = 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h[j] = k < K ? f32_to_f16(v[i][j]) : (f16_t)0;
            const float a = fabsf(f16_to_f32(h[j]));
            const bool big = threshold > 0.f && a >= threshold;
            out |= big ? 1u << j : 0u;
            amax = big ? amax : fmaxf(amax, a);
        }
        if (__builtin_amdgcn_ballot_w64(out != 0u) != 0ull) {  // eight lanes, a word
            out <<= k & 31;
            out |= __shfl_xor(out, 1);
            out |= __shfl_xor(out, 2);
            out |= __shfl_xor(out, 4);
            if ((threadIdx.x & 7) == 0 && out != 0u) atomicOr(mask + (k >> 5), out);
        }
        if (k < Kp) *(u32x2*)(xh + (int64_t)m * Kp + k) = u32x2{h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16)};
    }
    amax = block_max(amax, red);
    if (threadIdx.x == 0) sca[m] = amax;
}

// ---- 2. the int8 operand, the list of outlier columns (workgroup 0) and, by themselves, the outlier columns of the rows and of the weights: the
// epilogue then multiplies dense f16 matrices.  (It used to gather both per block of the product, a weight byte, a division and an f16 activation per element
// and token block: 295 us of a 512-token mlp.c_proj; and the list was one thread's chain of dependent loads: 25 of this launch's 30 us.)
// Workgroups 0 .. M - 1: a row each; the others: the weights, 16 rows x 32 columns per wave and turn.  Tables of the columns there are, and none of a
// call without outliers (2000 rows, N = K = 512, all launches of the product: 26.2 us with tables of 16 384 columns and 16 requests ahead above, 22.5 now; N = K = 1024 40.9, 37.1).
constexpr int kMaskWords = 512;  // of the mask per turn: 16 384 columns
constexpr int kQuantLds = 4 + 4 + 64;
__global__ __launch_bounds__(256) void i8_quant_kernel(const unsigned* mask, int8_t* ca, int* olist, const I8GemmParams p, int R) {
    extern __shared__ unsigned words[];  // kQuantLds bytes per word
    __shared__ int wave_tot[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int Kp = p.Kp, nw = Kp >> 5, m = blockIdx.x, held = nw < kMaskWords ? nw : kMaskWords;
    int* before = (int*)words + held;               // outlier columns in front of a word
    uint16_t* cols = (uint16_t*)(before + held);    // the outlier columns of this turn, from its first word on
    int n_out;
    {
        int c = 0;
        for (int w = threadIdx.x; w < nw; w += 256) c += __popc(mask[w]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
        if (lane == 0) wave_tot[wave] = c;
        __syncthreads();
        n_out = wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
    }
    const bool compact = is_compact(n_out, p.n_tiles, R, p.M);
    const int ld = compact_ld(n_out);
    const bool of_row = m < p.M;
    if (!of_row && !compact) return;
    const float a = of_row ? p.sca[m] : 0.f;
    const float inv = a > 0.f ? __fdiv_rn(127.0f, a) : 0.f;  // IEEE division: parity with the oracle
    if (m == 0 && threadIdx.x == 0) olist[0] = n_out;
    if (of_row && compact)
        for (int j = n_out + (int)threadIdx.x; j < ld; j += 256) p.xo[(int64_t)m * ld + j] = 0;
    int carry = 0;
    for (int w0 = 0; w0 < nw; w0 += kMaskWords) {
        const int cnt = nw - w0 < kMaskWords ? nw - w0 : kMaskWords;
        const int per = (cnt + 255) / 256, lo = threadIdx.x * per, hi = lo + per < cnt ? lo + per : cnt;
        const int j_lo = carry;  // outlier columns of this turn: j_lo .. j_hi - 1
        int j_hi = carry;
        if (n_out > 0) {
            __syncthreads();  // (the last turn is done with words, before and wave_tot)
            int c = 0;
            for (int w = lo; w < hi; ++w) {
                words[w] = mask[w0 + w];
                c += __popc(words[w]);
            }
            int incl = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(incl, o);
                if (lane >= o) incl += up;
            }
            if (lane == 63) wave_tot[wave] = incl;
            __syncthreads();
            int at = carry + incl - c;
            for (int w = 0; w < wave; ++w) at += wave_tot[w];
            j_hi = carry + wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
            carry = j_hi;
            for (int w = lo; w < hi; ++w) {
                before[w] = at;
                for (unsigned bits = words[w]; bits != 0u; ++at, bits &= bits - 1u) cols[at - j_lo] = (uint16_t)(w * 32 + __builtin_ctz(bits));
            }
            __syncthreads();
        }
        if (m == 0)
            for (int j = j_lo + (int)threadIdx.x; j < j_hi; j += 256) olist[1 + j] = w0 * 32 + cols[j - j_lo];
        if (of_row) {
            const f16_t* row = p.xh + (int64_t)m * Kp;
            constexpr int kAhead = 4;
            const int e4 = (w0 + cnt) * 8;
            for (int k0 = w0 * 8 + (int)threadIdx.x; k0 < e4; k0 += 256 * kAhead) {
                u32x2 hv[kAhead];
#pragma unroll
                for (int i = 0; i < kAhead; ++i) hv[i] = *(const u32x2*)(row + 4 * (k0 + 256 * i < e4 ? k0 + 256 * i : k0));
#pragma unroll
                for (int i = 0; i < kAhead; ++i) {
                    const int k4 = k0 + 256 * i;
                    if (k4 >= e4) continue;
                    const int k = 4 * k4, w = (k >> 5) - w0;
                    const unsigned bits = n_out > 0 ? words[w] >> (k & 31) : 0u;
                    uint32_t q4 = 0u;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f16_t h = (f16_t)((j & 1) ? (hv[i][j >> 1] >> 16) : (hv[i][j >> 1] & 0xffffu));
                        const bool out = (bits >> j) & 1u;
                        const float q = out ? 0.f : rintf(f16_to_f32(h) * inv);
                        q4 |= ((uint32_t)(int)q & 0xffu) << (8 * j);
                        if (out && compact) p.xo[(int64_t)m * ld + before[w] + __popc(words[w] & ((1u << ((k & 31) + j)) - 1u))] = h;
                    }
                    *(uint32_t*)(ca + (int64_t)m * Kp + k) = q4;
                }
            }
        } else {
            const int row = lane & 15, total = p.n_tiles * R;
            const bool last = w0 + cnt >= nw;
            const int jb0 = j_lo >> 5, jb1 = last ? ld >> 5 : (j_hi + 31) >> 5;
            // (items, units and bytes of the stream fit 32 bits; two items at a time, their bytes requested before the first is stored, eight columns to a store: 4096 rows, some 3000
            // outlier columns of 11 008 33 -> 22 us with the 512 rows beside them)
            const unsigned items = (unsigned)(jb1 - jb0) * (unsigned)total, stride = (gridDim.x - p.M) * 4u;
            for (unsigned it0 = (unsigned)(m - p.M) * 4u + wave; it0 < items; it0 += 2u * stride) {
                constexpr int kItems = 2;
                int8_t cb[kItems][8];
                float sc[kItems];
                int n[kItems], j0[kItems];
                f16_t* dst[kItems];
#pragma unroll
                for (int q = 0; q < kItems; ++q) {
                    const unsigned it = it0 + q * stride < items ? it0 + q * stride : it0, jb = it / (unsigned)total;
                    const int tr = (int)(it - jb * (unsigned)total), tl = tr / R, r1 = tr - tl * R;
                    n[q] = tl * 16 + row;
                    sc[q] = (r1 == 1 ? p.scb2 : p.scb)[n[q] < p.N ? n[q] : 0];
                    dst[q] = p.so + ((int64_t)tr * 16 + row) * ld;
                    j0[q] = (jb0 + (int)jb) * 32 + (lane >> 4) * 8;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int j = j0[q] + i;
                        const unsigned k = j >= j_lo && j < j_hi ? w0 * 32 + cols[j - j_lo] : 0;
                        cb[q][i] = (int8_t)p.w[((((unsigned)tl * p.units + (k >> 7)) * R + r1) * 2u + ((k >> 6) & 1u)) * 1024u + (((k >> 4) & 3u) * 16u + row) * 16u + (k & 15u)];
                    }
                }
#pragma unroll
                for (int q = 0; q < kItems; ++q) {
                    if (q > 0 && it0 + q * stride >= items) break;
                    if (nw <= kMaskWords) {  // (the only turn: every column of the row has its value, or zero, here)
                        u32x4 o;
#pragma unroll
                        for (int i = 0; i < 8; i += 2) {
                            auto at = [&](int e) { return n[q] < p.N && j0[q] + e < j_hi ? (uint32_t)f32_to_f16(__fdiv_rn((float)cb[q][e] * sc[q], 127.0f)) : 0u; };
                            o[i >> 1] = at(i) | (at(i + 1) << 16);
                        }
                        *(u32x4*)(dst[q] + j0[q]) = o;
                        continue;
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int j = j0[q] + i;
                        if (j >= j_lo && j < j_hi) dst[q][j] = n[q] < p.N ? f32_to_f16(__fdiv_rn((float)cb[q][i] * sc[q], 127.0f)) : (f16_t)0;
                        else if (last && j >= j_hi && j < ld) dst[q][j] = 0;
                    }
                }
            }
        }
    }
}

// ---- 3. the product
// MODE 0: product + epilogue; 1: product of one K-slice -> partial tiles; 2: sum of the partial tiles + epilogue
template <int EPI, bool PAIR, int MODE, int kWaves, int BM = kBM>
__global__ __launch_bounds__(64 * kWaves, 2) void i8_gemm_kernel(const I8GemmParams p) {
    static_assert(MODE != 2 || kWaves == 8, "a wave per token tile");
    static_assert(MODE == 0 || BM == kBM, "K-slices come in blocks of 128 tokens");
    constexpr int kXTile = BM * 128;  // bytes of one activation tile (int8)
    constexpr int kSlots = kWaves * kTPW, kThreads = 64 * kWaves;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int xcd = blockIdx.x & 7, j0 = blockIdx.x >> 3;
    const int L2 = xcd * p.per_xcd + j0;
    if (MODE != 2 && blockIdx.x == 0 && p.mask_next != nullptr)
        for (int i = threadIdx.x; i < p.mask_words; i += kThreads) p.mask_next[i] = 0u;
    // MODE 1: a workgroup per (block, K-slice); MODE 2: a workgroup per (block, 16-token tile) — 8 x the workgroups of the
    // product launch, so that summing the slices and the epilogue are not left to a dozen workgroups
    const int nsplit = MODE == 1 ? p.ksplit + 1 : MODE == 2 ? 8 : 1;
    if (j0 >= p.per_xcd || L2 >= p.total_blocks * nsplit) return;
    const int L = L2 / nsplit, ks = L2 - L * nsplit;
    // MODE 2: workgroup ks of a block finishes the rows of slot group ks (the rows wave ks owns in the product launch) for all 128
    // tokens, wave w its token tile w
    constexpr int kTT = MODE == 2 ? 1 : BM / 16;                               // token tiles a wave finishes, from tt0 on
    const int tt0 = MODE == 2 ? wave : 0;
    const int wslot = MODE == 2 ? ks : wave;                                   // slot group of this wave's row tiles
    // row block major: an XCD runs every token block of a few row blocks side by side, so their weights cross to its L2 once
    const int m_blocks = p.total_blocks / p.n_blocks, nb = L / m_blocks, mb = L - nb * m_blocks;
    const int m0 = mb * BM;
    const int u_lo = MODE == 1 ? (int)((int64_t)ks * p.units / p.ksplit) : 0;
    const int u_hi = MODE == 1 ? (int)((int64_t)(ks + 1) * p.units / p.ksplit) : p.units;
    constexpr int R = PAIR ? 2 : 1;

    int tile[kTPW], rr[kTPW];
#pragma unroll
    for (int t = 0; t < kTPW; ++t) {
        if (PAIR) {
            tile[t] = nb * (kSlots / 2) + (kTPW / 2) * wslot + (t >> 1);  // pair tile: 16 rows of c_fc1 (r = 0) and c_fc2 (r = 1)
            rr[t] = t & 1;
        } else {
            tile[t] = nb * kSlots + kTPW * wslot + t;
            rr[t] = 0;
        }
    }
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, (int)p.w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw0 = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void*)p.ca, 0, (int)((int64_t)p.M * p.Kp), 0x00020000);
    const unsigned lane_off = lane * 16;
    i32x4 acc[kTPW][kTT];
#pragma unroll
    for (int t = 0; t < kTPW; ++t)
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) acc[t][tt] = i32x4{0, 0, 0, 0};

    // The units of a product: int8 units of 128 columns, or (F16) units of 64 compact outlier columns — 128 B of a token either way.  The weights (registers) and
    // the activations (LDS, by DMA, the swizzle on the source's side) of the next kDepth - 1 units are under way; a unit waits for its own requests by
    // count, and the requests go out between the products (as gemm_deep_kernel: csrc/gemm.hip).  One unit ahead, waited for in front of its LDS stores, a unit
    // took 1.56 us at one workgroup per CU
    constexpr int kXI = BM / 8 / kWaves, kUnit = kXI + 2 * kTPW;  // requests per wave and unit: 1 KiB = 8 tokens of activations; weight pieces
    auto run_units = [&](auto f16, auto& sum, int lo, int hi, __amdgpu_buffer_rsrc_t rwt, __amdgpu_buffer_rsrc_t rxt, int64_t ldb) {
        constexpr bool F16 = decltype(f16)::value;
        typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_l;
        unsigned xoff[kXI];
        int xdst[kXI];
#pragma unroll
        for (int i = 0; i < kXI; ++i) {
            const int q = i * kWaves + wave, tok = q * 8 + (lane >> 3), slot = lane & 7;
            xoff[i] = m0 + tok < p.M ? (unsigned)((int64_t)(m0 + tok) * ldb) + (unsigned)((slot ^ swz8(tok)) * 16) : 0xFFFFFFF0u;
            xdst[i] = q * 1024;
        }
        const unsigned w_lane = F16 ? (unsigned)(c * ldb + g * 16) : lane_off;
        u32x4 wr[kDepth][kTPW][2];
        auto request = [&](int i, int u, int slot) __attribute__((always_inline)) {
            const bool in = u < hi;
            if (i < kXI) {
                const unsigned off = in && xoff[i < kXI ? i : 0] != 0xFFFFFFF0u ? xoff[i < kXI ? i : 0] + (unsigned)u * 128u : 0xFFFFFFF0u;
                i8_lds_from(rxt, smem + slot * kXTile + xdst[i < kXI ? i : 0], off);
            } else {
                const int t = (i - kXI) / 2, e = (i - kXI) % 2;
                const bool ok = tile[t] < p.n_tiles && in;
                const unsigned off = F16 ? (unsigned)((int64_t)(tile[t] * R + rr[t]) * 16 * ldb) + (unsigned)u * 128u + e * 64u
                                         : (unsigned)((tile[t] * p.units + u) * R + rr[t]) * 2048u + e * 1024u;
                wr[slot][t][e] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ok ? rwt : rw0, w_lane, ok ? off : 0u, 0));
            }
        };
#pragma unroll
        for (int d = 0; d < kDepth - 1; ++d) {
#pragma unroll
            for (int i = 0; i < kUnit; ++i) request(i, lo + d, d);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto products = [&](int slot, int ahead, int ahead_slot, auto more) __attribute__((always_inline)) {
            const char* xs = smem + slot * kXTile;
            constexpr int kT = BM / 16, kFrags = 2 * kT, kPipe = 4;  // fragment f = e * kT + tt
            auto bread = [&](int f) {
                const int tok = (f % kT) * 16 + c;
                return *(const i32x4*)(xs + tok * 128 + (((4 * (f / kT) + g) ^ swz8(tok)) << 4));
            };
            i32x4 bq[kPipe];
#pragma unroll
            for (int q = 0; q < kPipe; ++q) bq[q] = bread(q);
            __builtin_amdgcn_sched_group_barrier(0x100, kPipe, 0);
#pragma unroll
            for (int f = 0; f < kFrags; ++f) {
                const i32x4 b = bq[f % kPipe];
                if (f + kPipe < kFrags) bq[f % kPipe] = bread(f + kPipe);
#pragma unroll
                for (int t = 0; t < kTPW; ++t) {
                    if constexpr (F16)
                        sum[t][f % kT] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_l, wr[slot][t][f / kT]),
                                                                               __builtin_bit_cast(f16x8_l, b), sum[t][f % kT], 0, 0, 0);
                    else
                        sum[t][f % kT] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, wr[slot][t][f / kT]), b, sum[t][f % kT], 0, 0, 0);
                }
                if (f + kPipe < kFrags) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, kTPW, 0);
                constexpr int kEvery = kFrags / kUnit;  // (spread over the unit: csrc/gemm.hip)
                if (more && f % kEvery == 0 && f / kEvery < kUnit) {
                    request(f / kEvery, ahead, ahead_slot);
                    __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // (the last, shorter round stands behind the loop and requests nothing: with a way out between the units hipcc waited for every request once a round)
        auto unit = [&](auto slot, int u, auto more) __attribute__((always_inline)) {
            constexpr int d = slot, kNewer = more ? (kDepth - 2) * kUnit : (kDepth - 2 - d) * kUnit;
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kNewer) : "memory");
            products(d, u + kDepth - 1, (d + kDepth - 1) % kDepth, more);
        };
        using std::integral_constant;
        int u = lo;
        for (; u + kDepth <= hi; u += kDepth) {
            unit(integral_constant<int, 0>{}, u, std::true_type{});
            unit(integral_constant<int, 1>{}, u + 1, std::true_type{});
            unit(integral_constant<int, 2>{}, u + 2, std::true_type{});
            unit(integral_constant<int, 3>{}, u + 3, std::true_type{});
        }
        if (u < hi) {
            unit(integral_constant<int, 0>{}, u, std::false_type{});
            if (u + 1 < hi) {
                unit(integral_constant<int, 1>{}, u + 1, std::false_type{});
                if (u + 2 < hi) unit(integral_constant<int, 2>{}, u + 2, std::false_type{});
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (requests past the end wrote zeros: none may land in what follows)
        __syncthreads();
    };
    const int n_out = MODE == 1 && ks < p.ksplit ? 0 : p.olist[0];
    const bool compact = is_compact(n_out, p.n_tiles, R, p.M);
    f32x4 o[kTPW][kTT];  // the outlier columns' share
    auto no_outliers = [&]() {
#pragma unroll
        for (int t = 0; t < kTPW; ++t)
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) o[t][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    auto outliers = [&]() {
        no_outliers();
        const int ld = compact_ld(n_out);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)p.so, 0, p.n_tiles * R * 16 * ld * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void*)p.xo, 0, p.M * ld * 2, 0x00020000);
        run_units(std::true_type{}, o, 0, ld / 64, rs, ro, (int64_t)ld * 2);
    };
    if constexpr (MODE == 1) {
        if (ks == p.ksplit) {  // the launch's last slice: the outlier columns
            if (!compact) return;
            outliers();
#pragma unroll
            for (int tt = 0; tt < 8; ++tt) {
                const int m = m0 + tt * 16 + c;
                if (m >= p.M) continue;
#pragma unroll
                for (int t = 0; t < kTPW; ++t) {
                    const int n = tile[t] * 16 + 4 * g;
                    if (tile[t] < p.n_tiles && n < p.N)
                        *(f32x4*)((float*)p.part + ((int64_t)ks * p.M + m) * p.ldp + (PAIR && rr[t] == 1 ? p.ldn : 0) + n) = o[t][tt];
                }
            }
            return;
        }
    }
    if constexpr (MODE != 2) run_units(std::false_type{}, acc, u_lo, u_hi, rw, rx, (int64_t)p.Kp);
    // partial tiles of a K-slice: column n of c_fc2 sits at ldn + n
    if constexpr (MODE == 1) {
#pragma unroll
        for (int tt = 0; tt < 8; ++tt) {
            const int m = m0 + tt * 16 + c;
            if (m >= p.M) continue;
#pragma unroll
            for (int t = 0; t < kTPW; ++t) {
                const int n = tile[t] * 16 + 4 * g;
                if (tile[t] < p.n_tiles && n < p.N)
                    *(i32x4*)(p.part + ((int64_t)ks * p.M + m) * p.ldp + (PAIR && rr[t] == 1 ? p.ldn : 0) + n) = acc[t][tt];
            }
        }
        return;
    }
    if constexpr (MODE == 2) {  // all slices requested before the first is added (one at a time was a memory round trip each)
        const int m = m0 + tt0 * 16 + c;
#pragma unroll
        for (int t = 0; t < kTPW; ++t) {
            const int n = tile[t] * 16 + 4 * g;
            const int* at = p.part + (m < p.M && tile[t] < p.n_tiles && n < p.N ? (int64_t)m * p.ldp + (PAIR && rr[t] == 1 ? p.ldn : 0) + n : 0);
            i32x4 v[kMaxSplit];
#pragma unroll
            for (int s2 = 0; s2 < kMaxSplit; ++s2) v[s2] = *(const i32x4*)(at + (s2 < p.ksplit ? s2 : 0) * ((int64_t)p.M * p.ldp));
#pragma unroll
            for (int s2 = 0; s2 < kMaxSplit; ++s2)
                if (s2 < p.ksplit) acc[t][0] += v[s2];
            if (compact) o[t][0] = *(const f32x4*)((const float*)at + p.ksplit * ((int64_t)p.M * p.ldp));
        }
    }

    // ---- epilogue.  lane (g, c) holds rows 4 g .. 4 g + 3 of its tiles for token tt * 16 + c.  Loads without a branch between them
    float scb[kTPW][4], sa[kTT];
#pragma unroll
    for (int t = 0; t < kTPW; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = tile[t] * 16 + 4 * g + r;
            scb[t][r] = ((PAIR && rr[t] == 1) ? p.scb2 : p.scb)[n < p.N ? n : 0];
        }
#pragma unroll
    for (int tt = 0; tt < kTT; ++tt) {
        const int m = m0 + (tt0 + tt) * 16 + c;
        sa[tt] = p.sca[m < p.M ? m : 0];
    }
    typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
    if (compact) {
        if constexpr (MODE == 0) outliers();
    } else if (n_out > 0) {  // (too many for their region)
        // mixed-precision decomposition: the outlier columns in f16, ascending k, kOutChunk columns per pass through LDS
        f16_t* xo = (f16_t*)smem;                     // [BM tokens][kOutChunk]
        f16_t* so = xo + BM * kOutChunk;              // [kSlots x 16 rows][kOutChunk]: f16(CB[n, k] * SCB[n] / 127)
        // (the side product runs on v_mfma_f32_16x16x32_f16 — A = 16 rows x 32 outlier columns of `so`, B = 16 tokens x the same
        // columns of `xo`, result in the accumulators' own layout: lane (g, c) holds rows 4 g .. 4 g + 3 for token c.  The products of two f16
        // values are exact in f32 and the sum is f32 as before; its ORDER inside a block of 32 columns is the hardware's instead of
        // ascending k — bitsandbytes' own f16 GEMM promises no order either, and the tests allow the one f16 ulp this can move.  The scalar
        // loop it replaces (64 FMAs per lane and outlier column) took 1.4 ms per attn.c_proj / mlp.c_proj launch at T = 2048, where ~10 % of
        // the columns of a 2048-token call hold an outlier: profiles/r06_prefill_int8_outliers.txt.)
        no_outliers();
        for (int base = 0; base < n_out; base += kOutChunk) {
            const int nc = n_out - base < kOutChunk ? n_out - base : kOutChunk;
            __syncthreads();  // (the main loop / the previous pass is done with the LDS)
            // a thread's outlier column is the same in every iteration (kThreads is a multiple of kOutChunk): its list entry and
            // the column's place inside a unit are read once per pass, which leaves ONE gather per element in loops that can be unrolled
            // (with the list read inside, each of the 32 iterations waited for two dependent loads: ~40 us per pass of 64 columns)
            static_assert(kThreads % kOutChunk == 0 && (kOutChunk & (kOutChunk - 1)) == 0, "column index per thread is loop-invariant");
            const int oi = threadIdx.x & (kOutChunk - 1);
            const bool col_ok = oi < nc;
            const int k = col_ok ? p.olist[1 + base + oi] : 0;
#pragma unroll 8
            for (int idx = threadIdx.x; idx < BM * kOutChunk; idx += kThreads) {
                const int tok = idx / kOutChunk;
                const int m = m0 + tok;
                xo[idx] = (m < p.M && col_ok) ? p.xh[(int64_t)m * p.Kp + k] : (f16_t)0;
            }
            // weights: ROW fastest — 16 lanes = the 16 rows of a tile at one outlier column (16 B apart in the stream: two cache lines),
            // four columns per wave (the column-fastest order touched 64 lines per wave load); a thread sees kCols columns, kStep apart
            constexpr int kStep = kThreads / 16, kCols = kOutChunk / kStep;
            const int oc = threadIdx.x >> 4, row = threadIdx.x & 15;
            int k2[kCols];
#pragma unroll
            for (int h = 0; h < kCols; ++h) k2[h] = oc + kStep * h < nc ? p.olist[1 + base + oc + kStep * h] : -1;
            const int s_lo = MODE == 2 ? ks * kTPW : 0, s_hi = MODE == 2 ? s_lo + kTPW : kSlots;  // MODE 2: the rows of slot group ks only
#pragma unroll 4
            for (int slot = s_lo; slot < s_hi; ++slot) {
                const int wv = slot / kTPW, t = slot - wv * kTPW;
                int tl, r1;
                if (PAIR) {
                    tl = nb * (kSlots / 2) + (kTPW / 2) * wv + (t >> 1);
                    r1 = t & 1;
                } else {
                    tl = nb * kSlots + kTPW * wv + t;
                    r1 = 0;
                }
                const int n = tl * 16 + row;
#pragma unroll
                for (int h = 0; h < kCols; ++h) {
                    const int kk = k2[h];
                    f16_t sub = 0;
                    if (kk >= 0 && tl < p.n_tiles && n < p.N) {
                        const int ku = kk >> 7, ke = (kk >> 6) & 1, kgg = (kk >> 4) & 3, kjj = kk & 15;
                        const int64_t off = ((((int64_t)tl * p.units + ku) * R + r1) * 2 + ke) * 1024 + (kgg * 16 + row) * 16 + kjj;
                        const float cb = (float)(int8_t)p.w[off];
                        const float s = ((PAIR && r1 == 1) ? p.scb2 : p.scb)[n];
                        sub = f32_to_f16(__fdiv_rn(cb * s, 127.0f));
                    }
                    so[(slot * 16 + row) * kSoLd + oc + kStep * h] = sub;
                }
            }
            __syncthreads();
#pragma unroll
            for (int kb = 0; kb < kOutChunk / 32; ++kb) {
                if (kb * 32 >= nc) break;
                f16x8_t a[kTPW];
#pragma unroll
                for (int t = 0; t < kTPW; ++t) a[t] = *(const f16x8_t*)(so + ((wslot * kTPW + t) * 16 + c) * kSoLd + kb * 32 + 8 * g);
#pragma unroll
                for (int tt = 0; tt < kTT; ++tt) {
                    const f16x8_t b = *(const f16x8_t*)(xo + ((tt0 + tt) * 16 + c) * kOutChunk + kb * 32 + 8 * g);
#pragma unroll
                    for (int t = 0; t < kTPW; ++t) o[t][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b, o[t][tt], 0, 0, 0);
                }
            }
        }
    }
    // the result at row r of tile t, token tile tt; with outliers the mixed-precision decomposition over them, ascending k, comes on top
    auto value = [&](int t, int tt) {
        f32x4 d;
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = f16r_of_f32((((float)acc[t][tt][r] * 6.200012e-05f) * sa[tt]) * scb[t][r]);
        if (n_out > 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) d[r] = f16r(d[r] + f16r(o[t][tt][r]));
        return d;
    };
    // four consecutive output columns per lane and tile: one 16-B (f32) / 8-B (bf16, f16) access when the row allows it
    const bool vec = (p.N & 3) == 0 && (p.ldy & 3) == 0 && ((uintptr_t)p.y & 15) == 0;
    constexpr int kOld = kTT < 2 ? kTT : 2;
    [[maybe_unused]] f32x4 old[kTPW][kOld];  // ACCUM, f32 rows: of kOld token tiles at a time
#pragma unroll
    for (int tt = 0; tt < kTT; ++tt) {
        const int m = m0 + (tt0 + tt) * 16 + c;
        if constexpr (EPI == MI355_EPI_ACCUM) {
            if (tt % kOld == 0 && vec && p.y_dtype == MI355_F32) {
#pragma unroll
                for (int i = 0; i < kOld; ++i)
#pragma unroll
                    for (int t = 0; t < kTPW; ++t) {
                        const int mi = m + 16 * i, n = tile[t] * 16 + 4 * g;
                        old[t][i] = *(const f32x4*)((const float*)p.y + (mi < p.M && tile[t] < p.n_tiles && n < p.N ? (int64_t)mi * p.ldy + n : 0));
                    }
            }
        }
        if (m >= p.M) continue;
        if constexpr (EPI == MI355_EPI_SWIGLU) {
#pragma unroll
            for (int t = 0; t < kTPW; t += 2) {
                const int n = tile[t] * 16 + 4 * g;
                if (tile[t] >= p.n_tiles || n >= p.N) continue;
                const f32x4 a = value(t, tt), b = value(t + 1, tt);
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = swiglu_f32(a[r], b[r]);
                if (vec && p.y_dtype == MI355_BF16) {
                    u32x2 pk;
                    pk[0] = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
                    pk[1] = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
                    *(u32x2*)((bf16_t*)p.y + (int64_t)m * p.ldy + n) = pk;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n + r < p.N) st_from_f32(p.y, (int64_t)m * p.ldy + n + r, p.y_dtype, v[r]);
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < kTPW; ++t) {
                const int n = tile[t] * 16 + 4 * g;
                if (tile[t] >= p.n_tiles || n >= p.N) continue;
                const int64_t yi = (int64_t)m * p.ldy + n;
                const f32x4 d = value(t, tt);
                if (vec && p.y_dtype == MI355_F32) {
                    f32x4 o = d;
                    if constexpr (EPI == MI355_EPI_ACCUM) o += old[t][tt % kOld];
                    *(f32x4*)((float*)p.y + yi) = o;
                } else if (vec && p.y_dtype == MI355_BF16) {
                    float o[4] = {d[0], d[1], d[2], d[3]};
                    if constexpr (EPI == MI355_EPI_ACCUM) {
                        const u32x2 old = *(const u32x2*)((const bf16_t*)p.y + yi);
                        o[0] += __uint_as_float(old[0] << 16);
                        o[1] += __uint_as_float(old[0] & 0xffff0000u);
                        o[2] += __uint_as_float(old[1] << 16);
                        o[3] += __uint_as_float(old[1] & 0xffff0000u);
                    }
                    u32x2 pk;
                    pk[0] = (uint32_t)f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16);
                    pk[1] = (uint32_t)f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16);
                    *(u32x2*)((bf16_t*)p.y + yi) = pk;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (n + r >= p.N) continue;
                        float v = d[r];
                        if constexpr (EPI == MI355_EPI_ACCUM) v += ld_as_f32(p.y, yi + r, p.y_dtype);
                        st_from_f32(p.y, yi + r, p.y_dtype, v);
                    }
                }
            }
        }
    }
}

template <int EPI, bool PAIR, int MODE, int kWaves, int BM = kBM>
int launch_i8_mode(const I8GemmParams& q, hipStream_t s) {
    constexpr int lds = kLds<kWaves, BM>;
    static hipError_t attr_err =
        hipFuncSetAttribute((const void*)i8_gemm_kernel<EPI, PAIR, MODE, kWaves, BM>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr_err != hipSuccess) {
        mi355_set_error("hipFuncSetAttribute(i8_gemm) failed: %s", hipGetErrorString(attr_err));
        return (int)attr_err;
    }
    I8GemmParams r = q;
    r.n_blocks = (q.n_tiles + kWaves * kTPW / (PAIR ? 2 : 1) - 1) / (kWaves * kTPW / (PAIR ? 2 : 1));
    r.total_blocks = r.n_blocks * ((q.M + BM - 1) / BM);
    r.per_xcd = (r.total_blocks * (MODE == 1 ? q.ksplit + 1 : MODE == 2 ? 8 : 1) + 7) / 8;
    hipLaunchKernelGGL((i8_gemm_kernel<EPI, PAIR, MODE, kWaves, BM>), dim3(8 * r.per_xcd), dim3(64 * kWaves), lds, s, r);
    MI355_LAUNCH_CHECK();
    return 0;
}
// How a launch is cut: blocks of 128 tokens x 256 rows (8 waves) or x 128 (4 waves), and K-slices, which are a sum and its launch more; what an estimate takes for the
// fastest.  A launch in K-slices has one slice's workgroups more for the outlier columns, and a CU that gets one of them runs it beside or behind its other work: 64
// blocks of 4 waves (N = K = 8192, 33 tokens) take 44.7 / 39.5 / 34.2 / 41.3 / 38.1 us with 1 / 2 / 3 / 4 / 5 slices, since 4 are 320 workgroups and not 256.  So: the
// rounds of the chip, each the units of a slice or the launch's share of the weights from HBM, whichever is longer (a root of squares), and for slices a launch and the
// sums' way to memory and back.  How many outlier columns there are is on the device; the constants are those whose choice is best over 2688 launches (32 products of
// 768 to 32000 rows, 32 to 2048 tokens, 0, 0.3, 2 and 10 % of the columns, weights not in any cache: profiles/product_cuts_int8.txt): 0.5 % behind the fastest on average, 2 %
// at the 90th percentile; with the outliers' workgroups left out 1.6 % and 5 %, and N = 5120, K = 13824, 256 tokens 79 us (now 66).  Blocks of 8 waves throughout and
// slices for launches of less than 96 of them: 1.23 times as long on average, none more than 2.5 % shorter.
// Blocks of 64 tokens x 128 rows (whole rows only) where they bring work to idle CUs: 512 tokens, N = 4096, K = 4096 35.8 -> 31.4 us, K = 11008 73.2 -> 59.2, with 2750 outlier columns 154 -> 136
// (128 blocks -> 256; staging and quantisation with it); of 493 launches (13 products, 33 to 2048 tokens, 0, 2 and 25 % of the columns) the rule takes them in 167, 0.90 times as long, 2.6 % longer at worst
// (profiles/product_cuts_int8.txt has 585 of that kind).
struct I8Cut {
    int waves, ksplit, bm;
};
int i8_part_columns(int N) { return (N + 3) & ~3; }
I8Cut i8_cut(int M, int N, int units, bool pair) {
    struct Kind {
        int waves, bm;
        float start, unit;
    };
    static constexpr Kind kinds[] = {{4, kBM, 0.21f, 0.436f}, {8, kBM, 0.737f, 0.763f}, {4, 64, 0.f, 0.41f}};
    const size_t part = (size_t)M * i8_part_columns(N) * (pair ? 2 : 1) * 4;  // bytes of one slice's sums
    I8Cut cut = {8, 1, kBM};
    float best = 0.f;
    for (const Kind& k : kinds)
        for (int ks = 1; ks <= (k.bm == kBM ? kMaxSplit : 1) && (ks == 1 || (units >= 4 * ks && part * ks <= kSplitBudget)); ++ks) {
            const int rows = 16 * k.waves * kTPW / (pair ? 2 : 1), blocks = (N + rows - 1) / rows * ((M + k.bm - 1) / k.bm) * (ks == 1 ? 1 : ks + 1);
            auto round = [&](int of) {
                const float work = (float)((units + ks - 1) / ks) * k.unit, hbm = 0.557f + 128.f * units * N * (pair ? 2 : 1) / 2.03e6f * (float)of / (float)blocks;
                return sqrtf(work * work + hbm * hbm);
            };
            const float us = k.start + (float)(blocks / 256) * round(256) + (blocks % 256 ? round(blocks % 256) : 0.f) + (ks == 1 ? 0.f : 3.19f + (float)(part * ks) / 2.29e6f);
            if (best == 0.f || us < best) best = us, cut = {k.waves, ks, k.bm};
        }
    struct Force {
        int waves, bm, ksplit;
    };
    static const Force fo = [] {  // (sweeps: MI355_GEMM_FORCE as in csrc/gemm.hip)
        Force f = {0, 0, 0};
        if (const char* e = getenv("MI355_GEMM_FORCE")) sscanf(e, "%d:%d:%d", &f.waves, &f.bm, &f.ksplit);
        return f;
    }();
    if ((fo.waves == 4 || fo.waves == 8) && (fo.bm == 0 || fo.bm == kBM || (fo.bm == 64 && fo.waves == 4))) cut.waves = fo.waves, cut.bm = fo.bm ? fo.bm : cut.bm;
    if (fo.ksplit >= 1 && fo.ksplit <= kMaxSplit && units >= 4 * fo.ksplit && part * fo.ksplit <= kSplitBudget) cut.ksplit = fo.ksplit;
    if (cut.waves != 4 || cut.ksplit > 1) cut.bm = kBM;
    return cut;
}
template <int EPI, bool PAIR>
int launch_i8_gemm(const I8GemmParams& p, const I8Cut& cut, hipStream_t s) {
    const int waves = cut.waves;
    if (cut.bm == 64) return launch_i8_mode<EPI, PAIR, 0, 4, 64>(p, s);
    if (p.ksplit <= 1) return waves == 4 ? launch_i8_mode<EPI, PAIR, 0, 4>(p, s) : launch_i8_mode<EPI, PAIR, 0, 8>(p, s);
    if (int rc = waves == 4 ? launch_i8_mode<EPI, PAIR, 1, 4>(p, s) : launch_i8_mode<EPI, PAIR, 1, 8>(p, s)) return rc;
    return launch_i8_mode<EPI, PAIR, 2, 8>(p, s);
}

size_t pad16(size_t v) { return (v + 15) & ~(size_t)15; }

}  // namespace

extern "C" size_t mi355_linear_int8_gemm_workspace_bytes(int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    const size_t kp = ((size_t)K + 127) / 128 * 128;
    // xh f16 [M, Kp], CA int8 [M, Kp], absmax [M], column mask [Kp / 32], outlier list [1 + Kp]
    return pad16((size_t)M * kp * 2) + pad16((size_t)M * kp) + pad16((size_t)M * 4) + pad16(kp / 8) + pad16((1 + kp) * 4) + 256 +
           kPartBytes +                                      // partial tiles of the split-K launches (short prompts)
           pad16((size_t)M * kp * 2) + kOutlierBudget +      // outlier columns by themselves: of the rows, of the weights
           mi355_i8_chain_bytes(K);                          // the mask of a chain of products
}
extern "C" void mi355_linear_int8_gemm_plan(int M, int N, int K, int R, int* waves, int* ksplit) {
    const I8Cut cut = i8_cut(M, N, (K + 127) / 128, R == 2);
    *waves = cut.waves, *ksplit = cut.ksplit;
}
size_t mi355_i8_chain_bytes(int K) { return pad16(((size_t)K + 127) / 128 * 16); }

extern "C" int mi355_linear_int8_gemm(const mi355_int8_args* a, void* workspace, size_t workspace_bytes, mi355_stream_t stream) {
    return mi355_linear_int8_gemm_chained(a, nullptr, workspace, workspace_bytes, stream);
}

int mi355_linear_int8_gemm_chained(const mi355_int8_args* a, mi355_i8_chain* chain, void* workspace, size_t workspace_bytes, mi355_stream_t stream) {
    MI355_CHECK_ARG(a != nullptr && workspace != nullptr && a->w && a->scb && a->x && a->y, MI355_E_ARG, "linear_int8_gemm: null argument");
    MI355_CHECK_ARG(a->R == 1 || a->R == 2, MI355_E_ARG, "linear_int8_gemm: R must be 1 or 2");
    MI355_CHECK_ARG(a->M >= 1 && a->N > 0 && a->K > 0, MI355_E_SHAPE, "linear_int8_gemm: bad shape M=%d N=%d K=%d", a->M, a->N, a->K);
    MI355_CHECK_ARG(a->epi >= MI355_EPI_STORE && a->epi <= MI355_EPI_SWIGLU, MI355_E_ARG, "linear_int8_gemm: bad epi");
    const bool swiglu = a->epi == MI355_EPI_SWIGLU;
    MI355_CHECK_ARG(swiglu ? (a->R == 2 && a->scb2) : a->R == 1, MI355_E_ARG,
                    "linear_int8_gemm: STORE / ACCUM take the R = 1 stream, SWIGLU the interleaved R = 2 stream");
    MI355_CHECK_ARG(a->bias == nullptr && a->attn_partials == nullptr, MI355_E_ARG, "linear_int8_gemm: no bias / attention prologue");
    auto three = [](int d) { return d == MI355_F32 || d == MI355_BF16 || d == MI355_F16; };
    MI355_CHECK_ARG(three(a->x_dtype) && three(a->y_dtype), MI355_E_DTYPE, "linear_int8_gemm: x / y dtype");
    MI355_CHECK_ARG(a->norm_scale == nullptr || three(a->norm_dtype), MI355_E_DTYPE, "linear_int8_gemm: norm scale dtype");
    MI355_CHECK_ARG(workspace_bytes >= mi355_linear_int8_gemm_workspace_bytes(a->M, a->K) && (uintptr_t)workspace % 16 == 0,
                    MI355_E_SHAPE, "linear_int8_gemm: workspace of %zu bytes is too small (need %zu)", workspace_bytes,
                    mi355_linear_int8_gemm_workspace_bytes(a->M, a->K));
    hipStream_t s = (hipStream_t)stream;
    const int units = (a->K + 127) / 128, kp = units * 128;
    MI355_CHECK_ARG((size_t)a->M * kp < 0xFFFFFFF0ull, MI355_E_SHAPE, "linear_int8_gemm: M x K too large for one launch");
    char* ws = (char*)workspace;
    f16_t* xh = (f16_t*)ws;
    ws += pad16((size_t)a->M * kp * 2);
    int8_t* ca = (int8_t*)ws;
    ws += pad16((size_t)a->M * kp);
    float* sca = (float*)ws;
    ws += pad16((size_t)a->M * 4);
    MI355_CHECK_ARG(chain == nullptr || chain->words >= kp / 32, MI355_E_ARG, "linear_int8_gemm: a chain's mask of %d words for rows of %d", chain->words, a->K);
    unsigned* mask = chain != nullptr ? chain->mask : (unsigned*)ws;
    ws += pad16((size_t)kp / 8);
    int* olist = (int*)ws;
    ws += pad16((size_t)(1 + kp) * 4);
    int* part = (int*)ws;
    ws += kPartBytes;
    f16_t* xo = (f16_t*)ws;
    ws += pad16((size_t)a->M * kp * 2);
    f16_t* so = (f16_t*)ws;
    const I8Cut cut = i8_cut(a->M, a->N, units, swiglu);
    const int ksplit = cut.ksplit;
    const int ldn = i8_part_columns(a->N);
    // (a kernel, not hipMemsetAsync: a caller may capture this launch, and memset nodes have replayed wrongly)
    if (chain == nullptr || !chain->clear) {
        hipLaunchKernelGGL(i8_clear_mask_kernel, dim3((kp / 32 + 255) / 256), dim3(256), 0, s, mask, kp / 32);
        MI355_LAUNCH_CHECK();
    }
    auto stage = [&](auto type) {
        using T = decltype(type);
        const size_t norm_four = a->norm_dtype == MI355_F32 ? 16 : 8;
        const bool fours = a->K % 4 == 0 && a->ldx % 4 == 0 && (uintptr_t)a->x % (4 * sizeof(T)) == 0 && (uintptr_t)a->norm_scale % norm_four == 0 && kp <= 24 * 1024;
        auto held = kp <= 1024    ? i8_stage_fours_kernel<T, 1>
                    : kp <= 2048  ? i8_stage_fours_kernel<T, 2>
                    : kp <= 4096  ? i8_stage_fours_kernel<T, 4>
                    : kp <= 8192  ? i8_stage_fours_kernel<T, 8>
                    : kp <= 12288 ? i8_stage_fours_kernel<T, 12>
                    : kp <= 16384 ? i8_stage_fours_kernel<T, 16>
                    : kp <= 20480 ? i8_stage_fours_kernel<T, 20>
                                  : i8_stage_fours_kernel<T, 24>;
        auto kernel = fours ? held : kp <= 1024 ? i8_stage_kernel<T, 4> : kp <= 2048 ? i8_stage_kernel<T, 8> : i8_stage_kernel<T, 16>;
        hipLaunchKernelGGL(kernel, dim3(a->M), dim3(256), 0, s, (const T*)a->x, a->ldx, a->norm_scale, a->norm_dtype, a->eps, a->threshold, a->K, kp, xh, sca, mask);
    };
    if (a->x_dtype == MI355_F32) stage(float{});
    else if (a->x_dtype == MI355_BF16) stage(bf16_t{});
    else stage(f16_raw{});
    MI355_LAUNCH_CHECK();
    I8GemmParams p;
    memset(&p, 0, sizeof(p));
    p.w = (const uint8_t*)a->w;
    {
        const size_t wb = mi355_packed_bytes(MI355_W_I8, a->N, a->K, a->R, swiglu ? 1 : 0);
        MI355_CHECK_ARG(wb > 0 && wb < 0xFFFFFFF0ull, MI355_E_SHAPE, "linear_int8_gemm: weight stream of %zu B", wb);
        p.w_bytes = (unsigned)wb;
    }
    p.ca = ca;
    p.xh = xh;
    p.sca = sca;
    p.olist = olist;
    p.scb = a->scb;
    p.scb2 = a->scb2;
    p.y = a->y;
    p.ldy = a->ldy;
    p.M = a->M;
    p.N = a->N;
    p.K = a->K;
    p.Kp = kp;
    p.units = units;
    p.n_tiles = (a->N + 15) / 16;
    p.y_dtype = a->y_dtype;
    p.ksplit = ksplit;
    p.ldn = ldn;
    p.ldp = (int64_t)ldn * (swiglu ? 2 : 1);
    p.part = part;
    p.xo = xo;
    p.so = so;
    if (chain != nullptr) {
        p.mask_next = chain->mask;
        p.mask_words = chain->words;
        chain->clear = true;
    }
    hipLaunchKernelGGL(i8_quant_kernel, dim3(a->M + 512), dim3(256), (kp / 32 < kMaskWords ? kp / 32 : kMaskWords) * kQuantLds, s, mask, ca, olist, p, a->R);
    MI355_LAUNCH_CHECK();
    if (swiglu) return launch_i8_gemm<MI355_EPI_SWIGLU, true>(p, cut, s);
    if (a->epi == MI355_EPI_ACCUM) return launch_i8_gemm<MI355_EPI_ACCUM, false>(p, cut, s);
    return launch_i8_gemm<MI355_EPI_STORE, false>(p, cut, s);
}
