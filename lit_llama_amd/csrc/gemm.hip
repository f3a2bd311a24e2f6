// Wide (several tokens) linear over the int4 or the bf16 weight stream for gfx950: prompt prefill, no-cache evaluation, batches of decoding sequences.
//
// Replaces the reference's Triton `linear_kernel_4bit_weight` (lit_llama/quantization.py:187-333,
// reached from ColBlockQuantizedLinear.forward :413-421) at the shapes of evaluate/full.py:120-129 (T = 2048, no cache)
// and of generate.py's prompt pass — where the skinny weight-streaming kernel (gemv.hip) re-reads the whole weight
// stream once per 13 tokens.
//
// Design (gemm_q4_kernel, the int4 stream; BF16, launches of about one workgroup per CU and grouped scales: gemm_deep_kernel, up to three units of operands under way):
//  * the weights stay in the decode path's stream layout [tile of 16 rows][unit of 128 k][r][lane][16 B]: a wave reads
//    a (tile, unit) piece with ONE coalesced 1-KiB load straight into registers (no LDS for weights: a piece is
//    private to its wave) and turns it into four MFMA A fragments with 7 VALU ops per 8 weights — amortised over the
//    8 token tiles of the block, so the conversion that bounds the M = 1 path costs 1/8 MFMA slot here;
//  * the activations of a block (128 tokens x 128 k, bf16) go through LDS, double buffered, the 16-B chunks of a row
//    XOR-swizzled by swz(token & 15) — a GF(2)-linear map chosen by exhaustive search so that every ds_read_b128 lane
//    group of a B-fragment read (the hardware serves {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31}, ... together) touches
//    16 different 16-B slots: the obvious (token & 7) was 2-way conflicted and made the kernel LDS-bound;
//  * workgroup = 8 waves, block tile = 128 tokens x 16 row tiles (2 per wave; for the c_fc1 / c_fc2 pair stream the two
//    tiles of a wave are the fc1 / fc2 halves of the same 16 rows, so SwiGLU stays in the epilogue): every B fragment
//    read from LDS feeds two MFMAs, 64 x v_mfma_f32_16x16x32_bf16 per wave and unit (4 tiles per wave measured
//    slower: 184 VGPRs halve the waves per SIMD);
//  * XCD-aware block order: workgroup b runs on XCD b % 8 (each XCD has its own 4 MiB L2).  The (token block, row
//    block) pairs are cut, token-block major, into 8 contiguous ranges, one per XCD: the workgroups an XCD runs side by
//    side share one or two token blocks (1 MiB of activations each), fetched into that L2 once;
//  * operands are staged once per linear by stage_units_kernel (odd rows: stage_rows_kernel): bf16(norm_scale * x) with RMSNorm's 1/rms kept as a
//    per-row factor for the epilogue, and the per-row operand sum that undoes the +128 / zero-point offset:
//        y[m, n] = scale[n] * (acc[m, n] - (128 + zero[n]) * sum_k xb[m, k]) * rinv[m]      (same arithmetic as gemv.hip).
#include <type_traits>

#include <stdlib.h>

#include "common.h"
#include "gemm_fuse.h"
#include "l2_share.h"

// The epilogues' conversions on the hardware paths (with IEEE division + expf in SiLU and the six-instruction software rounding
// the c_fc1 / c_fc2 epilogue was VALU-bound — 33 us of a 269-us launch at T = 2048 against 9 us for its 45 MB of stores,
// profiles/r06_prefill_epilogue_cost.txt): v_cvt_pk_bf16_f32 rounds to nearest even exactly as f32_to_bf16 does (finite inputs),
// v_exp_f32 / v_rcp_f32 are within 1 ulp of f32 — 2^-15 of the bf16 step the result is rounded to.
__device__ __forceinline__ bf16_t bf16_hw(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }
template <int EPI>
__device__ __forceinline__ float pair_act_fast(float a, float b, float limit) {
    if constexpr (EPI == MI355_EPI_CLAMPGLU) {
        const float g = fminf(a, limit), u = fminf(fmaxf(b, -limit), limit);
        return (g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * (-1.702f * 1.44269504088896340736f)))) * (u + 1.0f);
    }
    // silu(a) * b = a / (1 + 2^(-a log2 e)) * b; a -> -inf: 2^(+inf) = inf, rcp = 0; a -> +inf: rcp(1) = 1
    // gelu(a) in the tanh form = a / (1 + 2^(-2 u log2 e)), u = sqrt(2 / pi) (a + 0.044715 a^3)
    const float t = EPI == MI355_EPI_GEGLU ? a * (1.59576912160573071176f + 0.07135481282792783f * (a * a)) : a;
    return (a * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t * -1.44269504088896340736f))) * b;
}

namespace {

constexpr int kBM = 128;     // tokens per block
#ifndef MI355_GEMM_TPW
#define MI355_GEMM_TPW 2
#endif
constexpr int kTPW = MI355_GEMM_TPW;
#ifndef MI355_GEMM_XDMA
#define MI355_GEMM_XDMA 1
#endif
#ifndef MI355_GEMM_BPIPE
#define MI355_GEMM_BPIPE 4   // 128-token blocks: B fragments requested this many LDS reads ahead of the MFMAs that take them (0: hipcc's
                             // order, which waits for every pair of reads right behind their issue); 2 / 3 / 4: -1.4 / -1.9 / -2.0 % per 2048-token
                             // prompt (profiles/r06_prefill_gemm_ab.txt); 124-127 VGPRs at 4, still two workgroups per CU
#endif
#ifndef MI355_GEMM_AND_OR
#define MI355_GEMM_AND_OR 1
#endif
struct GemmParams {
    const uint8_t* w;
    unsigned w_bytes;
    const bf16_t* xb;      // [M, ldxb] staged operands
    int64_t ldxb;
    const float* rinv;     // [M]
    const float* sx;       // [M]
    const void* scales;
    const void* zeros;
    const void* scales2;
    const void* zeros2;
    void* y;
    int64_t ldy;
    int M, N, K, units, n_tiles, n_blocks, per_xcd, total_blocks;
    int sz_dtype, y_dtype;
    // split-K (few blocks: short prompts against N = 4096): slice ks of the units -> part[ks][M][N] f32, summed in order
    // by splitk_reduce_kernel
    int ksplit;
    // Q4, gemm_deep_kernel: a slice's units go through the accumulators in up to `runs` runs of run_units (runs = 1: all its units), whose sums are added up beside
    // them (gemm_runs()).  sx: [M][ksplit][runs] operand sums
    int runs, run_units;
    float* part;
    int relu2;             // STORE: max(y, 0)^2
    float alpha;           // factor of the product where rinv is NULL (an operand that needed no staging)
    float limit;           // CLAMPGLU
    const float* bias;     // STORE: [N], or NULL
    mi355_reduce_norm rn;  // rn.done: the sum of the K-slices also leaves the rows' norm
    bool squares;          // BF16 blocks that may_run_in_squares(): an XCD's blocks are kSquare row blocks by some token blocks (square_blocks())
    bool streamed;         // MI355_LF_STREAMED
    int slice_blocks;      // != 0: row blocks [i slice_blocks, (i + 1) slice_blocks) read the operand at xb + i slice_stride
    int64_t slice_stride;
    // grouped scales (GRP kernels): gtab[group 0..n_groups][r][tab_ld rows] = bf16 scale | bf16 zero << 16 (row n_groups
    // is all zero).  Groups of 2^gq_shift units: sxt[unit][M] = operand sums per unit; of 32 << gq_shift columns (GRP 2): sxt[group][M]
    const uint32_t* gtab;
    const float* sxt;
    int n_groups, gq_shift, tab_ld;
    // producer / consumer fusion (gemm_fuse.h; FUSE kernels only).  f_in: xb is the caller's operand, 1/rms and the operand
    // sums of the block's rows are rebuilt from the partial sums in_ss / in_sx ([partial][M])
    int f_in, in_sx_n, in_ss_n, in_ppu;  // in_ppu: partial operand sums per 128-column unit (a K-slice sums its own units' shares)
    const float* in_sx;
    const float* in_ss;
    float eps;
    bf16_t* out_xb;       // ACCUM: bf16(next_norm * y_new)
    int64_t out_ld;
    const void* next_norm;
    int next_norm_dtype;
    float* out_ss;        // [n_blocks][M]
    float* out_sx;
    const float* rope;    // STORE of c_attn: k rotated + K / V cache rows written here
    const int32_t* pos;
    bf16_t* kcache;
    bf16_t* vcache;
    int S, C, rope_gathered;
    float q_scale;        // != 0: q leaves rotated, scaled by q_scale and rounded to bf16 (gemm_fuse.h: q_scale), rows of 2 * ldy bf16
};

// c_attn's q rows as the prompt attention multiplies them (flash_prefill.hip's own prologue, moved to the producer: the same f32
// arithmetic and the one rounding, so the same bits): four outputs = two interleaved pairs at row m, column n < C
__device__ __forceinline__ void store_q_ready(const GemmParams& p, int m, int n, const f32x4& cs, float o0, float o1, float o2, float o3) {
    const float qs = p.q_scale;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf2;
    const bf2 a = {(__bf16)(qs * (o0 * cs[0] - o1 * cs[1])), (__bf16)(qs * (o1 * cs[0] + o0 * cs[1]))};
    const bf2 b = {(__bf16)(qs * (o2 * cs[2] - o3 * cs[3])), (__bf16)(qs * (o3 * cs[2] + o2 * cs[3]))};
    u32x2 pk;
    pk[0] = __builtin_bit_cast(uint32_t, a);
    pk[1] = __builtin_bit_cast(uint32_t, b);
    *(u32x2*)((bf16_t*)p.y + (int64_t)m * (2 * p.ldy) + n) = pk;
}

constexpr size_t kSplitBudget = (size_t)32 << 20;  // bytes of split-K partials a workspace holds
constexpr int kMaxSplit = 16;
constexpr int kMaxRuns = 8;
constexpr int kMaxSums = 32;                       // operand sums of a row: K-slices x runs.  Slices are 7 at most where they have several runs (gemm_runs()): below units / run_units + 9
constexpr int kTableProducts = MI355_TABLE_PRODUCTS;
constexpr int kSharesAhead = 8;                   // partial sums that a thread of gemm_deep_kernel requests at a time
constexpr size_t kFuseScratch = (size_t)8 << 20;  // partial sums of the fused prompt chain: <= 2048 tokens x ~500 shares x 4 B
// first unit of K-slice s of `ksplit` (slice s = units [lo(s), lo(s + 1)))
__host__ __device__ __forceinline__ int slice_lo(int s, int units, int ksplit) { return (int)((unsigned)(s * units) / (unsigned)ksplit); }  // (s <= 16: 32 bits do)
// first unit of run i = slice * runs + run of a row cut into `ksplit` slices of `runs` runs (run i = units [run_lo(i), run_lo(i + 1)), possibly none)
__device__ __forceinline__ int run_lo(int i, int units, int ksplit, int runs, int run_units) {
    if (runs == 1) return slice_lo(i, units, ksplit);
    const unsigned ks = (unsigned)i / (unsigned)runs;
    const int lo = slice_lo(ks, units, ksplit) + (i - (int)ks * runs) * run_units, hi = slice_lo(ks + 1, units, ksplit);
    return lo < hi ? lo : hi;
}

// 16-B chunk swizzle of an activation row in LDS (see the header): bits 0, 1 of the token stay, bit 2 -> 8, bit 3 -> 12
#ifdef MI355_NO_SWZ
__device__ __forceinline__ int swz(int tok) { return tok & 7; }
#else
__device__ __forceinline__ int swz(int tok) { return (tok & 3) ^ (((tok >> 2) & 1) << 3) ^ (((tok >> 3) & 1) * 12); }
#endif

__device__ __forceinline__ float ldsz(const void* p, int i, int dtype) {
    return dtype == MI355_F32 ? ((const float*)p)[i] : bf16_to_f32(((const bf16_t*)p)[i]);
}

// four entries from i on (each at its own element: a table may start anywhere)
__device__ __forceinline__ f32x4 ldsz4(const void* p, int i, int dtype) {
    if (dtype == MI355_F32) return f32x4{((const float*)p)[i], ((const float*)p)[i + 1], ((const float*)p)[i + 2], ((const float*)p)[i + 3]};
    const bf16_t* b = (const bf16_t*)p + i;
    return f32x4{bf16_to_f32(b[0]), bf16_to_f32(b[1]), bf16_to_f32(b[2]), bf16_to_f32(b[3])};
}

// one row per workgroup: xb = bf16(norm_scale * x), rinv = alpha rsqrt(mean(x^2) + eps) (alpha without norm), sx[m][i] = sum of xb over
// run i (ksplit = runs = 1: the whole row).  Rows of any length at any address; whole aligned ones: stage_units_kernel
__global__ __launch_bounds__(256) void stage_rows_kernel(const void* x, int x_dtype, int64_t ldx, const void* norm_scale,
                                                         int norm_dtype, float eps, int K, int Kp, bf16_t* xb, int64_t ldxb,
                                                         float* rinv, float* sx, int ksplit, int runs, int run_units, float alpha, float norm_add) {
    __shared__ float red[32];
    const int m = blockIdx.x;
    const int units = Kp >> 7;
    float ss = 0.f;
    for (int s = 0; s < ksplit * runs; ++s) {
        const int k_lo = run_lo(s, units, ksplit, runs, run_units) << 7, k_hi = run_lo(s + 1, units, ksplit, runs, run_units) << 7;
        float sum = 0.f;
        for (int k = k_lo + threadIdx.x; k < k_hi; k += blockDim.x) {
            bf16_t o = 0;
            if (k < K) {
                float v = ld_as_f32(x, (int64_t)m * ldx + k, x_dtype);
                if (norm_scale != nullptr) {
                    ss += v * v;
                    v *= norm_add + ld_as_f32(norm_scale, k, norm_dtype);
                }
                o = bf16_hw(v);
                sum += bf16_to_f32(o);
            }
            xb[(int64_t)m * ldxb + k] = o;
        }
        const float tot = block_sum(sum, red);
        if (threadIdx.x == 0) sx[(int64_t)m * (ksplit * runs) + s] = tot;
    }
    const float tss = block_sum(ss, red);
    if (threadIdx.x == 0) rinv[m] = norm_scale != nullptr ? rsqrtf(tss / (float)K + eps) * alpha : alpha;
}

// As stage_rows_kernel for rows of whole 128-column units, four columns per lane and four loads ahead: 12 rows of 4096 f32 columns 13 -> 5 us (a load, a
// multiplication and a store at a time, and a sum of the block per K-slice).  Grouped scales: sxt[i][m] = sum of xb over columns [i * cols, (i + 1) * cols),
// cols = 32, 64 or 128, in place of the sums per slice; the workgroups behind the M rows then lay out the tables, [N][n_groups] bf16 scales / zeros ->
// gtab[grp][r][n] dwords (n fastest: the four rows a lane holds are one 16-B load; row n_groups and the rows past N are zero), a 64 x 64 piece each through
// LDS: 1000 x 4096 f32 rows 17 us, and the tables of 12288 rows 5 in a launch of their own -> 9 together by themselves, 14.7 within a prompt, whose rows the product
// before has just written (profiles/prompt_and_batch_kernels.txt).
constexpr int kStageLds = 64 * 65;  // dwords: a piece of the tables, or a sum per unit
struct GroupTables {
    const bf16_t *s0, *z0, *s1, *z1;
    int N, tab_ld, n_groups, R;
    uint32_t* out;
    __host__ __device__ int row_pieces() const { return (tab_ld + 63) / 64; }
    __host__ __device__ int pieces() const { return R * row_pieces() * ((n_groups + 64) / 64); }
};
__device__ __forceinline__ void group_table_piece(const GroupTables& t, int piece, uint32_t* lds) {  // lds: 64 x 65
    const int rp = t.row_pieces(), r = piece % t.R, n0 = piece / t.R % rp * 64, g0 = piece / t.R / rp * 64;
    const bf16_t* s = r == 1 ? t.s1 : t.s0;
    const bf16_t* z = r == 1 ? t.z1 : t.z0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = i * 4 + ((int)threadIdx.x >> 6), col = threadIdx.x & 63;
        const bool in = n0 + row < t.N && g0 + col < t.n_groups;
        const int64_t at = in ? (int64_t)(n0 + row) * t.n_groups + g0 + col : 0;
        const uint32_t v = s[at] | ((uint32_t)z[at] << 16);
        lds[row * 65 + col] = in ? v : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int grp = g0 + i * 4 + ((int)threadIdx.x >> 6), n = n0 + (threadIdx.x & 63);
        if (grp <= t.n_groups && n < t.tab_ld) t.out[((int64_t)grp * t.R + r) * t.tab_ld + n] = lds[(threadIdx.x & 63) * 65 + (grp - g0)];
    }
}
template <bool WIDE>  // rows and norm scale in whole aligned groups of four
__global__ __launch_bounds__(256) void stage_units_kernel(const void* x, int x_dtype, int64_t ldx, const void* norm_scale, int norm_dtype, float eps, int K,
                                                          bf16_t* xb, float* rinv, float* sx, int ksplit, int runs, int run_units, float alpha, float norm_add,
                                                          float* sxt, int M, int cols, const GroupTables tables) {
    __shared__ uint32_t lds[kStageLds];
    if ((int)blockIdx.x >= M) return group_table_piece(tables, blockIdx.x - M, lds);
    const int m = blockIdx.x;
    float* per_unit = (float*)lds + 32;
    auto load4 = [&](const void* src, int64_t at, int dtype) {
        f32x4 v;
        if constexpr (WIDE) {
            if (dtype == MI355_F32) return *(const f32x4*)((const float*)src + at);
            const u32x2 w = *(const u32x2*)((const bf16_t*)src + at);
            return f32x4{__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16), __uint_as_float(w[1] & 0xffff0000u)};
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ld_as_f32(src, at + j, dtype);
        return v;
    };
    constexpr int kAhead = 4;
    float ss = 0.f;
    for (int k0 = threadIdx.x * 4; k0 < K; k0 += 1024 * kAhead) {
        f32x4 v[kAhead], ns[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) v[i] = load4(x, (int64_t)m * ldx + (k0 + i * 1024 < K ? k0 + i * 1024 : k0), x_dtype);
        if (norm_scale != nullptr) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) ns[i] = load4(norm_scale, k0 + i * 1024 < K ? k0 + i * 1024 : k0, norm_dtype);
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int k = k0 + i * 1024;
            if (k >= K) break;  // (whole 128-column units: the 32 lanes of one leave together)
            if (norm_scale != nullptr) {
                ss += (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
                v[i] *= ns[i] + norm_add;
            }
            bf16_t o[4];
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                o[j] = bf16_hw(v[i][j]);
                sum += bf16_to_f32(o[j]);
            }
            *(u32x2*)(xb + (int64_t)m * K + k) = u32x2{o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16)};
            sum = group_sum(sum, cols >> 2);
            if (k % cols == 0) {
                if (sxt != nullptr)
                    sxt[(int64_t)(k / cols) * M + m] = sum;
                else
                    per_unit[k >> 7] = sum;
            }
        }
    }
    const float tss = block_sum(ss, (float*)lds);
    if (threadIdx.x == 0) rinv[m] = norm_scale != nullptr ? rsqrtf(tss / (float)K + eps) * alpha : alpha;
    if (sxt == nullptr) {  // (every wave has passed the block sum's barriers: the units' sums stand in LDS)
        // 16 lanes a sum: beside a large unit four roundings, not one per unit (and a thread's chain of 32 units took 1 us)
        for (int s0 = 0; s0 < ksplit * runs; s0 += 16) {
            const int s = s0 + (threadIdx.x >> 4), i = s < ksplit * runs ? s : 0;
            const int u_lo = run_lo(i, K >> 7, ksplit, runs, run_units), u_hi = run_lo(i + 1, K >> 7, ksplit, runs, run_units);
            float sum = 0.f;
            for (int u = u_lo + (threadIdx.x & 15); u < u_hi; u += 16) sum += per_unit[u];
            sum = group_sum(sum, 16);
            if ((threadIdx.x & 15) == 0 && s < ksplit * runs) sx[(int64_t)m * (ksplit * runs) + s] = sum;
        }
    }
}

// o += the K-slices' four values at row[0 .. 3], `stride` floats apart, in slice order.  All slices are requested before the first one is added: a
// loop over a runtime number of them was one memory round trip per slice, most of the 5-6 us such a launch took.
template <int N>
__device__ __forceinline__ void add_slices_n(const float* row, int64_t stride, int ksplit, f32x4& o) {
    f32x4 v[N];
#pragma unroll
    for (int s = 0; s < N; ++s) v[s] = *(const f32x4*)(row + (s < ksplit ? s : 0) * stride);
#pragma unroll
    for (int s = 0; s < N; ++s)
        if (s < ksplit) o += v[s];
}
__device__ __forceinline__ void add_slices(const float* row, int64_t stride, int ksplit, f32x4& o) {
    if (ksplit <= 2) return add_slices_n<2>(row, stride, ksplit, o);
    if (ksplit <= 4) return add_slices_n<4>(row, stride, ksplit, o);
    if (ksplit <= 8) return add_slices_n<8>(row, stride, ksplit, o);
    add_slices_n<kMaxSplit>(row, stride, ksplit, o);
}

// y[m][n] (+)= sum over the K-slices, in slice order (deterministic)
template <int EPI>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* part, int ksplit, int M, int N, void* y, int y_dtype,
                                                            int64_t ldy, int relu2, float limit, const float* bias) {
    const int64_t n4 = N >> 2;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (int64_t)M * n4; i += (int64_t)gridDim.x * blockDim.x) {
        const int m = (int)(i / n4), n = (int)(i - (int64_t)m * n4) * 4;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        if constexpr (is_pair_epi(EPI)) {
            f32x4 b = {0.f, 0.f, 0.f, 0.f};
            const float* row = part + (int64_t)m * (2 * (int64_t)N) + n;
            add_slices(row, (int64_t)M * 2 * N, ksplit, o);
            add_slices(row + N, (int64_t)M * 2 * N, ksplit, b);
            bf16_t* dst = (bf16_t*)y + (int64_t)m * ldy + n;
            u32x2 pk;
            pk[0] = (uint32_t)bf16_hw(pair_act_fast<EPI>(o[0], b[0], limit)) | ((uint32_t)bf16_hw(pair_act_fast<EPI>(o[1], b[1], limit)) << 16);
            pk[1] = (uint32_t)bf16_hw(pair_act_fast<EPI>(o[2], b[2], limit)) | ((uint32_t)bf16_hw(pair_act_fast<EPI>(o[3], b[3], limit)) << 16);
            *(u32x2*)dst = pk;
        } else if (y_dtype == MI355_F32) {
            float* dst = (float*)y + (int64_t)m * ldy + n;
            if constexpr (EPI == MI355_EPI_ACCUM) o = *(const f32x4*)dst;
            add_slices(part + (int64_t)m * N + n, (int64_t)M * N, ksplit, o);
            if (EPI == MI355_EPI_STORE && bias != nullptr) o += *(const f32x4*)(bias + n);
            if (EPI == MI355_EPI_STORE && relu2) o = f32x4{relu2_f32(o[0]), relu2_f32(o[1]), relu2_f32(o[2]), relu2_f32(o[3])};
            *(f32x4*)dst = o;
        } else {
            bf16_t* dst = (bf16_t*)y + (int64_t)m * ldy + n;
            if constexpr (EPI == MI355_EPI_ACCUM) {
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = bf16_to_f32(dst[r]);
            }
            add_slices(part + (int64_t)m * N + n, (int64_t)M * N, ksplit, o);
            if (EPI == MI355_EPI_STORE && bias != nullptr) o += *(const f32x4*)(bias + n);
            if (EPI == MI355_EPI_STORE && relu2) o = f32x4{relu2_f32(o[0]), relu2_f32(o[1]), relu2_f32(o[2]), relu2_f32(o[3])};
            u32x2 pk;
            pk[0] = (uint32_t)bf16_hw(o[0]) | ((uint32_t)bf16_hw(o[1]) << 16);
            pk[1] = (uint32_t)bf16_hw(o[2]) | ((uint32_t)bf16_hw(o[3]) << 16);
            *(u32x2*)dst = pk;
        }
    }
}

// A residual product's K-slices added to its rows (as splitk_reduce_kernel does), and the rows' RMSNorm, the operand of the next product: one row per
// workgroup, all slices of its columns requested at once.  16 rows of 4096: 4.6 us and 4.6 for the norm -> 5.8.
constexpr int kNormHeld = 2;  // column vectors of a thread: rows of up to 8192
__global__ __launch_bounds__(1024) void splitk_norm_kernel(const float* part, int ksplit, int M, int N, float* y, int64_t ldy, const mi355_reduce_norm rn) {
    __shared__ float red[32];
    const int m = blockIdx.x;
    f32x4 v[kNormHeld], sc[kNormHeld];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < kNormHeld; ++i) {
        const int n = (threadIdx.x + i * 1024) * 4;
        if (n < N) {
            float* dst = y + (int64_t)m * ldy + n;
            v[i] = *(const f32x4*)dst;
            sc[i] = ldsz4(rn.scale, n, rn.scale_dtype);
            add_slices(part + (int64_t)m * N + n, (int64_t)M * N, ksplit, v[i]);
            *(f32x4*)dst = v[i];
            ss += (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
        }
    }
    const float rinv = 1.0f / sqrtf(block_sum(ss, red) / (float)N + rn.eps);
#pragma unroll
    for (int i = 0; i < kNormHeld; ++i) {
        const int n = (threadIdx.x + i * 1024) * 4;
        if (n < N) {
            bf16_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = bf16_hw(v[i][j] * rinv * (sc[i][j] + rn.add));
            *(u32x2*)(rn.xb + (int64_t)m * N + n) = u32x2{o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16)};
        }
    }
}

// The split-K reduction of a launch of the fused chain (gemm_fuse.h): sums the K-slices in slice order as splitk_reduce_kernel
// does, and is the producer epilogue the whole-K kernel has — the residual rows also leave as the next linear's bf16 operand
// with their partial sums, the SwiGLU output with its partial operand sums, c_attn's k rotated and K / V written to the cache.
// One half wave (32 lanes x 4 columns) per (row, 128-column unit): a unit is what a consumer's K-slices are cut at.
template <int EPI>
__global__ __launch_bounds__(256) void splitk_fused_reduce_kernel(const GemmParams p) {
    const int units_n = p.N >> 7;  // N % 128 == 0 (host check)
    const int64_t groups = (int64_t)p.M * units_n;
    const int l32 = threadIdx.x & 31;
    for (int64_t grp = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 5; grp < groups; grp += (int64_t)gridDim.x * 8) {
        const int m = (int)(grp / units_n), un = (int)(grp - (int64_t)m * units_n);
        const int n = un * 128 + l32 * 4;
        if constexpr (is_pair_epi(EPI)) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
            const float* row = p.part + (int64_t)m * (2 * (int64_t)p.N) + n;
            add_slices(row, (int64_t)p.M * 2 * p.N, p.ksplit, a);
            add_slices(row + p.N, (int64_t)p.M * 2 * p.N, p.ksplit, b);
            bf16_t ob[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) ob[r] = bf16_hw(pair_act_fast<EPI>(a[r], b[r], p.limit));
            u32x2 pk;
            pk[0] = (uint32_t)ob[0] | ((uint32_t)ob[1] << 16);
            pk[1] = (uint32_t)ob[2] | ((uint32_t)ob[3] << 16);
            *(u32x2*)((bf16_t*)p.y + (int64_t)m * p.ldy + n) = pk;
            if (p.out_sx != nullptr) {
                const float s1 = group_sum((bf16_to_f32(ob[0]) + bf16_to_f32(ob[1])) + (bf16_to_f32(ob[2]) + bf16_to_f32(ob[3])), 32);
                if (l32 == 0) p.out_sx[(int64_t)un * p.M + m] = s1;
            }
        } else {
            float* dst = (float*)p.y + (int64_t)m * p.ldy + n;  // (f32 outputs only: host check)
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
            if constexpr (EPI == MI355_EPI_ACCUM) o = *(const f32x4*)dst;
            [[maybe_unused]] f32x4 ns = {0.f, 0.f, 0.f, 0.f}, cs = {0.f, 0.f, 0.f, 0.f};
            [[maybe_unused]] int posm = 0;
            if constexpr (EPI == MI355_EPI_ACCUM) {
                if (p.out_xb != nullptr) ns = ldsz4(p.next_norm, n, p.next_norm_dtype);
            } else if (p.rope != nullptr) {
                posm = p.pos[m];
                cs = *(const f32x4*)(p.rope + (int64_t)(p.rope_gathered ? m : posm) * 128 + (n & 127));
            }
            add_slices(p.part + (int64_t)m * p.N + n, (int64_t)p.M * p.N, p.ksplit, o);
            if constexpr (EPI == MI355_EPI_STORE) {
                const int sec = p.rope != nullptr ? (n >= p.C) + (n >= 2 * p.C) : 0;
                if (sec != 0) {  // as the whole-K epilogue: k rotated in f32, K / V rows to the bf16 cache
                    const int cn = n - sec * p.C, h = cn >> 7, d = cn & 127;
                    if (sec == 1) {
                        const float k0 = o[0] * cs[0] - o[1] * cs[1], k1 = o[1] * cs[0] + o[0] * cs[1];
                        const float k2 = o[2] * cs[2] - o[3] * cs[3], k3 = o[3] * cs[2] + o[2] * cs[3];
                        o = f32x4{k0, k1, k2, k3};
                    }
                    const int slot = posm < p.S - 1 ? posm : p.S - 1;
                    u32x2 pk;
                    pk[0] = (uint32_t)bf16_hw(o[0]) | ((uint32_t)bf16_hw(o[1]) << 16);
                    pk[1] = (uint32_t)bf16_hw(o[2]) | ((uint32_t)bf16_hw(o[3]) << 16);
                    *(u32x2*)((sec == 1 ? p.kcache : p.vcache) + ((int64_t)h * p.S + slot) * 128 + d) = pk;
                    continue;
                }
                if (p.rope != nullptr && p.q_scale != 0.f) {
                    store_q_ready(p, m, n, cs, o[0], o[1], o[2], o[3]);
                    continue;
                }
            }
            *(f32x4*)dst = o;
            if constexpr (EPI == MI355_EPI_ACCUM) {
                if (p.out_xb != nullptr) {
                    bf16_t ob[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) ob[r] = bf16_hw(o[r] * ns[r]);
                    u32x2 pk;
                    pk[0] = (uint32_t)ob[0] | ((uint32_t)ob[1] << 16);
                    pk[1] = (uint32_t)ob[2] | ((uint32_t)ob[3] << 16);
                    *(u32x2*)(p.out_xb + (int64_t)m * p.out_ld + n) = pk;
                    const float s1 = group_sum((bf16_to_f32(ob[0]) + bf16_to_f32(ob[1])) + (bf16_to_f32(ob[2]) + bf16_to_f32(ob[3])), 32);
                    const float s2 = group_sum((o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]), 32);
                    if (l32 == 0) {
                        p.out_sx[(int64_t)un * p.M + m] = s1;
                        p.out_ss[(int64_t)un * p.M + m] = s2;
                    }
                }
            }
        }
    }
}

// LDS of gemm_q4_kernel behind the two activation buffers: the tokens' factors (2 x BM floats), FUSE: the shares they are summed from (4 KiB), the
// tokens' positions, the rows' tables
template <int BM, int NB = 2>
constexpr int kPosAt = NB * BM * 256 + 2 * BM * 4 + 4096;
template <int BM, bool FUSE, int NB = 2>
constexpr int kRowAt = NB * BM * 256 + 2 * BM * 4 + (FUSE ? 4096 + BM * 4 : 0);

// The end of a block: lane (g, c) of a wave holds rows 4 g .. 4 g + 3 of the wave's tiles for token tt * 16 + c (acc: what the MFMAs summed, GRP: the scaled
// sums).  The tables `fr` (1/rms, operand sums of the tokens), `postab` and `rowtab` (scale, 128 + zero, next norm) stand in LDS; every wave has passed
// its last read of the activation buffers and no request into them is under way.
template <int EPI, bool PAIR, int FMT, int kWaves, int BM, int GRP, bool FUSE, int TPW>
__device__ __forceinline__ void gemm_epilogue(const GemmParams& p, f32x4 (&acc)[TPW][BM / 16], char* smem, const float* fr, const int* postab,
                                              const float* rowtab, const int (&tile)[TPW], int m0, int nb, int ks, int wave, int lane) {
    constexpr int kTT = BM / 16, kSlots = kWaves * TPW, kThreads = 64 * kWaves;
    const int g = lane >> 4, c = lane & 15;
    // old residual rows and rotations are requested for kEB token tiles at a time, without a branch between them (columns and tokens past the end read
    // entry 0): a load behind a branch of its own is waited for alone.  Four at a time: a bf16 prompt of 777 tokens (7B, 8 layers) 3.37 -> 3.25 ms on one box; int4 blocks of 128 tokens,
    // two to a CU, cover it themselves (2048 tokens: 1.8 % slower with four)
    constexpr int kEB = BM >= 128 && FMT == MI355_W_Q4 ? 1 : kTT < 4 ? kTT : 4;
    const bool emit = FUSE && EPI == MI355_EPI_ACCUM && p.out_xb != nullptr;
    const bool sums = FUSE && EPI != MI355_EPI_STORE && p.out_sx != nullptr;
    auto rows4 = [&](int table, int t) { return *(const f32x4*)(rowtab + (table * kSlots + TPW * wave + t) * 16 + 4 * g); };
    int nn[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) nn[t] = tile[t] * 16 + 4 * g;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        [[maybe_unused]] f32x4 sc, zp;
        if constexpr (FMT == MI355_W_Q4 && GRP == 0) sc = rows4(0, t), zp = rows4(1, t);
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) {
            const float ri = fr[tt * 16 + c];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (GRP != 0 || FMT == MI355_W_BF16)
                    acc[t][tt][r] *= ri;
                else
                    acc[t][tt][r] = sc[r] * (acc[t][tt][r] - zp[r] * fr[BM + tt * 16 + c]) * ri;
            }
        }
    }
    if (p.ksplit > 1) {  // partial sums of this K-slice; the SwiGLU pair keeps c_fc1 at column n, c_fc2 at N + n
        const int64_t ldp = PAIR ? 2 * (int64_t)p.N : (int64_t)p.N;
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) {
            const int m = m0 + tt * 16 + c;
#pragma unroll
            for (int t = 0; t < TPW; ++t)
                if (m < p.M && nn[t] < p.N) *(f32x4*)(p.part + ((int64_t)ks * p.M + m) * ldp + (PAIR && (t & 1) ? p.N : 0) + nn[t]) = acc[t][tt];
        }
        return;
    }
    [[maybe_unused]] float es1[kTT], es2[kTT];  // FUSE: this lane's share of the rows' partial sums (operand values, squares)
#pragma unroll
    for (int tb = 0; tb < kTT; tb += kEB) {
        [[maybe_unused]] f32x4 got[kEB][TPW];  // ACCUM: the old rows; STORE of c_attn: rotations
        if constexpr (EPI == MI355_EPI_ACCUM) {
            if (p.y_dtype == MI355_F32) {
#pragma unroll
                for (int i = 0; i < kEB && tb + i < kTT; ++i)
#pragma unroll
                    for (int t = 0; t < TPW; ++t) {
                        const int m = m0 + (tb + i) * 16 + c;
                        got[i][t] = *(const f32x4*)((const float*)p.y + (m < p.M && nn[t] < p.N ? (int64_t)m * p.ldy + nn[t] : 0));
                    }
            } else {
#pragma unroll
                for (int i = 0; i < kEB && tb + i < kTT; ++i)
#pragma unroll
                    for (int t = 0; t < TPW; ++t) {
                        const int m = m0 + (tb + i) * 16 + c;
                        const u32x2 w = *(const u32x2*)((const bf16_t*)p.y + (m < p.M && nn[t] < p.N ? (int64_t)m * p.ldy + nn[t] : 0));
                        got[i][t] = f32x4{__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16),
                                          __uint_as_float(w[1] & 0xffff0000u)};
                    }
            }
        }
        if constexpr (FUSE && EPI == MI355_EPI_STORE) {
            if (p.rope != nullptr) {
#pragma unroll
                for (int i = 0; i < kEB && tb + i < kTT; ++i) {
                    const int t16 = (tb + i) * 16 + c;
                    const int m = m0 + t16 < p.M ? m0 + t16 : p.M - 1;
#pragma unroll
                    for (int t = 0; t < TPW; ++t)
                        got[i][t] = *(const f32x4*)(p.rope + (int64_t)(p.rope_gathered ? m : postab[t16]) * 128 + (nn[t] & 127));
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kEB && tb + i < kTT; ++i) {
            const int tt = tb + i, m = m0 + tt * 16 + c;
            if constexpr (FUSE) es1[tt] = es2[tt] = 0.f;
            if (m >= p.M) continue;
            if constexpr (is_pair_epi(EPI)) {
#pragma unroll
                for (int t = 0; t < TPW; t += 2) {
                    if (nn[t] >= p.N) continue;  // N % 4 == 0 (host check)
                    bf16_t ob[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) ob[r] = bf16_hw(pair_act_fast<EPI>(acc[t][tt][r], acc[t + 1][tt][r], p.limit));
                    u32x2 o;
                    o[0] = (uint32_t)ob[0] | ((uint32_t)ob[1] << 16);
                    o[1] = (uint32_t)ob[2] | ((uint32_t)ob[3] << 16);
                    *(u32x2*)((bf16_t*)p.y + (int64_t)m * p.ldy + nn[t]) = o;
                    if constexpr (FUSE) es1[tt] += (bf16_to_f32(ob[0]) + bf16_to_f32(ob[1])) + (bf16_to_f32(ob[2]) + bf16_to_f32(ob[3]));
                }
            } else {
#pragma unroll
                for (int t = 0; t < TPW; ++t) {
                    const int n = nn[t];
                    if (n >= p.N) continue;
                    f32x4 o = acc[t][tt];
                    if constexpr (FUSE && EPI == MI355_EPI_STORE) {
                        // c_attn (model.py:197-221): rows [C, 2C) are k — rotated in f32 (model.py:306-323; the lane's four rows
                        // are two interleaved pairs) — rows [2C, 3C) are v; both go to their bf16 cache rows, q goes to y
                        const int sec = p.rope != nullptr ? (n >= p.C) + (n >= 2 * p.C) : 0;
                        if (sec != 0) {
                            const int cn = n - sec * p.C, h = cn >> 7, d = cn & 127;
                            if (sec == 1) {
                                const f32x4 cs = got[i][t];
                                const float k0 = o[0] * cs[0] - o[1] * cs[1], k1 = o[1] * cs[0] + o[0] * cs[1];
                                const float k2 = o[2] * cs[2] - o[3] * cs[3], k3 = o[3] * cs[2] + o[2] * cs[3];
                                o = f32x4{k0, k1, k2, k3};
                            }
                            const int posm = postab[tt * 16 + c];
                            const int slot = posm < p.S - 1 ? posm : p.S - 1;
                            bf16_t* dst = (sec == 1 ? p.kcache : p.vcache) + ((int64_t)h * p.S + slot) * 128 + d;
                            u32x2 pk;
                            pk[0] = (uint32_t)bf16_hw(o[0]) | ((uint32_t)bf16_hw(o[1]) << 16);
                            pk[1] = (uint32_t)bf16_hw(o[2]) | ((uint32_t)bf16_hw(o[3]) << 16);
                            *(u32x2*)dst = pk;
                            continue;
                        }
                        if (p.rope != nullptr && p.q_scale != 0.f) {
                            store_q_ready(p, m, n, got[i][t], o[0], o[1], o[2], o[3]);
                            continue;
                        }
                    }
                    if constexpr (!FUSE && EPI == MI355_EPI_STORE && FMT == MI355_W_BF16) {
                        if (p.bias != nullptr) o += *(const f32x4*)(p.bias + n);
                    }
                    if constexpr (EPI == MI355_EPI_ACCUM) o += got[i][t];
                    if (!FUSE && EPI == MI355_EPI_STORE && p.relu2) o = f32x4{relu2_f32(o[0]), relu2_f32(o[1]), relu2_f32(o[2]), relu2_f32(o[3])};
                    if (p.y_dtype == MI355_F32) {
                        *(f32x4*)((float*)p.y + (int64_t)m * p.ldy + n) = o;
                        if constexpr (FUSE && EPI == MI355_EPI_ACCUM) {
                            if (emit) {  // the next linear's operand: bf16(norm scale * x), as stage_rows_kernel rounds it
                                const f32x4 ns = rows4(2, t);
                                bf16_t ob[4];
#pragma unroll
                                for (int r = 0; r < 4; ++r) ob[r] = bf16_hw(o[r] * ns[r]);
                                u32x2 pk;
                                pk[0] = (uint32_t)ob[0] | ((uint32_t)ob[1] << 16);
                                pk[1] = (uint32_t)ob[2] | ((uint32_t)ob[3] << 16);
                                *(u32x2*)(p.out_xb + (int64_t)m * p.out_ld + n) = pk;
                                es1[tt] += (bf16_to_f32(ob[0]) + bf16_to_f32(ob[1])) + (bf16_to_f32(ob[2]) + bf16_to_f32(ob[3]));
                                es2[tt] += (o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]);
                            }
                        }
                    } else {
                        u32x2 pk;
                        pk[0] = (uint32_t)bf16_hw(o[0]) | ((uint32_t)bf16_hw(o[1]) << 16);
                        pk[1] = (uint32_t)bf16_hw(o[2]) | ((uint32_t)bf16_hw(o[3]) << 16);
                        *(u32x2*)((bf16_t*)p.y + (int64_t)m * p.ldy + n) = pk;
                    }
                }
            }
        }
    }
    if constexpr (FUSE && EPI != MI355_EPI_STORE) {
        // partial sums of the block's rows per token: lane groups (permlane swaps), then the waves through LDS in wave
        // order (the activation buffers are free: every wave is past its last unit's barrier), one entry per row block
        if (sums) {
            // (a block of 256 rows — 8 waves, no pair — writes one share per 128 rows: the granularity a K-split consumer's
            // slices are cut at; smaller blocks are shares of their own)
            constexpr int kHalves = (!PAIR && kSlots == 16) ? 2 : 1;
            float* red = (float*)smem;  // [kWaves][2][BM]
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) {
                float a = es1[tt], b = es2[tt];
                a += lane_xor16(a);
                a += lane_xor32(a);
                b += lane_xor16(b);
                b += lane_xor32(b);
                if (g == 0) {
                    red[(wave * 2 + 0) * BM + tt * 16 + c] = a;
                    red[(wave * 2 + 1) * BM + tt * 16 + c] = b;
                }
            }
            __syncthreads();
            for (int idx = threadIdx.x; idx < kHalves * BM; idx += kThreads) {
                const int t = idx % BM, half = idx / BM;
                const int m = m0 + t;
                const int share = nb * kHalves + half;
                if (m < p.M && share * (kHalves == 2 ? 128 : (PAIR ? kSlots / 2 : kSlots) * 16) < p.N) {
                    float a = 0.f, b = 0.f;
#pragma unroll
                    for (int w = 0; w < kWaves / kHalves; ++w) {
                        a += red[((half * (kWaves / kHalves) + w) * 2 + 0) * BM + t];
                        b += red[((half * (kWaves / kHalves) + w) * 2 + 1) * BM + t];
                    }
                    p.out_sx[(int64_t)share * p.M + m] = a;
                    if (p.out_ss != nullptr) p.out_ss[(int64_t)share * p.M + m] = b;
                }
            }
        }
    }
}

// The int4 stream, one 1-KiB piece per (tile, unit).
// GRP: 0 one (scale, zero) pair per output row; 2: one pair per row and group of 32 or 64 input columns (GPTQ "groupsize",
// lit_llama/quantization.py:284-333 with tile_cols > 0; groups of whole units: gemm_deep_kernel).  The MFMA accumulators keep running over K (cum_g =
// columns up to the end of group g) and at every group
// end     accf += (s_g - s_{g+1}) cum_g - s_g (128 + z_g) X_g      (Abel summation of sum_g s_g (A_g - (128 + z_g) X_g),
// s past the last group = 0; X_g = the group's operand sum from stage_units_kernel): two FMAs per output element
// and group, no accumulator reset.  The k columns of ONE MFMA are spread over the unit (lane group g holds columns
// 32 g + 8 d ..), so a unit takes one pass per group with the other lane groups' activations zeroed, as in gemv.hip.
// FUSE: the producer / consumer fusion of gemm_fuse.h (ungrouped launches without a K split): operand sums and 1/rms from
// partial sums instead of the staging pass; the residual epilogue emits the next linear's bf16 operand and its partial
// sums, the SwiGLU epilogue the partial operand sums of its output, the c_attn epilogue rotates k and writes the K / V cache
template <int EPI, bool PAIR, int kWaves, int BM, int GRP = 0, bool FUSE = false>
__global__ __launch_bounds__(64 * kWaves) void gemm_q4_kernel(const GemmParams p) {
    static_assert(!FUSE || GRP == 0, "the fused chain runs over per-row scales");
    constexpr int kTT = BM / 16;                   // 16-token tiles per block
    constexpr int kSlots = kWaves * kTPW;          // tile slots per block
    constexpr int kThreads = 64 * kWaves;
    constexpr int kXChunks = BM * 16 / kThreads;   // 16-B activation chunks per thread and unit
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c = lane & 15;
    // b -> (token block, row block): the (token block, row block) pairs, token block major, are cut into 8 contiguous
    // ranges, one per XCD (b % 8): the workgroups an XCD runs side by side share one or two token blocks
    const int n_blocks = p.n_blocks;
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    const int L2 = xcd * p.per_xcd + j;
    if (j >= p.per_xcd || L2 >= p.total_blocks * p.ksplit) return;
    const int L = L2 / p.ksplit, ks = L2 - L * p.ksplit;  // (ksplit = 1: ks = 0, all units)
    const int mb = L / n_blocks, nb = L - mb * n_blocks;
    const int m0 = mb * BM;
    float* fr = (float*)(smem + 2 * BM * 256);  // [BM] 1/rms, [BM] operand sums of the block's tokens
    [[maybe_unused]] int* postab = (int*)(smem + kPosAt<BM>);            // FUSE, STORE: [BM] positions
    [[maybe_unused]] float* rowtab = (float*)(smem + kRowAt<BM, FUSE>);  // [scale, 128 + zero, next norm's scale][rows of the block]
    const int u_lo = slice_lo(ks, p.units, p.ksplit), u_hi = slice_lo(ks + 1, p.units, p.ksplit);  // K-slice

    // this wave's row tiles
    int tile[kTPW], rr[kTPW];
#pragma unroll
    for (int t = 0; t < kTPW; ++t) {
        if (PAIR) {
            tile[t] = nb * (kSlots / 2) + (kTPW / 2) * wave + (t >> 1);  // pair tile: 16 rows of c_fc1 (r = 0) and c_fc2 (r = 1)
            rr[t] = t & 1;
        } else {
            tile[t] = nb * kSlots + kTPW * wave + t;
            rr[t] = 0;
        }
    }
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, (int)p.w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw0 = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, 0, 0x00020000);
    const unsigned xbytes = (unsigned)((int64_t)p.M * p.ldxb * 2);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)p.xb, 0, (int)xbytes, 0x00020000);
    const unsigned lane_off = lane * 16;
    auto wload = [&](int t, int u) {
        // past the last unit / tile the load goes through a zero-sized descriptor: the scalar offset operand of a raw
        // buffer load is NOT range-checked (an unconditional prefetch of unit `units` of the last tile faulted)
        const bool ok = tile[t] < p.n_tiles && u < u_hi;
        const unsigned off = (unsigned)((tile[t] * p.units + u) * (PAIR ? 2 : 1) + rr[t]) * 1024u;
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ok ? rw : rw0, lane_off, ok ? off : 0u, 0));
    };
    // activation block of unit u: 2048 chunks of 16 B, kXChunks per thread; chunk = (token, 16-B column)
    // The activation block of the NEXT unit goes global -> LDS by LDS-DMA (buffer_load ... lds, 16 B per lane: one instruction
    // fills 1 KiB = four token rows of the buffer; the XOR swizzle is applied on the SOURCE side — LDS slot c of token t takes column
    // c ^ swz(t)), requested at the unit's start.  The staged version held the block in 32 registers per thread, which hipcc could only
    // afford by sinking the requests to the unit's END, right in front of the LDS stores that wait for them: every unit paid the memory
    // latency in front of its barrier (rocprofv3 --pmc: SQ_WAIT_ANY 0.53 of the wave cycles, 0.28 issue stalls, 0.19 active;
    // profiles/r06_prefill_gemm_ab.txt).
    constexpr bool kXDma = MI355_GEMM_XDMA != 0 && GRP == 0;
    [[maybe_unused]] auto xdma = [&](int u, int buf) {
#pragma unroll
        for (int i = 0; i < kXChunks; ++i) {
            const int ch = i * kThreads + threadIdx.x;   // = LDS chunk: consecutive lanes, consecutive 16 B
            const int tok = ch >> 4, slot = ch & 15;
            const unsigned off = (unsigned)(((int64_t)(m0 + tok) * p.ldxb) * 2) + (unsigned)u * 256u + (unsigned)((slot ^ swz(tok)) * 16);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(smem + buf * (BM * 256) + (i * kThreads + wave * 64) * 16),
                                                     16, (m0 + tok) < p.M ? off : 0xFFFFFFF0u, 0, 0, 0);
        }
    };
    u32x4 stage[kXDma ? 1 : kXChunks];
    auto xload = [&](int u) {
        if constexpr (kXDma) return;
#pragma unroll
        for (int i = 0; i < kXChunks; ++i) {
            const int ch = i * kThreads + threadIdx.x;
            const int tok = ch >> 4, col = ch & 15;
            const unsigned off = (unsigned)(((int64_t)(m0 + tok) * p.ldxb) * 2) + (unsigned)u * 256u + (unsigned)col * 16u;
            stage[i] = __builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, (m0 + tok) < p.M ? off : 0xFFFFFFF0u, 0, 0));
        }
    };
    auto xstore = [&](int buf) {
        if constexpr (kXDma) return;
#pragma unroll
        for (int i = 0; i < kXChunks; ++i) {
            const int ch = i * kThreads + threadIdx.x;
            const int tok = ch >> 4, col = ch & 15;
            *(u32x4*)(smem + buf * (BM * 256) + tok * 256 + ((col ^ swz(tok)) << 4)) = stage[i];
        }
    };

    f32x4 acc[kTPW][kTT];
#pragma unroll
    for (int t = 0; t < kTPW; ++t)
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) acc[t][tt] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 wcur[kTPW], wnext[kTPW];
#pragma unroll
    for (int t = 0; t < kTPW; ++t) wcur[t] = wload(t, u_lo);
    if constexpr (kXDma) xdma(u_lo, u_lo & 1);
    xload(u_lo);
    if constexpr (FUSE) {
        if (p.f_in) {
            // (behind the first unit's operand requests, in front of its barrier)
            // partial sums -> per-row factors.  Every thread takes a row and every kP-th partial, eight loads in flight
            // (a plain loop over the partials is one memory round trip per partial: 13-15 us per launch, measured), the
            // kP shares are added in share order through LDS: a fixed order, deterministic
            constexpr int kP = kThreads >= BM ? kThreads / BM : 1;
            float* frp = fr + 2 * BM;  // [kP][2][BM]
            for (int idx = threadIdx.x; idx < kP * BM; idx += kThreads) {
                const int t = idx % BM, part = idx / BM;
                const int64_t m = m0 + t < p.M ? m0 + t : p.M - 1;
                // (a K-slice of a split launch takes the shares of its own units: the operand sum of ITS columns)
                const int jlo = p.ksplit > 1 ? slice_lo(ks, p.units, p.ksplit) * p.in_ppu : 0;
                const int jhi = p.ksplit > 1 ? slice_lo(ks + 1, p.units, p.ksplit) * p.in_ppu : p.in_sx_n;
                auto add_shares = [&](const float* in, int lo, int hi) {
                    constexpr int kIn = 8;  // in flight
                    float sum = 0.f;
                    for (int j0 = lo + part; j0 < hi; j0 += kIn * kP) {
                        float v[kIn];
#pragma unroll
                        for (int i = 0; i < kIn; ++i) v[i] = in[(j0 + i * kP < hi ? j0 + i * kP : j0) * (int64_t)p.M + m];
#pragma unroll
                        for (int i = 0; i < kIn; ++i) sum += j0 + i * kP < hi ? v[i] : 0.f;
                    }
                    return sum;
                };
                const float sxs = add_shares(p.in_sx, jlo, jhi), sss = add_shares(p.in_ss, 0, p.in_ss_n);
                frp[(part * 2 + 0) * BM + t] = sss;
                frp[(part * 2 + 1) * BM + t] = sxs;
            }
        }
    }
    // what the epilogue needs of the block's rows and tokens, fetched behind the first unit's operands: there each of these loads, behind a branch of
    // its own, was waited for alone (24 memory round trips per launch)
    if constexpr (GRP == 0) {
        for (int i = threadIdx.x; i < kSlots * 16; i += kThreads) {
            const int slot = i >> 4;
            const int n = (PAIR ? nb * (kSlots / 2) + (slot >> 1) : nb * kSlots + slot) * 16 + (i & 15);
            const bool ok = n < p.N, second = PAIR && (slot & 1);
            const void* sp = second ? p.scales2 : p.scales;
            const void* zq = second ? p.zeros2 : p.zeros;
            float sv, zv;
            if (p.sz_dtype == MI355_F32) {
                sv = ((const float*)sp)[ok ? n : 0];
                zv = ((const float*)zq)[ok ? n : 0];
            } else {
                sv = bf16_to_f32(((const bf16_t*)sp)[ok ? n : 0]);
                zv = bf16_to_f32(((const bf16_t*)zq)[ok ? n : 0]);
            }
            rowtab[i] = ok ? sv : 0.f;
            rowtab[kSlots * 16 + i] = ok ? 128.f + zv : 0.f;
        }
    }
    if constexpr (FUSE && EPI == MI355_EPI_ACCUM) {
        if (p.out_xb != nullptr) {
            for (int i = threadIdx.x; i < kSlots * 16; i += kThreads) {
                const int n = nb * kSlots * 16 + i;
                const float v = ldsz(p.next_norm, n < p.N ? n : 0, p.next_norm_dtype);
                rowtab[2 * kSlots * 16 + i] = n < p.N ? v : 0.f;
            }
        }
    }
    if (!(FUSE && p.f_in)) {
        for (int t = threadIdx.x; t < BM; t += kThreads) {
            const int m = m0 + t < p.M ? m0 + t : p.M - 1;
            fr[t] = p.rinv != nullptr ? p.rinv[m] : p.alpha;
            fr[BM + t] = GRP ? 0.f : p.sx[(int64_t)m * p.ksplit + ks];
        }
    }
    if constexpr (FUSE && EPI == MI355_EPI_STORE) {
        if (p.rope != nullptr)
            for (int t = threadIdx.x; t < BM; t += kThreads) postab[t] = p.pos[m0 + t < p.M ? m0 + t : p.M - 1];
    }
    xstore(u_lo & 1);
    __syncthreads();
    if constexpr (FUSE) {
        if (p.f_in) {
            constexpr int kP = kThreads >= BM ? kThreads / BM : 1;
            const float* frp = fr + 2 * BM;
            for (int t = threadIdx.x; t < BM; t += kThreads) {
                float sss = 0.f, sxs = 0.f;
#pragma unroll
                for (int part = 0; part < kP; ++part) {
                    sss += frp[(part * 2 + 0) * BM + t];
                    sxs += frp[(part * 2 + 1) * BM + t];
                }
                fr[t] = p.in_ss_n > 0 ? rsqrtf(sss / (float)p.K + p.eps) : 1.0f;
                fr[BM + t] = sxs;
            }
        }
    }

    // next unit's operands, requested UNCONDITIONALLY (a load inside `if (more)` makes hipcc drain vmcnt at the join,
    // i.e. wait for these very loads before the first MFMA): past the last unit the offsets fall into the next row /
    // tile or out of the descriptors (zeros) and the values are never used
    auto prefetch = [&](int u) {
        if constexpr (kXDma) {
            // (weights first: HBM latency; both pinned at the unit's start — they cost 8 registers now, not 40)
#pragma unroll
            for (int t = 0; t < kTPW; ++t) wnext[t] = wload(t, u + 1);
            xdma(u + 1, (u & 1) ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            return;
        }
        xload(u + 1);
#pragma unroll
        for (int t = 0; t < kTPW; ++t) wnext[t] = wload(t, u + 1);
    };
    // the 4 x kTT x kTPW MFMAs of a unit; sub >= 0 (GRP 2): only the lane groups of sub-group `sub` contribute
    // (explicitly software-pipelined B-fragment reads — 16 fragments in registers, pinned with sched_barrier —
    // measured SLOWER, 600-670 vs 760-800 TFLOP/s: with 4 waves per SIMD the hardware hides the LDS latency itself)
#if MI355_GEMM_AND_OR
    uint32_t cmask = 0x000F000Fu, cmagic = 0x43004300u;
    asm volatile("" : "+s"(cmask));
    asm volatile("" : "+v"(cmagic));
#endif
    constexpr int kBPipe = (GRP == 0 && BM == 128) ? MI355_GEMM_BPIPE : 0;
    auto bread = [&](const char* xs, int d, int tt, bool mine) {
        const int tok = tt * 16 + c;
        u32x4 braw = *(const u32x4*)(xs + tok * 256 + (((4 * g + d) ^ swz(tok)) << 4));
        if constexpr (GRP == 2) braw = mine ? braw : u32x4{0u, 0u, 0u, 0u};
        return braw;
    };
    auto mfmas = [&](int buf, int sub, int sub_shift) {
        const char* xs = smem + buf * (BM * 256);
        const bool mine = GRP != 2 || (g >> sub_shift) == sub;
        [[maybe_unused]] u32x4 bq[kBPipe > 0 ? kBPipe : 1];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            // int4 -> bf16 MFMA A fragments of k-quarter d: (w >> 4i) & 0x000F000F | 0x43004300 = (128 + q_2i, 128 + q_2i+1)
            bf16x8 a[kTPW];
#pragma unroll
            for (int t = 0; t < kTPW; ++t) {
                const uint32_t v = wcur[t][d];
                u32x4 f;
#if MI355_GEMM_AND_OR
                // (mask and exponent pattern as OPAQUE register values: hipcc then selects one v_and_or_b32 per field
                // — from literals it emits v_and + v_or, 11 instead of 7 VALU per dword — and pads the VALU -> MFMA
                // hazard itself, which an inline-asm v_and_or_b32 does not get: csrc/fused_step_ring.hip nib2f16)
                f[0] = (v & cmask) | cmagic;
                f[1] = ((v >> 4) & cmask) | cmagic;
                f[2] = ((v >> 8) & cmask) | cmagic;
                f[3] = ((v >> 12) & cmask) | cmagic;
#else
                f[0] = (v & 0x000F000Fu) | 0x43004300u;
                f[1] = ((v >> 4) & 0x000F000Fu) | 0x43004300u;
                f[2] = ((v >> 8) & 0x000F000Fu) | 0x43004300u;
                f[3] = ((v >> 12) & 0x000F000Fu) | 0x43004300u;
#endif
                a[t] = __builtin_bit_cast(bf16x8, f);
            }
            if constexpr (kBPipe > 0) {
                // fragment s = d * kTT + tt of the unit; bq holds the next kBPipe of them.  The group barriers pin "one LDS read (of
                // fragment s + kBPipe), then the MFMAs of fragment s": without them hipcc sinks every read to its use again
#pragma unroll
                for (int tt = 0; tt < kTT; ++tt) {
                    const int s = d * kTT + tt;
                    if (s == 0) {
#pragma unroll
                        for (int q = 0; q < kBPipe; ++q) bq[q] = bread(xs, q / kTT, q % kTT, mine);
                        __builtin_amdgcn_sched_group_barrier(0x100, kBPipe, 0);  // the unit's first kBPipe reads up front
                    }
                    const bf16x8 b = __builtin_bit_cast(bf16x8, bq[s % kBPipe]);
                    if (s + kBPipe < 4 * kTT) bq[s % kBPipe] = bread(xs, (s + kBPipe) / kTT, (s + kBPipe) % kTT, mine);
#pragma unroll
                    for (int t = 0; t < kTPW; ++t) acc[t][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b, acc[t][tt], 0, 0, 0);
                    if (s + kBPipe < 4 * kTT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, kTPW, 0);
                }
            } else {
#pragma unroll
                for (int tt = 0; tt < kTT; ++tt) {
                    const bf16x8 b = __builtin_bit_cast(bf16x8, bread(xs, d, tt, mine));
#pragma unroll
                    for (int t = 0; t < kTPW; ++t) acc[t][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b, acc[t][tt], 0, 0, 0);
                }
            }
        }
    };
    auto rotate = [&](int buf) {
        xstore(buf ^ 1);
#pragma unroll
        for (int t = 0; t < kTPW; ++t) wcur[t] = wnext[t];
        __syncthreads();
    };

    f32x4 accf[GRP ? kTPW : 1][GRP ? kTT : 1];
    if constexpr (GRP == 0) {
        for (int u = u_lo; u < u_hi; ++u) {
            prefetch(u);
            mfmas(u & 1, 0, 0);
            rotate(u & 1);
        }
    } else {
#pragma unroll
        for (int t = 0; t < kTPW; ++t)
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) accf[t][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
        u32x4 tabc[kTPW], tabn[kTPW];
        float sxv[kTT];
        auto tload = [&](int grp, u32x4 (&dst)[kTPW]) {  // rows 4 g .. 4 g + 3 of this wave's tiles: one 16-B load each
#pragma unroll
            for (int t = 0; t < kTPW; ++t) {
                const int tl = tile[t] < p.n_tiles ? tile[t] : 0;
                dst[t] = *(const u32x4*)(p.gtab + ((int64_t)grp * (PAIR ? 2 : 1) + rr[t]) * p.tab_ld + tl * 16 + 4 * g);
            }
        };
        auto sxload = [&](int grp) {
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) {
                const int m = m0 + tt * 16 + c;
                sxv[tt] = p.sxt[(int64_t)grp * p.M + (m < p.M ? m : 0)];
            }
        };
        auto apply = [&]() {  // end of a group: tabc = this group's pairs, tabn = the next group's
            // two FMAs per output element on register pairs (the VALU, not the matrix pipe, bounds
            // the grouped kernel: 64-token blocks halve the MFMAs a weight conversion is amortised over)
            f32x2 ds[kTPW][2], szp[kTPW][2];
#pragma unroll
            for (int t = 0; t < kTPW; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float s_c = __uint_as_float(tabc[t][r] << 16), z_c = __uint_as_float(tabc[t][r] & 0xffff0000u);
                    const float s_n = __uint_as_float(tabn[t][r] << 16);
                    ds[t][r >> 1][r & 1] = s_c - s_n;
                    szp[t][r >> 1][r & 1] = -(s_c * (128.f + z_c));
                }
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) {
                const f32x2 sx2 = {sxv[tt], sxv[tt]};
#pragma unroll
                for (int t = 0; t < kTPW; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const f32x2 a2 = {acc[t][tt][2 * h], acc[t][tt][2 * h + 1]};
                        f32x2 f2 = {accf[t][tt][2 * h], accf[t][tt][2 * h + 1]};
                        f2 = __builtin_elementwise_fma(ds[t][h], a2, f2);
                        f2 = __builtin_elementwise_fma(szp[t][h], sx2, f2);
                        accf[t][tt][2 * h] = f2[0];
                        accf[t][tt][2 * h + 1] = f2[1];
                    }
            }
#pragma unroll
            for (int t = 0; t < kTPW; ++t) tabc[t] = tabn[t];
        };
        // (a K-slice is a sum of its own: past its last group the scale is 0 — table row n_groups)
        const int sub_shift = p.gq_shift;  // lane groups per sub-group = 1 << gq_shift (0: 32 columns, 1: 64)
        const int nsub = 4 >> sub_shift;
        tload(u_lo * nsub, tabc);
        for (int u = u_lo; u < u_hi; ++u) {
            prefetch(u);
#pragma unroll 1
            for (int sub = 0; sub < nsub; ++sub) {
                const int grp = u * nsub + sub < p.n_groups ? u * nsub + sub : p.n_groups - 1;
                tload((u == u_hi - 1 && sub == nsub - 1) ? p.n_groups : grp + 1, tabn);
                sxload(grp);
                mfmas(u & 1, sub, sub_shift);
                apply();
            }
            rotate(u & 1);
        }
    }

    if constexpr (GRP != 0) {
#pragma unroll
        for (int t = 0; t < kTPW; ++t)
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) acc[t][tt] = accf[t][tt];
    }
    gemm_epilogue<EPI, PAIR, MI355_W_Q4, kWaves, BM, GRP, FUSE, kTPW>(p, acc, smem, fr, postab, rowtab, tile, m0, nb, ks, wave, lane);
}

// 16 B per lane from `off` + `scalar_off` of a buffer to 1 KiB of LDS (lane i's bytes at 16 i); out of range: zeros
__device__ __forceinline__ void lds_from(__amdgpu_buffer_rsrc_t r, char* lds, unsigned off, int scalar_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, scalar_off, 0, 0);
}

// Four bytes per lane, each lane's from its own place, to 256 B of LDS that nobody reads: what this is for are the cache lines
__device__ __forceinline__ void lds_touch(__amdgpu_buffer_rsrc_t r, char* lds, unsigned off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4, off, 0, 0, 0);
}

// The same product for launches that leave a CU one or two workgroups (short prompts, batches of decoding sequences, the N = 4096 products of longer ones):
// there nothing else covers a unit's memory latency, and gemm_q4_kernel, one unit ahead, paid it per unit (1.3-1.5 us a unit at T = 777, 16 rows: 1 TB/s
// of weights).  Here the weights (registers) and the activations (LDS, by DMA) of the next DEPTH - 1 units are under way; a unit waits for its own requests
// alone (a counted vmcnt, then the workgroup's barrier), so 3 x 16 KiB of weights (int4) or 3 x 64 KiB (bf16) per 8 waves are always in flight; bf16 blocks of 96 to 192 tokens and int4 ones of 160
// and 192, whose activations fill the LDS, have two units under way, bf16 ones of 208 and 256 one.
// BM: 16 / 32 / 48 / 64 / 128 tokens, int4 also 96 / 160 / 192 (groups not 192), BF16 96 / 160 / 192 / 208 / 256.  Sums run in the order of gemm_q4_kernel (RUNS: within a run).
// BF16: what bounds it is the CU's memory pipeline, which returns data in the order of the requests and holds some 50 KB of them: with nothing but its requests (no
// products) a block of 128 tokens x 256 rows took 1.67 us for the 96 KB of a unit, 0.95 when all of it lay in L2.  So the requests of a unit are spread over all of its
// products (in the first half of them, as before, the waves stood at requests that the pipeline had no room for: N = 4096, K = 16512, 2048 tokens 248 -> 226 us with what follows,
// N = 12288, K = 4096 214 -> 186); large blocks ask for fewer bytes per product; and where four blocks or more of a row block run on an XCD, they bring its weights to
// the XCD's L2 a round ahead, each a share, one lane per cache line: a block then waits for HBM once per round for its share and not for every line behind
// every other (N = 4096, K = 11008, 777 tokens in blocks of 64 x 256 102 -> 90 us; blocks of 64 x 128 7 % less on average, of 128 x 128 4 %; 8 waves from 128 tokens on nothing).  The
// activations likewise: 5-25 % slower, few blocks of an XCD share them.  A last block of few tokens runs ahead of the others and does it for them.
// GRP with FUSE: a unit's operand sums are the producer's shares, the tables come from group_tables_kernel.  1000 tokens, 7B, 8 layers with a staging pass in front
// of each product 4.59 ms, in the chain 4.31 (the products themselves 3-5 % slower: 1/rms from shares, operand and shares of the next product).
// GRP (Q4, groups of whole 128-column units): the products of a unit start from 0, and accf += s_unit * them, one FMA per output element and unit on the
// VALU beside the next unit's products; the zero points, accf -= sum over units of s (128 + z) X_unit (X: the unit's operand sums), are a product with K =
// units / 4 of their own on the f32 MFMA in front of the loop.
// RUNS (Q4): a slice of several runs (gemm_runs()).  The second set of sums is 32 registers, with which two workgroups of 8 waves no longer share a CU: kernels of
// their own.
// ONCE: one token block (BM tokens at most) and weights that come from HBM (MI355_LF_STREAMED), so nothing reads a piece of them again: they are requested non-temporal and push no activations
// out of the L2 caches.  BF16, 16 products of 2048 to 32000 rows, weights in no cache: 16 tokens 0.89 times as long (0.86 to 0.94; N = 4096, K = 16512 30.9 -> 26.8 us, N = 32000, K = 4096 52.0 ->
// 46.0), 24 tokens 0.91, 40 0.93, 64 0.95 (two of 16 up to 1.01).  Int4 of one scale per row, nine products, 600 MB of copies, 16 / 32 / 37 / 48 tokens 0.92 / 0.93 / 0.94 / 0.95, groups of 128 columns 0.92 / 0.95 / 0.96 / 0.98.
// Weights that a cache holds it costs: ten BF16 products of 1024 to 8192 rows, all copies read in turn 100 / 200 / 256 / 288 / 320 / 352 / 600 MB, 16 tokens 1.07 / 1.08 / 1.05 / 1.02 / 0.97 / 0.95 / 0.92 times
// as long (100 MB: N = 6144, K = 2048 1.28), one copy again and again 1.12 (1.54).
template <int EPI, bool PAIR, int FMT, int kWaves, int BM, bool FUSE, int DEPTH, int GRP = 0, bool RUNS = false, int TPW = kTPW, bool ONCE = false>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_deep_kernel(const GemmParams p) {
    static_assert(GRP == 0 || (FMT == MI355_W_Q4 && GRP == 1), "grouped scales are a Q4 feature");
    static_assert(!RUNS || (FMT == MI355_W_Q4 && GRP == 0), "runs: int4 sums, one scale per row");
    static_assert(TPW == 2 || (TPW == 1 && !PAIR), "a pair is two row tiles");
    static_assert(DEPTH >= 2 && DEPTH <= 4, "units under way + 1");
    constexpr int kTT = BM / 16, kSlots = kWaves * TPW, kThreads = 64 * kWaves;
    constexpr int kWP = FMT == MI355_W_BF16 ? 4 : 1;
    constexpr int kXI = (BM / 4 + kWaves - 1) / kWaves;  // activation requests (1 KiB: four tokens) per wave and unit
    constexpr int kUnit = kXI + TPW * kWP + (GRP ? TPW : 0);  // requests per wave and unit
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int n_blocks = p.n_blocks;
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    const int L2 = xcd * p.per_xcd + j;
    if (j >= p.per_xcd || L2 >= p.total_blocks * p.ksplit) return;
    const int L = L2 / p.ksplit, ks = L2 - L * p.ksplit;
    const int m_blocks = p.total_blocks / n_blocks;
    int mb, nb;
    if constexpr (FMT == MI355_W_BF16) {  // (orders: see gemm_q4_kernel)
        const BlockAt at = block_at(L, n_blocks, m_blocks, may_run_in_squares(kWaves, BM) && p.squares);
        nb = at.nb, mb = at.mb;
    } else {
        mb = L / n_blocks;
        nb = L - mb * n_blocks;
    }
    const int m0 = mb * BM;
    const int u_lo = slice_lo(ks, p.units, p.ksplit), u_hi = slice_lo(ks + 1, p.units, p.ksplit);
    float* fr = (float*)(smem + DEPTH * BM * 256);
    [[maybe_unused]] float* frp = fr + 2 * BM;
    [[maybe_unused]] int* postab = (int*)(smem + kPosAt<BM, DEPTH>);
    [[maybe_unused]] float* rowtab = (float*)(smem + kRowAt<BM, FUSE, DEPTH>);
    [[maybe_unused]] float* runtab = rowtab + 3 * kSlots * 16;  // [part of a run's sum][run][BM] operand sums
    int tile[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t)
        tile[t] = PAIR ? nb * (kSlots / 2) + (TPW / 2) * wave + (t >> 1) : nb * kSlots + TPW * wave + t;
    // this block's share of its row block's weights (see above): thread i's line of every round of DEPTH units, at touch_off from the round's first unit
    constexpr bool kTouch = FMT == MI355_W_BF16 && shares_weights(kWaves, BM) && !ONCE;
    constexpr int kTouchAhead = 2 * DEPTH - 1, kStreams = PAIR ? kSlots / 2 : kSlots, kRun = DEPTH * (PAIR ? 64 : 32);  // kRun: lines of DEPTH units of a tile
    constexpr unsigned kNone = 0xFFFFFFF0u;
    [[maybe_unused]] unsigned touch_off = kNone;
    if constexpr (kTouch) {
        const L2Share mine = l2_share(kStreams * kRun, L, nb, m_blocks, p.ksplit, xcd, p.per_xcd);
        const int line = mine.first + (int)threadIdx.x, stream = line / kRun, at = line - stream * kRun;
        if ((p.M - 1) % BM >= BM / 2 && (int)threadIdx.x < mine.count && line < kStreams * kRun && nb * kStreams + stream < p.n_tiles)
            touch_off = (unsigned)((nb * kStreams + stream) * p.units) * (PAIR ? 8192u : 4096u) + at * 128u;
    }
    [[maybe_unused]] const bool touching = __builtin_amdgcn_ballot_w64(touch_off != kNone) != 0;
    const bf16_t* xbase = p.xb;
    if constexpr (EPI == MI355_EPI_STORE && FMT == MI355_W_BF16 && !FUSE) {
        if (p.slice_blocks != 0) xbase += (int64_t)(nb / p.slice_blocks) * p.slice_stride;
    }
    const int x_bytes = (int)(unsigned)((int64_t)p.M * p.ldxb * 2);
    const unsigned lane_off = lane * 16;
    // this lane's token and column of its activation requests (waves beyond the block's BM / 4 requests repeat one: the same bytes to the same place)
    unsigned xoff[kXI];
    int xdst[kXI];
#pragma unroll
    for (int i = 0; i < kXI; ++i) {
        const int q = (i * kWaves + wave) % (BM / 4);
        const int tok = q * 4 + (lane >> 4), slot = lane & 15;
        xoff[i] = m0 + tok < p.M ? (unsigned)((int64_t)(m0 + tok) * p.ldxb * 2) + (unsigned)((slot ^ swz(tok)) * 16) : 0xFFFFFFF0u;
        xdst[i] = q * 1024;
    }
    u32x4 wr[DEPTH][TPW][kWP];
    [[maybe_unused]] u32x4 tb[GRP ? DEPTH : 1][TPW];  // (scale, zero) of rows 4 g .. 4 g + 3 in the unit's group
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc((void*)p.gtab, 0, GRP ? (p.n_groups + 1) * (PAIR ? 2 : 1) * p.tab_ld * 4 : 0, 0x00020000);
    [[maybe_unused]] const int tbstep = (PAIR ? 2 : 1) * p.tab_ld * 4;
    [[maybe_unused]] int tboff[TPW];  // (tiles past the last read the first one's)
#pragma unroll
    for (int t = 0; t < TPW; ++t) tboff[t] = ((PAIR ? t & 1 : 0) * p.tab_ld + (tile[t] < p.n_tiles ? tile[t] * 16 : 0) + 4 * g) * 4;
    // request i of unit u: activations first.  What tells the units apart is scalar (offsets, and the size in the descriptor): no address
    // instruction on the VALU.  Past the slice or the tiles: a size of 0, nothing is read (the scalar offset is not range-checked), zeros go to a buffer that
    // nobody reads
    auto request = [&](int i, int u, int slot) __attribute__((always_inline)) {
        const bool in = u < u_hi;
        if (i < kXI) {
            const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)xbase, 0, in ? x_bytes : 0, 0x00020000);
            lds_from(rx, smem + slot * (BM * 256) + xdst[i < kXI ? i : 0], xoff[i < kXI ? i : 0], in ? u * 256 : 0);
        } else if (i >= kXI + TPW * kWP) {
            const int t = i - (kXI + TPW * kWP) < TPW ? i - (kXI + TPW * kWP) : 0;
            tb[GRP ? slot : 0][t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rt, tboff[t], ((in ? u : u_hi - 1) >> p.gq_shift) * tbstep, 0));
        } else {
            const int t = (i - kXI) / kWP, d = (i - kXI) % kWP;
            const bool ok = tile[t] < p.n_tiles && in;
            const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, ok ? (int)p.w_bytes : 0, 0x00020000);
            const unsigned off = (unsigned)((tile[t] * p.units + u) * (PAIR ? 2 : 1) + (PAIR ? t & 1 : 0)) * (1024u * kWP) + d * 1024u;
            wr[slot][t][d] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, lane_off, ok ? off : 0u, ONCE ? 2 : 0));
        }
    };

    [[maybe_unused]] auto touch = [&](int u) __attribute__((always_inline)) {  // (a round that is not whole: a size of 0)
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, u + DEPTH <= u_hi ? (int)p.w_bytes : 0, 0x00020000);
        lds_touch(rw, smem + kRowAt<BM, FUSE, DEPTH> + 3 * kSlots * 64, touch_off == kNone ? kNone : touch_off + (unsigned)u * (PAIR ? 8192u : 4096u));
    };

    // ---- tables of the epilogue: requested ahead of the units, written to LDS behind their requests
    constexpr bool kScales = FMT == MI355_W_Q4 && GRP == 0;
    constexpr int kRT = (kSlots * 16 + kThreads - 1) / kThreads;
    [[maybe_unused]] float t_sc[kRT], t_zp[kRT], t_ns[kRT];
    if constexpr (kScales) {
        const bool f32 = p.sz_dtype == MI355_F32;
#pragma unroll
        for (int i = 0; i < kRT; ++i) {
            const int r = i * kThreads + threadIdx.x, slot = r >> 4;
            const int n = (PAIR ? nb * (kSlots / 2) + (slot >> 1) : nb * kSlots + slot) * 16 + (r & 15);
            const int at = n < p.N ? n : 0;
            const void* sp = PAIR && (slot & 1) ? p.scales2 : p.scales;
            const void* zq = PAIR && (slot & 1) ? p.zeros2 : p.zeros;
            float sv, zv;
            if (f32) {
                sv = ((const float*)sp)[at];
                zv = ((const float*)zq)[at];
            } else {
                sv = bf16_to_f32(((const bf16_t*)sp)[at]);
                zv = bf16_to_f32(((const bf16_t*)zq)[at]);
            }
            t_sc[i] = n < p.N ? sv : 0.f;
            t_zp[i] = n < p.N ? 128.f + zv : 0.f;
        }
    }
    const bool norm_tab = FUSE && EPI == MI355_EPI_ACCUM && p.out_xb != nullptr;
    if constexpr (FUSE && EPI == MI355_EPI_ACCUM) {
        if (norm_tab) {
#pragma unroll
            for (int i = 0; i < kRT; ++i) {
                const int n = nb * kSlots * 16 + i * kThreads + (int)threadIdx.x;
                t_ns[i] = n < p.N ? ldsz(p.next_norm, n, p.next_norm_dtype) : 0.f;
            }
        }
    }
    const int mt = (int)threadIdx.x < BM ? (m0 + (int)threadIdx.x < p.M ? m0 + (int)threadIdx.x : p.M - 1) : p.M - 1;
    const bool own = !(FUSE && p.f_in);  // factors of the tokens as they are, not as shares
    float t_ri = p.alpha;
    if (own && p.rinv != nullptr) t_ri = p.rinv[mt];
    constexpr int kSX = RUNS ? (kMaxRuns * BM + kThreads - 1) / kThreads : 1;
    [[maybe_unused]] float t_sx[kSX];  // operand sum of token (i kThreads + thread) % BM in run (...) / BM
    if constexpr (kScales) {
        if (own) {
            if constexpr (!RUNS) {
                t_sx[0] = p.sx[(int64_t)mt * p.ksplit + ks];
            } else {
#pragma unroll
                for (int i = 0; i < kSX; ++i) {
                    const int at = i * kThreads + (int)threadIdx.x, run = at / BM < p.runs ? at / BM : 0, m = m0 + at % BM;
                    t_sx[i] = p.sx[((int64_t)(m < p.M ? m : p.M - 1) * p.ksplit + ks) * p.runs + run];
                }
            }
        }
    }
    [[maybe_unused]] int t_pos = 0;
    if constexpr (FUSE && EPI == MI355_EPI_STORE) {
        if (p.rope != nullptr) t_pos = p.pos[mt];
    }
    // shares of the tokens' factors (gemm_fuse.h): every thread a token and every kP-th share, in share order; the first kIn of them now.  Operand sums of several
    // runs: kP / runs threads take a run's shares in turn, and end_run() adds their sums
    constexpr int kP = kThreads / BM < 8 ? kThreads / BM : 8, kIn = kSharesAhead;
    const int s_tok = threadIdx.x % BM, s_part = threadIdx.x / BM;
    [[maybe_unused]] const int64_t s_m = m0 + s_tok < p.M ? m0 + s_tok : p.M - 1;
    [[maybe_unused]] const int s_lo = FUSE && p.ksplit > 1 ? u_lo * p.in_ppu : 0, s_hi = FUSE && p.ksplit > 1 ? u_hi * p.in_ppu : p.in_sx_n;
    // (kP <= 8 and two runs at least: quotients of up to 4, without a division in front of the first request)
    auto over_runs = [&](int v) { return (v >= p.runs) + (v >= 2 * p.runs) + (v >= 3 * p.runs) + (v >= 4 * p.runs); };
    [[maybe_unused]] const int subs = RUNS && !own && kP >= 2 * p.runs ? over_runs(kP) : 1;
    [[maybe_unused]] const int s_sub = subs > 1 ? over_runs(s_part) : 0, s_run = s_part - s_sub * p.runs;
    [[maybe_unused]] const int s_first = s_lo + (RUNS ? s_run * p.run_units * p.in_ppu + s_sub : s_part);
    [[maybe_unused]] auto run_end = [&](int run) { return (u_lo + (run + 1) * p.run_units < u_hi ? u_lo + (run + 1) * p.run_units : u_hi) * p.in_ppu; };
    [[maybe_unused]] float vx[kIn], vs[kIn];
    auto shares = [&](const float* in, int j0, int step, int hi, float (&v)[kSharesAhead]) {
#pragma unroll
        for (int i = 0; i < kIn; ++i) v[i] = in[(j0 + i * step < hi ? j0 + i * step : 0) * (int64_t)p.M + s_m];
    };
    auto add_shares = [&](int j0, int step, int hi, const float (&v)[kSharesAhead], float sum) {
#pragma unroll
        for (int i = 0; i < kIn; ++i) sum += j0 + i * step < hi ? v[i] : 0.f;
        return sum;
    };
    if constexpr (FUSE) {
        if (!own && s_part < kP) {
            if constexpr (GRP == 0) shares(p.in_sx, s_first, RUNS ? subs : kP, RUNS ? run_end(s_run) : s_hi, vx);  // (GRP takes them unit by unit, below)
            if (p.in_ss_n > 0) shares(p.in_ss, s_part, kP, p.in_ss_n, vs);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < DEPTH - 1; ++s) {
#pragma unroll
        for (int i = 0; i < kUnit; ++i) request(i, u_lo + s, s);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kTouch) {
            if (s == 0 && touching) touch(u_lo + DEPTH - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    [[maybe_unused]] float sxs = 0.f, sss = 0.f;
    if constexpr (FUSE) {
        if (!own && s_part < kP) {
            if constexpr (RUNS) {
                for (int run = s_run; run < p.runs && s_sub < subs; run += kP) {
                    float sum = 0.f;
                    for (int j0 = s_lo + run * p.run_units * p.in_ppu + s_sub, hi = run_end(run); j0 < hi; j0 += kIn * subs) {
                        if (run != s_run || j0 != s_first) shares(p.in_sx, j0, subs, hi, vx);
                        sum = add_shares(j0, subs, hi, vx, sum);
                    }
                    runtab[(run + s_sub * p.runs) * BM + s_tok] = sum;
                }
            } else if constexpr (GRP == 0) {
                sxs = add_shares(s_first, kP, s_hi, vx, 0.f);
            }
            if (p.in_ss_n > 0) sss = add_shares(s_part, kP, p.in_ss_n, vs, 0.f);
            if constexpr (GRP != 0) {  // (all of them now: the zero points' product in front of the loop waits for its loads anyway, and the loop has no register to spare)
                for (int j0 = s_part + kIn * kP; j0 < p.in_ss_n; j0 += kIn * kP) {
                    shares(p.in_ss, j0, kP, p.in_ss_n, vs);
                    sss = add_shares(j0, kP, p.in_ss_n, vs, sss);
                }
                frp[(s_part * 2 + 0) * BM + s_tok] = sss;
            }
        }
    }
    if constexpr (kScales) {
#pragma unroll
        for (int i = 0; i < kRT; ++i) {
            const int r = i * kThreads + (int)threadIdx.x;
            if (kSlots * 16 % kThreads == 0 || r < kSlots * 16) rowtab[r] = t_sc[i], rowtab[kSlots * 16 + r] = t_zp[i];
        }
    }
    if constexpr (FUSE && EPI == MI355_EPI_ACCUM) {
        if (norm_tab) {
#pragma unroll
            for (int i = 0; i < kRT; ++i) {
                const int r = i * kThreads + (int)threadIdx.x;
                if (kSlots * 16 % kThreads == 0 || r < kSlots * 16) rowtab[2 * kSlots * 16 + r] = t_ns[i];
            }
        }
    }
    if constexpr (kScales) {
        if (own) {
#pragma unroll
            for (int i = 0; i < kSX; ++i) {
                const int at = i * kThreads + (int)threadIdx.x;
                if (RUNS && at < p.runs * BM) runtab[at] = t_sx[i];
                if (at < BM) fr[BM + at] = RUNS ? 0.f : t_sx[i];
            }
        }
    }
    if ((int)threadIdx.x < BM) {
        if (own) fr[threadIdx.x] = t_ri;
        if constexpr (FUSE && EPI == MI355_EPI_STORE) postab[threadIdx.x] = t_pos;
    }

    f32x4 acc[TPW][kTT];
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) acc[t][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t cmask = 0x000F000Fu, cmagic = 0x43004300u;  // (opaque: see gemm_q4_kernel)
    asm volatile("" : "+s"(cmask));
    asm volatile("" : "+v"(cmagic));
    auto levels = [&](uint32_t v) __attribute__((always_inline)) {  // eight int4 levels as bf16 128 + q
        return __builtin_bit_cast(bf16x8, u32x4{(v & cmask) | cmagic, ((v >> 4) & cmask) | cmagic, ((v >> 8) & cmask) | cmagic, ((v >> 12) & cmask) | cmagic});
    };
    if constexpr (GRP != 0) {
        // lane (g, c): units u0 + 4 g + i of product i; a chunk's factors are requested while the one before is multiplied
        struct Chunk { uint32_t sz[4][TPW]; float x[4][kTT]; };
        const bool halves = FUSE && p.in_ppu == 2;  // a producer in blocks of 64 hidden rows leaves two shares a unit
        const int64_t x_step = halves ? 2 * (int64_t)p.M : p.M;
        auto fetch = [&](int u0, Chunk& k) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int u = u0 + 4 * g + i < u_hi ? u0 + 4 * g + i : u_hi - 1;
#pragma unroll
                for (int t = 0; t < TPW; ++t)
                    k.sz[i][t] = p.gtab[((int64_t)(u >> p.gq_shift) * (PAIR ? 2 : 1) + (PAIR ? t & 1 : 0)) * p.tab_ld + (tile[t] < p.n_tiles ? tile[t] * 16 : 0) + c];
#pragma unroll
                for (int tt = 0; tt < kTT; ++tt) k.x[i][tt] = p.sxt[(int64_t)u * x_step + (m0 + tt * 16 + c < p.M ? m0 + tt * 16 + c : p.M - 1)];
                if constexpr (FUSE) {
                    if (halves) {
#pragma unroll
                        for (int tt = 0; tt < kTT; ++tt) k.x[i][tt] += p.sxt[(int64_t)u * x_step + p.M + (m0 + tt * 16 + c < p.M ? m0 + tt * 16 + c : p.M - 1)];
                    }
                }
            }
        };
        Chunk cur, nxt;
        fetch(u_lo, cur);
        for (int u0 = u_lo; u0 < u_hi; u0 += 16) {
            fetch(u0 + 16 < u_hi ? u0 + 16 : u0, nxt);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = u0 + 4 * g + i < u_hi;
                float a[TPW];
#pragma unroll
                for (int t = 0; t < TPW; ++t)
                    a[t] = in ? -__uint_as_float(cur.sz[i][t] << 16) * (128.f + __uint_as_float(cur.sz[i][t] & 0xffff0000u)) : 0.f;
#pragma unroll
                for (int tt = 0; tt < kTT; ++tt) {
                    const float x = in ? cur.x[i][tt] : 0.f;
#pragma unroll
                    for (int t = 0; t < TPW; ++t) acc[t][tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], x, acc[t][tt], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): registers of a load whose result nobody takes are waited for where they are used next, in the loop
    }
    constexpr int kFrags = 4 * kTT, kPipe = 4;
    // the requests of unit `ahead` go out between the products: a request takes the CU's memory pipeline 16 cycles, and in one burst behind the barrier
    // the waves of a workgroup stood in line for it with no product under way
    constexpr int kEvery = kFrags >= kUnit ? kFrags / kUnit : 1;  // fragments from one request to the next
    constexpr int kPer = (kUnit + kFrags - 1) / kFrags;                      // requests behind one fragment
    // GRP: token tile by token tile, so the sums of one unit live in two token tiles' registers: those being summed, and those being scaled
    auto mfmas_grouped = [&](int slot, u32x4 (&w)[TPW][kWP], u32x4 (&sz)[TPW], int ahead, int ahead_slot, auto more) __attribute__((always_inline)) {
        const char* xs = smem + slot * (BM * 256);
        auto bread = [&](int f) {  // fragment f = tt * 4 + d
            const int tok = (f >> 2) * 16 + c;
            return *(const u32x4*)(xs + tok * 256 + (((4 * g + (f & 3)) ^ swz(tok)) << 4));
        };
        u32x4 bq[kPipe];
#pragma unroll
        for (int q = 0; q < kPipe; ++q) bq[q] = bread(q);
        __builtin_amdgcn_sched_group_barrier(0x100, kPipe, 0);
        bf16x8 a[4][TPW];
        f32x4 sc[TPW];
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                a[d][t] = levels(w[t][0][d]);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[t][r] = __uint_as_float(sz[t][r] << 16);
        }
        f32x4 un[2][TPW];
#pragma unroll
        for (int f = 0; f < kFrags; ++f) {
            const int tt = f >> 2, d = f & 3;
            const bf16x8 b = __builtin_bit_cast(bf16x8, bq[f % kPipe]);
            if (f + kPipe < kFrags) bq[f % kPipe] = bread(f + kPipe);
#pragma unroll
            for (int t = 0; t < TPW; ++t)
                un[tt & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][t], b, d == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : un[tt & 1][t], 0, 0, 0);
            if (f + kPipe < kFrags) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, TPW, 0);
            if (more && f % kEvery == 0) {
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    const int r = f / kEvery * kPer + i;
                    if (r >= kUnit) continue;
                    request(r, ahead, ahead_slot);
                    __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
                }
            }
            if (tt > 0 && d > 0 && d <= TPW) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[d - 1][tt - 1][r] = __builtin_fmaf(sc[d - 1][r], un[(tt - 1) & 1][d - 1][r], acc[d - 1][tt - 1][r]);
                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][kTT - 1][r] = __builtin_fmaf(sc[t][r], un[(kTT - 1) & 1][t][r], acc[t][kTT - 1][r]);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mfmas = [&](int slot, u32x4 (&w)[TPW][kWP], int ahead, int ahead_slot, auto more) __attribute__((always_inline)) {
        const char* xs = smem + slot * (BM * 256);
        auto bread = [&](int f) {  // fragment f = d * kTT + tt
            const int tok = (f % kTT) * 16 + c;
            return *(const u32x4*)(xs + tok * 256 + (((4 * g + f / kTT) ^ swz(tok)) << 4));
        };
        u32x4 bq[kPipe];
#pragma unroll
        for (int q = 0; q < kPipe; ++q) bq[q] = bread(q);
        __builtin_amdgcn_sched_group_barrier(0x100, kPipe, 0);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            bf16x8 a[TPW];
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                if constexpr (FMT == MI355_W_BF16)
                    a[t] = __builtin_bit_cast(bf16x8, w[t][d]);
                else
                    a[t] = levels(w[t][0][d]);
            }
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) {
                const int f = d * kTT + tt;
                const bf16x8 b = __builtin_bit_cast(bf16x8, bq[f % kPipe]);
                if (f + kPipe < kFrags) bq[f % kPipe] = bread(f + kPipe);
#pragma unroll
                for (int t = 0; t < TPW; ++t) acc[t][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b, acc[t][tt], 0, 0, 0);
                if (f + kPipe < kFrags) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, TPW, 0);
                if (more && f % kEvery == 0) {
#pragma unroll
                    for (int i = 0; i < kPer; ++i) {
                        const int r = f / kEvery * kPer + i;
                        if (r >= kUnit) continue;
                        request(r, ahead, ahead_slot);
                        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // DEPTH units a round: own requests of a unit have landed (those of the DEPTH - 2 units behind it may be under way); every wave's have, and every wave is
    // done with the unit before: its buffer and registers take the unit DEPTH - 1 ahead.  The last, shorter round stands behind the loop and requests nothing:
    // with a way out between the units hipcc joins all of them in front of the loop's head and waits there for every request under way, once a round.
    auto unit = [&](auto slot, int u, auto more) __attribute__((always_inline)) {
        constexpr int s = slot, kNewer = more ? (DEPTH - 2) * kUnit : (DEPTH - 2 - s) * kUnit;
        if constexpr (kTouch && s > 0 && s < DEPTH - 1 && more) {
            if (touching)
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kNewer + 1) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kNewer) : "memory");
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kNewer) : "memory");
        }
        if constexpr (kTouch && s == 0 && more) {
            if (touching) touch(u + kTouchAhead);
        }
        if constexpr (GRP != 0)
            mfmas_grouped(s, wr[s], tb[s], u + DEPTH - 1, (s + DEPTH - 1) % DEPTH, more);
        else
            mfmas(s, wr[s], u + DEPTH - 1, (s + DEPTH - 1) % DEPTH, more);
    };
    using std::integral_constant;
    // the sum of a run, its levels' offset and zero points taken off, leaves the accumulators
    [[maybe_unused]] f32x4 of_runs[RUNS ? TPW : 1][RUNS ? kTT : 1];
    [[maybe_unused]] int run = 0, left = p.run_units;
    [[maybe_unused]] auto end_run = [&]() __attribute__((always_inline)) {
        float x[kTT];
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) x[tt] = runtab[run * BM + tt * 16 + c];
        for (int q = 1; q < subs; ++q)
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) x[tt] += runtab[(run + q * p.runs) * BM + tt * 16 + c];
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            const f32x4 zp = *(const f32x4*)(rowtab + (kSlots + TPW * wave + t) * 16 + 4 * g);
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    of_runs[t][tt][r] += acc[t][tt][r] - zp[r] * x[tt];
                    acc[t][tt][r] = 0.f;
                }
            }
        }
        ++run;
        left = p.run_units;
    };
    if constexpr (RUNS) {
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) of_runs[t][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int u = u_lo;
    for (; u + DEPTH <= u_hi; u += DEPTH) {
        unit(integral_constant<int, 0>{}, u, std::true_type{});
        unit(integral_constant<int, 1>{}, u + 1, std::true_type{});
        if constexpr (DEPTH > 2) unit(integral_constant<int, 2>{}, u + 2, std::true_type{});
        if constexpr (DEPTH == 4) unit(integral_constant<int, 3>{}, u + 3, std::true_type{});
        if constexpr (RUNS) {
            left -= DEPTH;
            if (left == 0) end_run();
        }
    }
    [[maybe_unused]] const bool open = u < u_hi || left != p.run_units;  // the last run has units
    if (u < u_hi) {
        unit(integral_constant<int, 0>{}, u, std::false_type{});
        if constexpr (DEPTH > 2) {
            if (u + 1 < u_hi) {
                unit(integral_constant<int, 1>{}, u + 1, std::false_type{});
                if constexpr (DEPTH == 4) {
                    if (u + 2 < u_hi) unit(integral_constant<int, 2>{}, u + 2, std::false_type{});
                }
            }
        }
    }
    if constexpr (RUNS) {
        if (open) end_run();
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int tt = 0; tt < kTT; ++tt) acc[t][tt] = of_runs[t][tt];
    }
    if constexpr (FUSE) {
        if (p.f_in) {  // the rest of the shares
            if (GRP == 0 && s_part < kP) {
                for (int j0 = s_first + kIn * kP; !RUNS && j0 < s_hi; j0 += kIn * kP) {
                    shares(p.in_sx, j0, kP, s_hi, vx);
                    sxs = add_shares(j0, kP, s_hi, vx, sxs);
                }
                for (int j0 = s_part + kIn * kP; j0 < p.in_ss_n; j0 += kIn * kP) {
                    shares(p.in_ss, j0, kP, p.in_ss_n, vs);
                    sss = add_shares(j0, kP, p.in_ss_n, vs, sss);
                }
                frp[(s_part * 2 + 1) * BM + s_tok] = sxs;
                frp[(s_part * 2 + 0) * BM + s_tok] = sss;
            }
            __syncthreads();
            if ((int)threadIdx.x < BM) {
                sss = sxs = 0.f;
#pragma unroll
                for (int q = 0; q < kP; ++q) {
                    sss += frp[(q * 2 + 0) * BM + threadIdx.x];
                    if constexpr (GRP == 0) sxs += frp[(q * 2 + 1) * BM + threadIdx.x];
                }
                fr[threadIdx.x] = p.in_ss_n > 0 ? rsqrtf(sss / (float)p.K + p.eps) : 1.0f;
                fr[BM + threadIdx.x] = sxs;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (requests past the slice wrote zeros: none may land in what the epilogue keeps there)
    __syncthreads();
    gemm_epilogue<EPI, PAIR, FMT, kWaves, BM, GRP, FUSE, TPW>(p, acc, smem, fr, postab, rowtab, tile, m0, nb, ks, wave, lane);
}

// BF16 blocks of 8 waves.  Row block by row block, the 32 blocks that an XCD runs side by side are all token blocks of two or three row blocks: with 16 token blocks of 128 they
// bring 2 x 64 KB of weights and 16 x 32 of activations to its L2 per unit.  As 4 row blocks by 8 token blocks 4 x 64 + 8 x 32, a fifth less of what all of them wait for: 2048 tokens, N =
// 4096, K = 16512 246 -> 218 us, 1800 tokens 211 -> 195.  Over 15 products, 129 to 2048 tokens: more than 12 token blocks 0.987 times (0.90 to 1.03: the same launch differs by 2 % between
// processes), 9 to 12 1.00 times where K is above 8192 (0.94 to 1.04) and 1.01 below, fewer 1.01 (the two divisions).
bool square_blocks(int m_blocks, int units) { return m_blocks > 12 || (m_blocks > 8 && units > 64); }
template <int EPI, bool PAIR, int kWaves, int BM, bool FUSE, int TPW, typename Kernel>
int launch_blocks(Kernel kernel, int lds, const GemmParams& p, hipStream_t s) {  // p.n_tiles: 16-row tiles (pair tiles for the SwiGLU stream)
    constexpr int kSlots = kWaves * TPW;
    const int per_block = PAIR ? kSlots / 2 : kSlots;
    MI355_CHECK_ARG(p.slice_blocks % (16 * per_block) == 0, MI355_E_STATE, "linear_gemm: blocks of %d rows do not divide operand slices of %d", 16 * per_block, p.slice_blocks);
    GemmParams q = p;
    q.n_blocks = (p.n_tiles + per_block - 1) / per_block;
    q.slice_blocks = p.slice_blocks / (16 * per_block);  // (in: rows)
    q.total_blocks = q.n_blocks * ((p.M + BM - 1) / BM);
    q.per_xcd = (q.total_blocks * q.ksplit + 7) / 8;
    q.squares = square_blocks((p.M + BM - 1) / BM, p.units);
    if constexpr (FUSE) {
        if (q.ksplit > 1) {  // the producer roles move to the reduction of the K-slices
            q.out_xb = nullptr;
            q.out_ss = q.out_sx = nullptr;
            q.rope = nullptr;
        }
    }
    hipLaunchKernelGGL(kernel, dim3(8 * q.per_xcd), dim3(64 * kWaves), lds, s, q);
    MI355_LAUNCH_CHECK();
    if constexpr (FUSE) {
        if (q.ksplit > 1) {
            const int64_t groups = (int64_t)p.M * (p.N >> 7);
            const int grid = (int)((groups + 7) / 8 < 4096 ? (groups + 7) / 8 : 4096);
            hipLaunchKernelGGL(splitk_fused_reduce_kernel<EPI>, dim3(grid), dim3(256), 0, s, p);
            MI355_LAUNCH_CHECK();
            return 0;
        }
    }
    if (q.ksplit > 1 && EPI == MI355_EPI_ACCUM && q.rn.done) {
        hipLaunchKernelGGL(splitk_norm_kernel, dim3(p.M), dim3(1024), 0, s, q.part, q.ksplit, p.M, p.N, (float*)p.y, p.ldy, q.rn);
        MI355_LAUNCH_CHECK();
    } else if (q.ksplit > 1) {
        const int64_t n = (int64_t)p.M * (p.N >> 2);
        const int grid = (int)((n + 255) / 256 < 2048 ? (n + 255) / 256 : 2048);
        hipLaunchKernelGGL(splitk_reduce_kernel<EPI>, dim3(grid), dim3(256), 0, s, q.part, q.ksplit, p.M, p.N, p.y, p.y_dtype, p.ldy, p.relu2, p.limit,
                           p.bias);
        MI355_LAUNCH_CHECK();
    }
    return 0;
}
template <int EPI, bool PAIR, int FMT, int kWaves, int BM, bool FUSE, int GRP = 0, int TPW = kTPW, bool RUNS = false, bool ONCE = false>
int launch_deep(const GemmParams& p, hipStream_t s) {
    if constexpr (FMT == MI355_W_Q4 && GRP == 0 && BM <= 64 && !RUNS) {
        if (p.runs > 1) return launch_deep<EPI, PAIR, FMT, kWaves, BM, FUSE, GRP, TPW, true>(p, s);
    }
    if constexpr (!ONCE && (FMT == MI355_W_BF16 ? BM <= 64 : BM <= 48 && (GRP == 1 || BM >= 32))) {  // (int4 of one scale per row: fewer than 32 tokens are multiplied unit by unit, GRP 1)
        if (p.streamed && p.M <= BM) return launch_deep<EPI, PAIR, FMT, kWaves, BM, FUSE, GRP, TPW, RUNS, true>(p, s);
    }
    constexpr int kDepth = BM > 192 ? 2 : BM > kBM || (BM >= 96 && FMT == MI355_W_BF16) ? 3 : 4;
    constexpr int kLds = kRowAt<BM, FUSE, kDepth> + 3 * kWaves * TPW * 64 + (RUNS ? kMaxRuns * BM * 4 : 0) + (FMT == MI355_W_BF16 ? 256 : 0);
    static hipError_t attr_err = hipFuncSetAttribute((const void*)gemm_deep_kernel<EPI, PAIR, FMT, kWaves, BM, FUSE, kDepth, GRP, RUNS, TPW, ONCE>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr_err != hipSuccess) {
        mi355_set_error("hipFuncSetAttribute(gemm) failed: %s", hipGetErrorString(attr_err));
        return (int)attr_err;
    }
    return launch_blocks<EPI, PAIR, kWaves, BM, FUSE, TPW>(gemm_deep_kernel<EPI, PAIR, FMT, kWaves, BM, FUSE, kDepth, GRP, RUNS, TPW, ONCE>, kLds, p, s);
}
template <int EPI, bool PAIR, int kWaves, int BM, int GRP = 0, bool FUSE = false>
int launch_gemm_w(const GemmParams& p, hipStream_t s) {
    constexpr int kLdsW = kRowAt<BM, FUSE> + 3 * kWaves * kTPW * 64;
    static hipError_t attr_err = hipFuncSetAttribute((const void*)gemm_q4_kernel<EPI, PAIR, kWaves, BM, GRP, FUSE>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLdsW);
    if (attr_err != hipSuccess) {
        mi355_set_error("hipFuncSetAttribute(gemm) failed: %s", hipGetErrorString(attr_err));
        return (int)attr_err;
    }
    return launch_blocks<EPI, PAIR, kWaves, BM, FUSE, kTPW>(gemm_q4_kernel<EPI, PAIR, kWaves, BM, GRP, FUSE>, kLdsW, p, s);
}
// How a launch of one scale per row is cut: waves and tokens of a block, gemm_deep_kernel (or gemm_q4_kernel), K-slices
struct GemmCut {
    int waves, bm;
    bool deep;
    int ksplit;
    int tiles = kTPW;  // row tiles of a wave
};
// tuning override for sweeps: MI355_GEMM_FORCE="waves:bm:ksplit:deep", 0 = the rule's choice.  deep: 1 / 2 for gemm_deep_kernel / gemm_q4_kernel (the latter int4 only), of int4 3 for waves of
// one row tile (q4_narrow()) and 4 for blocks of 96 to 192 tokens x 8 waves (q4_whole(), grouped scales of whole units 96 and 160).  Where waves, tokens or 1 / 2 are given, the rest is
// q4_cut()'s, with 3 and 4 the rule's as a whole.  A cut that no kernel is instantiated for is ignored as a whole, a number of slices that does not fit by itself; blocks that only BF16 streams have need the kernel named (deep = 1)
struct GemmForce {
    int waves, bm, ksplit, deep;
};
GemmForce gemm_force() {
    // parsed ONCE per process (a change of the variable between mi355_linear_gemm_plan and the launch would desynchronise the share layout of
    // the fused chain)
    static const GemmForce f = [] {
        GemmForce g = {0, 0, 0, 0};
        if (const char* e = getenv("MI355_GEMM_FORCE")) sscanf(e, "%d:%d:%d:%d", &g.waves, &g.bm, &g.ksplit, &g.deep);
        return g;
    }();
    return f;
}
bool launch_gemm_has(const GemmCut& c, bool bf16, int kernel, bool grouped = false) {  // (what a sweep may force of the kernels of launch_gemm(); kernel: GemmForce::deep)
    if (c.tiles == 1) return !bf16 && c.waves == 4 && c.deep && (c.bm == 16 || c.bm == 32 || c.bm == 48 || c.bm == 64);
    if (kernel == 4) return !bf16 && c.waves == 8 && (c.bm == 96 || c.bm == 160 || (c.bm == 192 && !grouped));
    if (bf16 && kernel == 1 && ((c.waves == 4 && (c.bm == 96 || c.bm == kBM)) || (c.waves == 8 && (c.bm == 160 || c.bm == 192 || c.bm == 208 || c.bm == 256)))) return true;
    if (c.waves == 2 || c.waves == 3) return bf16 && c.deep && (c.bm == 16 || c.bm == 32 || c.bm == 64);
    if (c.waves == 4) return c.deep && (c.bm == 16 || c.bm == 32 || c.bm == 64 || (c.bm == 48 && !bf16));
    return c.waves == 8 && (c.bm == kBM || c.bm == 64) && (c.deep || (!bf16 && c.bm == kBM));
}
// blocks of `waves` waves and `bm` tokens
int gemm_blocks(int M, int N, bool pair, int waves, int bm, int tiles = kTPW) {
    const int rows = 16 * (pair ? waves * tiles / 2 : waves * tiles);
    return (N + rows - 1) / rows * ((M + bm - 1) / bm);
}
// bytes of the K-slices' partial sums
size_t gemm_part_bytes(int M, int N, bool pair, int ksplit) { return (size_t)ksplit * M * N * (pair ? 2 : 1) * 4; }
// (blocks of 48 tokens, int4: of eight products of 2048 to 13824 rows at 33 / 40 / 48 tokens 2-10 / 2-9 / 2-7 % less than blocks of 64, groups of 128 columns 3-9 / 3-8 /
// 3-7 % (N = 12288, K = 4096: 22.2 -> 20.9, 22.1 -> 21.0, 22.4 -> 21.3 us).  BF16, bound by the weights, the same either way)
int short_block(int M, bool bf16) { return M <= 16 ? 16 : M <= 32 ? 32 : M <= 48 && !bf16 ? 48 : 64; }

// Int4: up to 64 tokens, and what q4_narrow() and q4_whole() start from.  (Narrow SwiGLU pairs of up to 128 tokens are left behind: 5632 rows, K = 2048, 128 tokens 24.5 us against 17.4 in blocks of
// 4 waves.)
// Waves of a block: up to 64 tokens blocks of 128 rows x 4 waves: N = 4096 is 32 of them, which 4-5 K-slices bring to a workgroup for two CUs of three;
// 256-row blocks x 8 waves need twice the slices (37 tokens, N = K = 4096, with staging: 20.5 us against 22.7).  Longer prompts likewise while the 256-row
// blocks leave half of the CUs idle, except where the 128-row blocks of a launch without slices are one for 5/8 of the CUs (8 / 4 waves, with staging: N = K = 4096,
// 128 tokens 29.3 / 24.5 us, 512 38.9 / 32.0; N = 12288, 128 tokens 34.6 / 29.6; K = 11008, 300 tokens 57.5 / 64.0, 512 71.2 / 66.7).  The SwiGLU pair does
// not gain (128 tokens 36.5 / 39.4).
// Slices: as many as bring the launch to the workgroups wanted, none below 6 units, from the third on of blocks of 4 waves 4 (each is one run then, gemm_runs(): 40
// tokens, N = K = 4096, 15.8 us with 8 slices, 16.4 with 5; 2048, 12.5 with 4, 14.3 with 2; but N = 2816 pair, K = 1024, 12.5 with 2, 10.6 with 1).  Their sums, written and read again, take at most half the partial buffer,
// 16 MB: past that a slice costs more than the CUs that it fills (1 / 2 slices, 600 tokens, N = 4096: K = 4096 38.1 / 45.6 us, 11008 77 / 84; 120, N = 11008 pair 35.4 /
// 42.1).  Blocks of 4 waves stop at one workgroup per CU: a few more than 256 leave the chip to those few (37 rows, K = 11008, N = 4096: 28.4 / 26.7 / 25.6 /
// 24.7 with 4 / 5 / 6 / 8).
// Tokens: blocks of 128 x 256 rows with two workgroups per CU (gemm_q4_kernel) when a launch has a few of them per CU: 2048 tokens, c_fc1/c_fc2 271 us against
// 303 (gemm_deep_kernel, one workgroup per CU), c_attn 158 / 174.  Fewer: 64-token blocks, twice as many, of the deep kernel: 128 tokens, c_fc1/c_fc2 49.6 -> 39.9
// us, 777 tokens N = 4096 47.8 -> 42.1 us.  A launch of exactly one 128-token block per CU (N = 4096 at 2048 tokens) keeps those.
GemmCut q4_cut(int M, int N, int K, bool pair) {
    const int units = (K + 127) / 128, blocks8 = (N + 255) / 256 * ((M + 63) / 64);
    GemmCut cut = {M <= 64 || (!pair && (blocks8 <= 64 || (blocks8 >= 96 && blocks8 <= 128))) ? 4 : 8, short_block(M, false), true, 1};
    const int blocks = gemm_blocks(M, N, pair, cut.waves, 64), want = cut.waves == 8 ? 192 : 256, most = cut.waves == 8 ? 1 << 20 : 256;
    while (cut.ksplit < 8 && blocks * cut.ksplit < want && blocks * (cut.ksplit + 1) <= most && units >= (cut.waves == 4 && cut.ksplit > 1 ? 4 : 6) * (cut.ksplit + 1) &&
           gemm_part_bytes(M, N, pair, cut.ksplit + 1) <= kSplitBudget / 2)
        ++cut.ksplit;
    const int wide = gemm_blocks(M, N, pair, 8, kBM) * cut.ksplit;
    if (wide >= 384 || wide == 256) cut.bm = kBM, cut.deep = false;
    return cut;
}
// Int4: the units that one accumulator sums.  Levels enter as 128 + q: beside an activation 10^5 times the others a sum is 10^7 times its other terms, and every
// product of 32 columns costs it another rounding of that size.  So a sum ends behind 1 / cuts of K at the latest, cuts = 2, 4, 8 while 128-token blocks of 256 rows
// number less than 96 / cuts and a run keeps 4 units; a K-slice that is longer takes several runs, each with its own operand sum.  Error beside one activation of
// 2^17 (rms, in units of its product's last bit), N = K = 4096 / N = 4096, K = 11008 / N = 12288, K = 4096, a run per slice -> runs: 40 tokens 3.0 / 3.9 / 4.8 -> 2.6 /
// 3.8 / 4.8, 100 tokens 3.5 / 5.6 / 6.8 -> 2.6 / 3.5 / 4.8, 512 tokens 6.8 / 11.2 / 6.8 -> 4.8 / 7.5 / 6.7.  A second run takes a launch 0.5-0.7 us (a prompt of 37
// tokens, 7B: 2.48 -> 2.49 ms).  Runs of K / 8 for longer prompts too would cost them registers: 400 tokens 239 -> 268 us a layer.
void gemm_runs(int M, int N, int K, bool pair, const GemmCut& cut, int* runs, int* run_units) {
    const int units = (K + 127) / 128, longest = (units + cut.ksplit - 1) / cut.ksplit, blocks = gemm_blocks(M, N, pair, 8, kBM);
    int cuts = 1;
    while (cuts < 8 && blocks * cuts < 96 && units >= 8 * cuts) cuts *= 2;
    *runs = 1, *run_units = units;
    if (longest <= (units + cuts - 1) / cuts || !cut.deep || cut.bm > 64) return;  // (q4_whole() takes blocks of more than 64 tokens only where they need no runs)
    *run_units = units / cuts / 4 * 4;
    *runs = (longest + *run_units - 1) / *run_units;
}
// ... whether a launch holds the sums of its rows (the rules' cuts do: at most 8 runs, 21 sums), and how many units one is in this cut
bool gemm_sums_fit(int M, int N, int K, bool pair, const GemmCut& cut) {
    int runs, run_units;
    gemm_runs(M, N, K, pair, cut, &runs, &run_units);
    return runs <= kMaxRuns && cut.ksplit * runs <= kMaxSums;
}
int gemm_longest(int M, int N, int K, bool pair, const GemmCut& cut) {
    int runs, run_units;
    gemm_runs(M, N, K, pair, cut, &runs, &run_units);
    return runs > 1 ? run_units : ((K + 127) / 128 + cut.ksplit - 1) / cut.ksplit;
}
// Int4 products other than pairs, where blocks of 64 rows x 4 waves are one per CU at most: a wave of one row tile.  A wave alone on its SIMD is bound by what it issues (37 tokens: two row tiles take
// 0.45 us a unit, one 0.31 to 0.34, with all operands in the L2 caches as well, and no barrier 0.42), so half the rows per wave on idle CUs are worth more than K-slices, whose sums are a launch more:
// 37 tokens, N = 12288, K = 4096 20.6 us in two slices of 128-row blocks, 18.1 whole in 64-row blocks; N = K = 4096 16.2 in 8 slices, 15.4 in 4; 128 tokens, N = 6144, K = 2048 19.6 / 14.5.  The
// estimate: per unit of a slice `unit` us and `crowd` more when every CU has a block, `slices` and `bytes` for partial sums, fitted to 1422 launches (18 products of 1024 to 32000 rows, 32 to 300
// tokens, weights in no cache; 7 % off on average; those of 18 products again in profiles/product_cuts_int4.txt).  Where it takes these blocks or not: 0.96 / 0.95 / 0.94 / 0.93 times the time of 128-row blocks (32, to 48, to 64, more tokens), 3 % slower at worst but for one (72 tokens,
// N = 6656, K = 17920 in two slices 5 %).
// In the chain, whose blocks add up shares first and whose sums of slices write the next ones, whole rows only (37 tokens, 7B: c_attn 12.8 + 4.2 us for the sum of its slices -> 15.9; attn.c_proj in 4
// narrow slices 8.4 + 4.2, in 8 wide ones 7.8 + 4.4).  No accumulator sums more than in the cut that they replace: N = 1024, K = 3584 in 4 slices of 7 units for 7 of 4 rounds beside an activation of
// 2^17 by 2.1 last bits rms for 1.7.
void q4_narrow(int M, int N, int K, bool pair, bool chain, GemmCut* cut) {
    struct Cost {
        float start, wide, wide_crowd, unit, crowd, slices, bytes;
    };
    static constexpr Cost costs[] = {{-0.476f, 0.369f, 0.24f, 0.288f, 0.148f, 3.485f, 1.2e6f},
                                     {-0.67f, 0.451f, 0.158f, 0.333f, 0.116f, 3.491f, 1.167e6f},
                                     {-0.796f, 0.539f, 0.073f, 0.383f, 0.083f, 3.592f, 1.153e6f},
                                     {-0.872f, 0.531f, 0.027f, 0.416f, -0.021f, 3.362f, 1.555e6f}};
    const int units = (K + 127) / 128, wide = gemm_blocks(M, N, false, 4, cut->bm) * cut->ksplit;
    if (pair || cut->waves != 4 || !cut->deep || wide > 256) return;
    const Cost& c = costs[M <= 32 ? 0 : M <= 48 ? 1 : M <= 64 ? 2 : 3];
    auto slices = [&](int ks) { return ks == 1 ? 0.f : c.slices + (float)gemm_part_bytes(M, N, false, ks) / c.bytes; };
    float best = (float)((units + cut->ksplit - 1) / cut->ksplit) * (c.wide + c.wide_crowd * (float)wide / 256.f) + slices(cut->ksplit);
    const int bm = cut->bm, blocks = gemm_blocks(M, N, false, 4, bm, 1), most = gemm_longest(M, N, K, false, *cut);
    for (int ks = 1; ks <= (chain ? 1 : 8) && blocks * ks <= 256 && (ks == 1 || (units >= 2 * ks && gemm_part_bytes(M, N, false, ks) <= kSplitBudget / 2)); ++ks) {
        const GemmCut narrow = {4, bm, true, ks, 1};
        int runs, run_units;
        gemm_runs(M, N, K, false, narrow, &runs, &run_units);
        const float us = c.start + (float)((units + ks - 1) / ks) * (c.unit + c.crowd * (float)(blocks * ks) / 256.f) + slices(ks);
        if (us < best && runs <= kMaxRuns && ks * runs <= kMaxSplit && gemm_longest(M, N, K, false, narrow) <= most) best = us, *cut = narrow;
    }
}
// Int4, from 65 tokens on: whole rows in blocks of 64, 96, 160 or 192 tokens x 8 waves where an estimate takes them for 3 % faster than q4_cut()'s and q4_narrow()'s cut and no accumulator sums
// more than there; against two workgroups per CU, whose estimate is the least certain, for 7 %, and no blocks of 64 (2048 tokens, N = K = 4096 64 us, in those 66).  Rows of up to 16 units 14 %: two workgroups of a CU write one's results beside the other's products, which
// is the more of a launch the shorter its rows are (K = 2048, two per CU / one: N = 32000, 1195 tokens 139 us / 146, 1518 167 / 172).  Blocks of 64 and 128 tokens
// leave the rounds of the chip two sizes to fit: 777 tokens, N = 12288, K = 4096, 624 blocks of 64 83.6 us, 240 of 160 67.2; the N = 11008 pair 131 / 112; 450, N = 19968, K = 6656 125 / 98 (160);
// 130, the N = 11008 pair, 258 blocks of 64 51.2, 172 of 96 42.6; 1500, N = 4096, K = 11008 136 / 114 (96); 384 of the N = 13824 pair, K = 5120 94.7 / 82.7 (192).  The estimate is a start and the
// rounds one behind the other, as in bf16_cut_long(), fitted to 3000 launches (profiles/product_cuts_int4.txt: 22 products of 1024 to 24576 rows, 72 to 2048 tokens; 3 to 5 % off on average): of 506 launches 169 take
// other blocks than before these and q4_narrow(), 0.87 times as long, none more than 0.8 % longer, and all together 0.6 % behind the best of each; of 533 between and beside them (N = 32000 too) three are 2 % longer.  Whole prompts of 72 to 2048 tokens, widths 2048 to 6656, one scale per row or groups
// of 128 columns: 0.965 times as long on average, 0.89 at best, the rest within the noise.
void q4_whole(int M, int N, int K, bool pair, GemmCut* cut) {
    struct Kind {
        int waves, bm, tiles;
        float start, unit, crowd, slices, bytes;  // (the last two: of the sums of K-slices)
    };
    static constexpr Kind whole[] = {{8, 64, 2, 10.63f, 0.715f, 0.054f, 4.06f, 2.86e6f}, {8, 96, 2, 11.03f, 0.981f, 0.126f}, {8, 160, 2, 12.34f, 1.37f, 0.252f}, {8, 192, 2, 13.4f, 1.55f, 0.327f}};
    static constexpr Kind narrow = {4, 64, 1, 8.35f, 0.261f, 0.154f, 1.33f, 0.77e6f}, half = {4, 64, 2, 10.42f, 0.392f, 0.148f, 6.15f, 5.75e6f}, two_per_cu = {8, kBM, 2, 18.84f, 0.705f, 0.647f, 2.2f, 2.5e6f};
    if (M <= 64) return;
    const int units = (K + 127) / 128;
    auto longest = [&](const GemmCut& c) {  // units of a sum (as good as none where there are more runs than a launch takes)
        int runs, run_units;
        gemm_runs(M, N, K, pair, c, &runs, &run_units);
        return runs > kMaxRuns || c.ksplit * runs > kMaxSplit ? units + 1 : runs > 1 ? run_units : (units + c.ksplit - 1) / c.ksplit;
    };
    auto estimate = [&](const Kind& k, int ks) {
        const int blocks = gemm_blocks(M, N, pair, k.waves, k.bm, k.tiles) * ks;
        auto round = [&](int of) { return of == 0 ? 0.f : (float)((units + ks - 1) / ks) * (k.unit + k.crowd * (float)of / 256.f); };
        return k.start + (float)(blocks / 256) * round(256) + round(blocks % 256) + (ks == 1 ? 0.f : k.slices + (float)gemm_part_bytes(M, N, pair, ks) / k.bytes);
    };
    const int most = longest(*cut);
    const bool crowded = cut->bm == kBM;
    float best = (!crowded ? 0.97f : units > 16 ? 0.93f : 0.86f) * estimate(crowded ? two_per_cu : cut->tiles == 1 ? narrow : cut->waves == 4 ? half : whole[0], cut->ksplit);
    for (const Kind& k : whole) {
        if (crowded && k.bm == 64) continue;
        const GemmCut c = {k.waves, k.bm, true, 1};
        const float us = estimate(k, 1);
        if (us < best && longest(c) <= most) best = us, *cut = c;
    }
}
// Up to 64 tokens, outside the fused chain (whose shares are 64 or 128 rows), where blocks of 4 waves do not fill the chip: blocks of 2, 3 or 4 waves (64, 96, 128 rows).  A CU
// asks for no more than its memory pipeline holds, so 129 blocks of 128 rows leave half of what HBM gives, and a slice that would fill the other CUs costs a launch; smaller
// blocks cost their activations again.  16 tokens, 4 / 3 / 2 waves without slices: N = 16512, K = 4096 29.7 / 26.1 / 35.0 us (129, 172, 258 blocks), 12416 33.2 (24.9 in two
// slices) / 27.4 / 21.4; K = 16384, N = 4096 28.8 in 4-wave blocks x 6 slices, 27.9 in 2-wave blocks x 3.  The estimate is the rounds of the chip, each unit of one `unit` us, `unit_wave`
// more for each wave of a block and `crowd` more when every CU has one, `wave` for each wave's start, and a launch for the slices.  Slices go down to 2 units where a row is 4 to 31 of them (385 to
// 3968 columns): a short product is a wait for memory that more blocks share out (N = K = 2048, weights from HBM, 16 / 24 / 32 tokens 8.2 / 9.3 / 9.6 us whole in 32 blocks, 6.8 / 7.5 / 7.8 in 8 slices).
// Longer rows have units enough (N = 2048, K = 8448, 16 tokens 11.1 us in 6 slices, 11.7 in 8; N = 5120, K = 20736 36.7 in 2 waves x 3, 37.4 in 4 x 6), up to 8 tokens (N = 4672, K = 3456, 2 tokens
// 10.6 us in 3 slices, 11.3 in 7) and in pairs, whose sums are twice as long (25 products at 24 to 64 tokens 0.99-1.00 on average, the worst 1.13), more sums cost what they give: there slices keep 4 units.
// Weights that a cache holds (not MI355_LF_STREAMED) are asked for faster, so fewer blocks fill the chip: up to 32 tokens constants of their own (110 MB of copies, N = 5856, K = 3456, 16 tokens
// 8.9 us in blocks of 2 waves, whole, 11.5 in 4 slices of blocks of 3).  Times of every cut: profiles/product_cuts_bf16_few.txt.  From HBM, 52 products of 1024 to 32000 rows and 512 to 20736 columns: up to 32 tokens 0.6 % behind the
// fastest cut on average, 6 % at most, 40 and 64 tokens 1.1 % (9 %); from a cache, 56 products of 512 to 12288 rows and 512 to 3968 columns, 9 and 16 tokens 0.4 % (7 %), 24 and 32 0.7 % (9 %).
GemmCut bf16_cut_few(int M, int N, int K, bool pair, bool sliced, bool streamed) {
    struct Cost {
        float wave, unit, unit_wave, crowd, slices, bytes;
    };
    static constexpr Cost costs[] = {{0.f, 0.007f, 0.066f, 0.193f, 1.5f, 2.7e6f}, {0.25f, 0.21f, 0.023f, 0.041f, 0.3f, 2.3e6f},               // slices of 4 units: up to 32 tokens, up to 64
                                     {0.494f, 0.0935f, 0.0402f, 0.17f, 1.56f, 2.33e6f}, {0.607f, 0.045f, 0.0371f, 0.0182f, 0.861f, 4.79e6f},  // of 2, from HBM: up to 16, up to 32
                                     {0.516f, 0.066f, 0.0195f, 0.481f, 1.85f, 6.21e6f}, {0.57f, 0.0732f, 0.0415f, 0.153f, 1.36f, 1.44e6f},    // of 2, from a cache
                                     {0.256f, 0.207f, 0.025f, 0.0058f, 0.576f, 2.31e6f}};                                                     // of 2, up to 64
    const int units = (K + 127) / 128;
    const bool shorter = !pair && M > 8 && units >= 4 && units < 32;
    const int least = shorter ? 2 : 4, line = !shorter ? (M > 32) : M > 32 ? 6 : (streamed ? 2 : 4) + (M > 16);
    const Cost& c = costs[line];
    GemmCut cut = {4, short_block(M, true), true, 1};
    float best = 0.f;
    for (int waves = 2; waves <= 4; waves += sliced ? 2 : 1)  // (operand slices start at multiples of 256 rows, which blocks of 96 do not divide)
        for (int ks = 1; ks <= 8 && (ks == 1 || (units >= least * ks && gemm_part_bytes(M, N, pair, ks) <= kSplitBudget / 2)); ++ks) {
            const int blocks = gemm_blocks(M, N, pair, waves, cut.bm) * ks;
            auto round = [&](int of) { return of == 0 ? 0.f : (float)((units + ks - 1) / ks) * (c.unit + (float)waves * (c.unit_wave + c.crowd * (float)of / 256.f)); };
            const float us = c.wave * (float)waves + (float)(blocks / 256) * round(256) + round(blocks % 256) +
                             (ks == 1 ? 0.f : c.slices + (float)gemm_part_bytes(M, N, pair, ks) / c.bytes);
            if (best == 0.f || us < best) best = us, cut.waves = waves, cut.ksplit = ks;
        }
    return cut;
}
// Up to 64 tokens in the chain, blocks of 4 waves no more than the CUs: as many slices as bring them to three quarters of the CUs and none to a few more than all (16 rows,
// N = 16512, K = 4096, 129 blocks: 30.1 / 38.8 / 32.2 / 36.3 us with 1 / 2 / 3 / 4; K = 11008, N = 4096, 32 blocks 24.2 / 21.9 / 21.3 / 21.9 / 23.2 with 4 / 5 / 6 / 8 / 13).
GemmCut bf16_cut_few_chained(int M, int N, int K, bool pair) {
    const int units = (K + 127) / 128, few = gemm_blocks(M, N, pair, 4, 64);
    GemmCut cut = {4, short_block(M, true), true, 1};
    while (cut.ksplit < kMaxSplit && few * cut.ksplit < 192 && few * (cut.ksplit + 1) <= 256 && units >= 4 * (cut.ksplit + 1) &&
           gemm_part_bytes(M, N, pair, cut.ksplit + 1) <= kSplitBudget / 2)
        ++cut.ksplit;
    return cut;
}
// Up to 64 tokens, blocks of 4 waves more than the CUs: the weights bound them, 6.6 TB/s behind 4.3 us, beside the busiest CU's units (48 tokens of the N = 17920 pair, K = 6656: 104 /
// 95 us with 4 / 8 waves).
GemmCut bf16_cut_many(int M, int N, int K, bool pair) {
    struct Kind {
        int waves, bm;
        float start, unit;
    };
    const int units = (K + 127) / 128, bm = short_block(M, true);
    const Kind kinds[] = {{4, bm, bm == 16 ? 0.9f : bm == 32 ? 1.3f : 3.0f, bm == 16 ? 0.67f : bm == 32 ? 0.71f : 0.75f}, {8, 64, 3.4f, 1.23f}};
    const float bytes = 2.f * N * K * (pair ? 2 : 1) + 2.f * M * K + 4.f * M * N, hbm = 4.3f + bytes / 6.6e6f;
    GemmCut cut = {4, bm, true, 1};
    float best = 0.f;
    for (const Kind& k : kinds)
        for (int ks = 1; ks <= kMaxSplit && (ks == 1 || (units >= 4 * ks && gemm_part_bytes(M, N, pair, ks) <= kSplitBudget * 3 / 4)); ++ks) {
            const float work = k.start + (float)((gemm_blocks(M, N, pair, k.waves, k.bm) * ks + 255) / 256 * ((units + ks - 1) / ks)) * k.unit;
            const float us = sqrtf(work * work + hbm * hbm) + (ks == 1 ? 0.f : 1.6f + (float)gemm_part_bytes(M, N, pair, ks) / 2.3e6f);
            if (best == 0.f || us < best) best = us, cut = {k.waves, k.bm, true, ks};
        }
    return cut;
}
// From 65 tokens on: what an estimate takes for the fastest, a start and the rounds of the chip one behind the other, each the units of a slice, `unit` us when a CU is alone with its
// block and `crowd` more when every CU has one, whatever of a block is padding; slices cost their sums' way to memory and back, no less than a launch.  Blocks of 192 and 256 tokens x 256
// rows ask for 75 and 64 KB per 8.4 MFLOP instead of the 96 of 128 x 256, and give the rounds more sizes to fit: 2048 tokens, N = 16512, K = 4096, 4.1 rounds of 128 tokens 278 us, 2.8 of
// 192 234; N = 6208, 1.6 of 128 108, 0.8 of 256 94; 777 tokens, N = 12288, 1.3 of 128 105, 0.9 of 192 79; N = 4096, K = 11008 in 128 x 128 85 (64 x 256: 104).  The constants are
// those whose choice is best over 1078 launches (41 products of 512 to 32000 rows, 65 to 2048 tokens; those below 20 MB with their weights in the 256-MB cache and without, the others
// without: profiles/product_cuts_bf16.txt): 0.8 % behind the fastest of 25 000 cuts on average, 2.7 % at the 90th percentile.  Fitted to rows of 2048 columns and more, without
// a launch as the least that slices cost, 1.6 % and 5.4 %: short rows were cut (512 tokens, N = K = 2048 16.1 us in two slices, 12.7 whole; 96 of the N = 2816 pair, K = 1024 11.6, 8.2).
// Blocks of 160 and 208 tokens came later, their constants fitted to 270 launches without slices (15 products, 129 to 2048 tokens): whole rows only, and where the estimate takes them for 4 %
// faster than the others.  288 of 355 launches (40 products) that they would take by the lower estimate are 0.94 times as long then, two to six of them, run by run, more than 2 % longer, 5 % at most (777 tokens, N = 15360, K = 5120
// in 256 / 208 tokens 123 / 107 us; N = 12288, K = 4096 in 192 / 160 75 / 69, the N = 11008 pair 138 / 128; 2048, N = 12416 in 256 / 208 199 / 179).  The 32 within 4 % are 1.3 % faster in the other blocks, up to
// 10 % (2048 tokens, N = 32000 in 208 / 256: K = 2048 282 / 258 us, 4096 474 / 450; 1772 of the N = 2816 pair, K = 1024 in 208 / 192 26.8 / 25.0), the 35 in slices 0.4 %, up to 9 % (129 tokens, N = 4096,
// K = 16512 11 slices of 160 tokens 46.3 us, 4 of 96 42.4; 146, N = 8192, K = 22016 100.3 / 96.0): profiles/product_cuts_bf16.txt.
GemmCut bf16_cut_long(int M, int N, int K, bool pair) {
    struct Kind {
        int waves, bm;
        float start, unit, crowd;
    };
    static constexpr Kind kinds[] = {{4, 64, 2.744f, 0.518f, 0.181f},  {4, 96, 4.059f, 0.484f, 0.333f}, {4, kBM, 2.751f, 0.78f, 0.272f}, {8, 64, 6.209f, 0.684f, 0.474f},
                                     {8, kBM, 8.323f, 0.926f, 0.424f}, {8, 192, 11.38f, 1.231f, 0.501f}, {8, 256, 9.51f, 1.344f, 1.146f}};
    static constexpr Kind whole[] = {{8, 160, 8.129f, 1.217f, 0.283f}, {8, 208, 8.519f, 1.703f, 0.271f}};
    const int units = (K + 127) / 128;
    auto estimate = [&](const Kind& k, int ks) {
        const int blocks = gemm_blocks(M, N, pair, k.waves, k.bm) * ks;
        auto round = [&](int of) { return of == 0 ? 0.f : (float)((units + ks - 1) / ks) * (k.unit + k.crowd * (float)of / 256.f); };
        return k.start + (float)(blocks / 256) * round(256) + round(blocks % 256);
    };
    GemmCut cut = {4, 64, true, 1};
    float best = 0.f;
    for (const Kind& k : kinds)
        for (int ks = 1; ks <= kMaxSplit && (ks == 1 || (units >= 4 * ks && gemm_part_bytes(M, N, pair, ks) <= kSplitBudget * 3 / 4)); ++ks) {
            float us = estimate(k, ks);
            if (ks > 1) us += fmaxf(0.976f + (float)gemm_part_bytes(M, N, pair, ks) / 2.486e6f, 2.17f);
            if (best == 0.f || us < best) best = us, cut = {k.waves, k.bm, true, ks};
        }
    best *= 0.96f;
    for (const Kind& k : whole)
        if (const float us = estimate(k, 1); us < best) best = us, cut = {k.waves, k.bm, true, 1};
    return cut;
}
GemmCut bf16_cut(int M, int N, int K, bool pair, bool chain, bool sliced, bool streamed) {
    if (M > 64) return bf16_cut_long(M, N, K, pair);
    if (gemm_blocks(M, N, pair, 4, 64) > 256) return bf16_cut_many(M, N, K, pair);
    return chain ? bf16_cut_few_chained(M, N, K, pair) : bf16_cut_few(M, N, K, pair, sliced, streamed);
}
// chain: a launch of the fused prompt chain (gemm_fuse.h); sliced: a launch of operand slices; streamed: weights that come from HBM
GemmCut gemm_cut(int M, int N, int K, bool pair, bool bf16, bool chain, bool sliced, bool streamed) {
    const GemmForce fo = gemm_force();
    const GemmCut first = bf16 ? bf16_cut(M, N, K, pair, chain, sliced, streamed) : q4_cut(M, N, K, pair);
    GemmCut cut = first;
    if (!bf16) q4_narrow(M, N, K, pair, chain, &cut), q4_whole(M, N, K, pair, &cut);
    const GemmCut& from = fo.deep >= 3 || (fo.waves == 0 && fo.bm == 0 && fo.deep == 0) ? cut : first;
    const GemmCut forced = {fo.waves ? fo.waves : from.waves, fo.bm ? fo.bm : from.bm, fo.deep ? fo.deep != 2 : from.deep, from.ksplit, fo.deep == 3 && !pair ? 1 : fo.deep ? kTPW : from.tiles};
    if (launch_gemm_has(forced, bf16, fo.deep) && (!chain || forced.waves >= 4) && (!sliced || forced.waves != 3)) cut = forced;
    if (fo.ksplit >= 1 && fo.ksplit <= kMaxSplit && (K + 127) / 128 >= fo.ksplit && gemm_part_bytes(M, N, pair, fo.ksplit) <= (bf16 ? kSplitBudget : kSplitBudget / 2)) {
        GemmCut sliced_so = cut;
        sliced_so.ksplit = fo.ksplit;
        if (bf16 || gemm_sums_fit(M, N, K, pair, sliced_so)) cut = sliced_so;
    }
    return cut;
}
// Grouped scales, groups of whole units.  Blocks of 256 rows x 64 tokens and of 256 x 128 fill a CU alone, two of 128 x 64 share one; per round of the chip
// they take 1 : 1.75 : 1, a round of at most one 128 x 64 block per CU 0.75 (N = 4096, K = 11008: 256 x 64 blocks 104 us at 512 tokens, 106 at 777, 108 at 1000;
// 256 x 128 165 / 168 / 169; 128 x 64 78 / 106 / 114): the fewest.  1000 tokens, 7B: 235 / 101 / 137 us for c_fc1 / c_fc2, c_proj on average, c_attn with blocks
// of 64 x 128 one unit ahead -> 185 / 75 / 120.
// Blocks of 96 or 160 tokens x 8 waves where an estimate as in q4_whole(), the slices given, takes them for 2 % faster: 777 tokens, N = 12288, K = 4096 104 us in blocks of 64, 89 of 160; 130, the
// N = 11008 pair 65.9 / 56.5 (96); 1500, N = 4096, K = 11008 170 / 145 (96); 1000, N = K = 4096 48 in blocks of 128 rows x 64 as before (96: 59).  Of 506 launches 104 take them, 0.90 times as long as before, none more
// than 1 % longer.  (Blocks of 192 tokens would spill; those of 160 hold 24 to 36 bytes a lane of what is made once outside the registers.)
GemmCut gemm_cut_grouped(int n_tiles, int M, bool pair, int units, int ksplit) {
    struct Kind {
        int waves, bm;
        float start, unit, crowd;
        int round;  // blocks that the chip holds
    };
    static constexpr Kind kinds[] = {{4, 64, 12.67f, 0.481f, 0.592f, 512}, {8, 64, 13.47f, 0.868f, 0.226f, 256}, {8, kBM, 16.17f, 1.132f, 0.711f, 256}, {8, 96, 14.75f, 1.255f, 0.21f, 256},
                                     {8, 160, 17.46f, 1.939f, 0.237f, 256}};
    const GemmForce fo = gemm_force();
    GemmCut sh = {4, short_block(M, false), true, ksplit};
    if (M > 64) {
        auto blocks = [&](int waves, int bm) {
            const int per_block = pair ? waves * kTPW / 2 : waves * kTPW;
            return (n_tiles + per_block - 1) / per_block * ksplit * ((M + bm - 1) / bm);
        };
        const int half = blocks(4, 64), full = blocks(8, 64), wide = blocks(8, 128);
        const int t_half = half / 512 * 4 + (half % 512 == 0 ? 0 : half % 512 <= 256 ? 3 : 4), t_full = (full + 255) / 256 * 4, t_wide = (wide + 255) / 256 * 7;
        if (t_wide < t_half && t_wide <= t_full)
            sh = {8, 128, true, ksplit};
        else if (t_full <= t_half)
            sh.waves = 8;
        auto estimate = [&](const Kind& k) {
            const int of = blocks(k.waves, k.bm), rest = of % k.round;
            const float all = k.unit + k.crowd, part = rest == 0 ? 0.f : k.unit + k.crowd * (float)rest / (float)k.round;
            return k.start + (float)((units + ksplit - 1) / ksplit) * ((float)(of / k.round) * all + part);
        };
        float best = 0.98f * estimate(kinds[sh.bm == kBM ? 2 : sh.waves == 8]);
        for (int i = 3; i < 5; ++i)
            if (const float us = estimate(kinds[i]); us < best) best = us, sh.waves = kinds[i].waves, sh.bm = kinds[i].bm;
    }
    const GemmCut forced = {fo.waves ? fo.waves : sh.waves, fo.bm ? fo.bm : sh.bm, true, ksplit};
    return launch_gemm_has(forced, false, fo.deep == 4 ? 4 : 0, true) ? forced : sh;
}
template <int EPI, bool PAIR, int FMT, bool FUSE>
int launch_gemm(const GemmParams& p, hipStream_t s) {
    const GemmCut sh = gemm_cut(p.M, p.N, p.K, PAIR, FMT == MI355_W_BF16, FUSE, p.slice_blocks != 0, p.streamed);
    if constexpr (FMT == MI355_W_BF16 && !FUSE) {
        if (sh.waves == 3) {
            if (sh.bm == 64) return launch_deep<EPI, PAIR, FMT, 3, 64, FUSE>(p, s);
            return sh.bm == 16 ? launch_deep<EPI, PAIR, FMT, 3, 16, FUSE>(p, s) : launch_deep<EPI, PAIR, FMT, 3, 32, FUSE>(p, s);
        }
        if (sh.waves == 2) {
            if (sh.bm == 64) return launch_deep<EPI, PAIR, FMT, 2, 64, FUSE>(p, s);
            return sh.bm == 16 ? launch_deep<EPI, PAIR, FMT, 2, 16, FUSE>(p, s) : launch_deep<EPI, PAIR, FMT, 2, 32, FUSE>(p, s);
        }
    }
    if constexpr (FMT == MI355_W_Q4 && !PAIR) {
        if (sh.tiles == 1) {
            if (sh.bm == 16) return launch_deep<EPI, PAIR, FMT, 4, 16, FUSE, 0, 1>(p, s);
            if (sh.bm == 32) return launch_deep<EPI, PAIR, FMT, 4, 32, FUSE, 0, 1>(p, s);
            if (sh.bm == 48) return launch_deep<EPI, PAIR, FMT, 4, 48, FUSE, 0, 1>(p, s);
            return launch_deep<EPI, PAIR, FMT, 4, 64, FUSE, 0, 1>(p, s);
        }
    }
    if (sh.waves == 4) {
        if (sh.bm == 16) return launch_deep<EPI, PAIR, FMT, 4, 16, FUSE>(p, s);
        if (sh.bm == 32) return launch_deep<EPI, PAIR, FMT, 4, 32, FUSE>(p, s);
        if constexpr (FMT == MI355_W_Q4) {
            if (sh.bm == 48) return launch_deep<EPI, PAIR, FMT, 4, 48, FUSE>(p, s);
        }
        if constexpr (FMT == MI355_W_BF16) {
            if (sh.bm == 96) return launch_deep<EPI, PAIR, FMT, 4, 96, FUSE>(p, s);
            if (sh.bm == kBM) return launch_deep<EPI, PAIR, FMT, 4, kBM, FUSE>(p, s);
        }
        return launch_deep<EPI, PAIR, FMT, 4, 64, FUSE>(p, s);
    }
    if (sh.bm == 64) return launch_deep<EPI, PAIR, FMT, 8, 64, FUSE>(p, s);
    if constexpr (FMT == MI355_W_BF16) {
        if (sh.bm == 160) return launch_deep<EPI, PAIR, FMT, 8, 160, FUSE>(p, s);
        if (sh.bm == 192) return launch_deep<EPI, PAIR, FMT, 8, 192, FUSE>(p, s);
        if (sh.bm == 208) return launch_deep<EPI, PAIR, FMT, 8, 208, FUSE>(p, s);
        if (sh.bm == 256) return launch_deep<EPI, PAIR, FMT, 8, 256, FUSE>(p, s);
        return launch_deep<EPI, PAIR, FMT, 8, kBM, FUSE>(p, s);
    } else {
        if (sh.bm == 96) return launch_deep<EPI, PAIR, FMT, 8, 96, FUSE>(p, s);
        if (sh.bm == 160) return launch_deep<EPI, PAIR, FMT, 8, 160, FUSE>(p, s);
        if (sh.bm == 192) return launch_deep<EPI, PAIR, FMT, 8, 192, FUSE>(p, s);
        if (sh.deep) return launch_deep<EPI, PAIR, FMT, 8, kBM, FUSE>(p, s);
        return launch_gemm_w<EPI, PAIR, 8, kBM, 0, FUSE>(p, s);
    }
}
// grouped scales.  Groups of 32 or 64 columns: blocks of 64 tokens x 4 waves (the second accumulator set costs the registers of more tokens or waves).
template <int EPI, bool PAIR>
int launch_gemm_subgroups(const GemmParams& p, hipStream_t s) {
    const int per_block8 = PAIR ? 8 * kTPW / 2 : 8 * kTPW;
    const int blocks8 = ((p.n_tiles + per_block8 - 1) / per_block8) * ((p.M + 63) / 64);
    if (p.ksplit > 1 || blocks8 >= 128) return launch_gemm_w<EPI, PAIR, 4, 64, 2>(p, s);
    if (blocks8 * 4 >= 128) return launch_gemm_w<EPI, PAIR, 2, 64, 2>(p, s);
    return launch_gemm_w<EPI, PAIR, 1, 64, 2>(p, s);
}
template <int EPI, bool PAIR, bool FUSE>
int launch_gemm_grouped(const GemmParams& p, bool subgroups, hipStream_t s) {
    if constexpr (!FUSE) {
        if (subgroups) return launch_gemm_subgroups<EPI, PAIR>(p, s);
    }
    const GemmCut sh = gemm_cut_grouped(p.n_tiles, p.M, PAIR, (p.K + 127) / 128, p.ksplit);
    if (sh.waves == 4) {
        if (sh.bm == 16) return launch_deep<EPI, PAIR, MI355_W_Q4, 4, 16, FUSE, 1>(p, s);
        if (sh.bm == 32) return launch_deep<EPI, PAIR, MI355_W_Q4, 4, 32, FUSE, 1>(p, s);
        if (sh.bm == 48) return launch_deep<EPI, PAIR, MI355_W_Q4, 4, 48, FUSE, 1>(p, s);
        return launch_deep<EPI, PAIR, MI355_W_Q4, 4, 64, FUSE, 1>(p, s);
    }
    if (sh.bm == 64) return launch_deep<EPI, PAIR, MI355_W_Q4, 8, 64, FUSE, 1>(p, s);
    if (sh.bm == 96) return launch_deep<EPI, PAIR, MI355_W_Q4, 8, 96, FUSE, 1>(p, s);
    if (sh.bm == 160) return launch_deep<EPI, PAIR, MI355_W_Q4, 8, 160, FUSE, 1>(p, s);
    return launch_deep<EPI, PAIR, MI355_W_Q4, 8, kBM, FUSE, 1>(p, s);
}
template <bool FUSE>
int launch_gemm_grouped_epi(const GemmParams& p, int epi, bool subgroups, hipStream_t s) {
    if (epi == MI355_EPI_SWIGLU) return launch_gemm_grouped<MI355_EPI_SWIGLU, true, FUSE>(p, subgroups, s);
    if (epi == MI355_EPI_ACCUM) return launch_gemm_grouped<MI355_EPI_ACCUM, false, FUSE>(p, subgroups, s);
    return launch_gemm_grouped<MI355_EPI_STORE, false, FUSE>(p, subgroups, s);
}
template <int FMT, bool FUSE>
int launch_gemm_epi(const GemmParams& p, int epi, hipStream_t s) {
    if (epi == MI355_EPI_SWIGLU) return launch_gemm<MI355_EPI_SWIGLU, true, FMT, FUSE>(p, s);
    if constexpr (FMT == MI355_W_BF16 && !FUSE) {
        if (epi == MI355_EPI_GEGLU) return launch_gemm<MI355_EPI_GEGLU, true, FMT, FUSE>(p, s);
        if (epi == MI355_EPI_CLAMPGLU) return launch_gemm<MI355_EPI_CLAMPGLU, true, FMT, FUSE>(p, s);
    }
    if (epi == MI355_EPI_ACCUM) return launch_gemm<MI355_EPI_ACCUM, false, FMT, FUSE>(p, s);
    return launch_gemm<MI355_EPI_STORE, false, FMT, FUSE>(p, s);
}

// floats from the 1/rms of the staged rows to their operand sums per unit
size_t unit_sums_at(int M) { return (size_t)M * (1 + kMaxSums); }

}  // namespace

extern "C" size_t mi355_linear_gemm_workspace_bytes(int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    const size_t kp = ((size_t)K + 127) / 128 * 128;
    // staged operands, 1/rms, per-slice operand sums, operand sums per unit, split-K partials (used when a launch would be a few dozen blocks)
    // ... and, at the very end, the partial sums of the fused prompt chain (gemm_fuse.h)
    return (size_t)M * kp * 2 + unit_sums_at(M) * 4 + (size_t)M * (kp / 128) * 4 + 256 + kSplitBudget + kFuseScratch;
}

namespace {
struct TableBytes {
    size_t tables, sums;  // [n_groups + 1][R][tab_ld] dwords; operand sums per group
};
TableBytes table_bytes(int M, int N, int R, int n_groups) { return {((size_t)(n_groups + 1) * R * ((N + 15) / 16 * 16) * 4 + 15) & ~(size_t)15, (size_t)n_groups * M * 4}; }
}  // namespace
bool mi355_linear_gemm_tables_fit(int M, int N, int K, int R, int group_cols) {
    const TableBytes t = table_bytes(M, N, R, (K + group_cols - 1) / group_cols);
    return t.tables + t.sums <= kSplitBudget;
}

size_t mi355_linear_gemm_fuse_scratch_bytes() { return kFuseScratch; }

extern "C" int mi355_linear_gemm(const mi355_linear_args* a, void* workspace, size_t workspace_bytes,
                                 mi355_stream_t stream) {
    return mi355_linear_gemm_fused(a, nullptr, workspace, workspace_bytes, stream);
}

namespace {
// K-slices of grouped scales: blocks of 8 row tiles x 64 tokens, doubled to 256 by slices of at least 4 cuts (groups; units where a group holds several: a slice may end
// within a group, whose products are scaled unit by unit).  Partial sums in the first half of the region, the tables in the second
int grouped_split(int M, int N, int K, bool pair, int group_cols) {
    const int rows_per_block = pair ? 16 * 4 * kTPW / 2 : 16 * 4 * kTPW, n_groups = (K + group_cols - 1) / group_cols;
    const int blocks = ((N + rows_per_block - 1) / rows_per_block) * ((M + 63) / 64), cuts = group_cols >= 128 ? n_groups : (K + 127) / 128;
    const TableBytes t = table_bytes(M, N, pair ? 2 : 1, n_groups);
    int ksplit = 1;
    while (ksplit < kMaxSplit && blocks * ksplit < 256 && cuts >= 8 * ksplit && t.tables + t.sums <= kSplitBudget / 2 &&
           gemm_part_bytes(M, N, pair, 2 * ksplit) <= kSplitBudget / 2)
        ksplit *= 2;
    return ksplit;
}
void plan_shares(const GemmCut& cut, int N, bool pair, int* ksplit, int* shares, int* shares_per_unit) {
    // rows (hidden rows of a pair stream) behind one share of a producer's partial sums: a 128-column unit when the K-slices'
    // reduction writes them or a block holds 256 rows, else the block's rows
    int rows = (pair ? cut.waves * cut.tiles / 2 : cut.waves * cut.tiles) * 16;
    if (cut.ksplit > 1 || rows > 128) rows = 128;
    *ksplit = cut.ksplit;
    *shares = (N + rows - 1) / rows;
    *shares_per_unit = 128 / rows;
}
}  // namespace
extern "C" void mi355_linear_gemm_plan(int M, int N, int K, int R, bool bf16, int* ksplit, int* shares, int* shares_per_unit) {
    plan_shares(gemm_cut(M, N, K, R == 2, bf16, true, false, false), N, R == 2, ksplit, shares, shares_per_unit);
}
extern "C" void mi355_linear_gemm_cut(int M, int N, int K, int R, bool bf16, bool chain, bool sliced, int* waves, int* tokens, int* ksplit) {
    const GemmCut cut = gemm_cut(M, N, K, R == 2, bf16, chain, sliced, false);
    *waves = cut.waves, *tokens = cut.bm, *ksplit = cut.ksplit;
}
extern "C" void mi355_linear_gemm_cut_streamed(int M, int N, int K, int R, bool sliced, int* waves, int* tokens, int* ksplit) {
    const GemmCut cut = gemm_cut(M, N, K, R == 2, true, false, sliced, true);
    *waves = cut.waves, *tokens = cut.bm, *ksplit = cut.ksplit;
}
extern "C" void mi355_linear_gemm_sums(int M, int N, int K, int R, bool chain, int* tiles, int* ksplit, int* runs, int* longest, int* longest_of_wide) {
    const GemmCut cut = gemm_cut(M, N, K, R == 2, false, chain, false, false);
    int run_units;
    gemm_runs(M, N, K, R == 2, cut, runs, &run_units);
    *tiles = cut.tiles, *ksplit = cut.ksplit, *longest = gemm_longest(M, N, K, R == 2, cut), *longest_of_wide = gemm_longest(M, N, K, R == 2, q4_cut(M, N, K, R == 2));
}
void mi355_linear_gemm_plan_grouped(int M, int N, int K, int R, int group_cols, int* ksplit, int* shares, int* shares_per_unit) {
    plan_shares(gemm_cut_grouped((N + 15) / 16, M, R == 2, (K + 127) / 128, grouped_split(M, N, K, R == 2, group_cols)), N, R == 2, ksplit, shares, shares_per_unit);
}

extern "C" void mi355_linear_gemm_cut_grouped(int M, int N, int K, int R, int group_cols, int* waves, int* tokens, int* ksplit) {
    const GemmCut cut = gemm_cut_grouped((N + 15) / 16, M, R == 2, (K + 127) / 128, grouped_split(M, N, K, R == 2, group_cols));
    *waves = cut.waves, *tokens = cut.bm, *ksplit = cut.ksplit;
}

// The tables of several products in one launch: a 7B prompt's layers take theirs 10 products at a time, 15 us (13 MB read, 13 written) instead of a launch in front of
// each, 5 us and its gap, or with the staging pass, 10.5 to 16.6 us for rows and tables
namespace {
struct TableSet {
    GroupTables of[kTableProducts];
    int end[kTableProducts];  // pieces up to the end of each product's
};
__global__ __launch_bounds__(256) void group_tables_kernel(const TableSet set) {
    __shared__ uint32_t lds[kStageLds];
    int i = 0, from = 0;
    while (i < kTableProducts - 1 && (int)blockIdx.x >= set.end[i]) from = set.end[i++];
    group_table_piece(set.of[i], (int)blockIdx.x - from, lds);
}
GroupTables group_tables(const mi355_linear_args& a, int cols, uint32_t* out) {
    return {(const bf16_t*)a.scales, (const bf16_t*)a.zeros, (const bf16_t*)a.scales2, (const bf16_t*)a.zeros2, a.N, (a.N + 15) / 16 * 16, (a.K + cols - 1) / cols, a.R, out};
}
}  // namespace
size_t mi355_linear_gemm_table_bytes(int N, int K, int R, int group_cols) { return table_bytes(0, N, R, (K + group_cols - 1) / group_cols).tables; }
size_t mi355_linear_gemm_table_room() { return kSplitBudget / 2 - 256; }  // (the region itself starts up to 15 bytes past its place)
int mi355_linear_gemm_tables(const mi355_linear_args* products, uint32_t* const* out, int n, mi355_stream_t stream) {
    MI355_CHECK_ARG(n >= 1 && n <= kTableProducts, MI355_E_ARG, "linear_gemm: tables of %d products", n);
    TableSet set;
    memset(&set, 0, sizeof(set));
    int pieces = 0;
    for (int i = 0; i < kTableProducts; ++i) {
        if (i < n) {
            set.of[i] = group_tables(products[i], products[i].group_cols, out[i]);
            pieces += set.of[i].pieces();
        }
        set.end[i] = pieces;
    }
    hipLaunchKernelGGL(group_tables_kernel, dim3(pieces), dim3(256), 0, (hipStream_t)stream, set);
    MI355_LAUNCH_CHECK();
    return 0;
}

static int run_linear_gemm(const mi355_linear_args* a, const mi355_gemm_fuse* f, mi355_reduce_norm* norm, void* workspace, size_t workspace_bytes, mi355_stream_t stream);

int mi355_linear_gemm_fused(const mi355_linear_args* a, const mi355_gemm_fuse* f, void* workspace, size_t workspace_bytes, mi355_stream_t stream) {
    return run_linear_gemm(a, f, nullptr, workspace, workspace_bytes, stream);
}

int mi355_linear_gemm_norm(const mi355_linear_args* a, mi355_reduce_norm* norm, void* workspace, size_t workspace_bytes, mi355_stream_t stream) {
    return run_linear_gemm(a, nullptr, norm, workspace, workspace_bytes, stream);
}

static int run_linear_gemm(const mi355_linear_args* a, const mi355_gemm_fuse* f, mi355_reduce_norm* norm, void* workspace, size_t workspace_bytes, mi355_stream_t stream) {
    MI355_CHECK_ARG(a != nullptr && workspace != nullptr, MI355_E_ARG, "linear_gemm: null argument");
    MI355_CHECK_ARG(a->fmt == MI355_W_Q4 || a->fmt == MI355_W_BF16, MI355_E_ARG,
                    "linear_gemm: the wide path handles the Q4 and BF16 streams (fmt %d)", a->fmt);
    const bool q4 = a->fmt == MI355_W_Q4, streamed = (a->flags & MI355_LF_STREAMED) != 0;
    MI355_CHECK_ARG(a->w && a->x && a->y && (!q4 || (a->scales && a->zeros)), MI355_E_ARG, "linear_gemm: null w/x/y/scales/zeros");
    // grouped scales: group_cols = input columns per (scale, zero) pair; 0 or >= K: one pair per output row
    const bool scale_groups = q4 && a->group_cols > 0 && a->group_cols < a->K;
    // Few rows of one pair per output row: as one group, unit by unit.  The levels enter as 128 + q, and with single activations 10^4 times the others a sum of
    // those over a whole K-slice in one accumulator loses what the row kernel, whose eight waves sum a part each, keeps (logits of a full-depth model with a
    // trained model's statistics, 14 tokens: off by 0.05 of their spread there, 0.08 here, unit by unit 0.03).
    const bool unit_sums = q4 && !scale_groups && f == nullptr && a->M < 32 && a->K % 128 == 0 && a->sz_dtype == MI355_BF16 && (a->alpha == 0.f || a->alpha == 1.f) &&
                           !(a->flags & MI355_LF_NORM_ONE) && mi355_linear_gemm_tables_fit(a->M, a->N, a->K, a->R, a->K);
    const bool grouped = scale_groups || unit_sums;
    int gq_shift = 0;
    if (scale_groups) {
        while ((32 << gq_shift) < a->group_cols) ++gq_shift;
        MI355_CHECK_ARG((32 << gq_shift) == a->group_cols && a->K % 128 == 0, MI355_E_SHAPE,
                        "linear_gemm: group size %d is not 32 * 2^n or K %% 128 != 0 (use the generic kernel)", a->group_cols);
        MI355_CHECK_ARG(a->sz_dtype == MI355_BF16, MI355_E_DTYPE, "linear_gemm: grouped scales / zeros must be bf16");
    }
    MI355_CHECK_ARG(a->M >= 1 && a->N > 0 && a->K > 0, MI355_E_SHAPE, "linear_gemm: bad shape M=%d N=%d K=%d", a->M, a->N, a->K);
    MI355_CHECK_ARG(a->attn_partials == nullptr, MI355_E_ARG, "linear_gemm: no attention prologue");
    MI355_CHECK_ARG(a->bias == nullptr || (!q4 && f == nullptr && a->epi == MI355_EPI_STORE && a->sz_dtype == MI355_F32 && (uintptr_t)a->bias % 16 == 0), MI355_E_ARG,
                    "linear_gemm: an f32 bias goes with the STORE epilogue of the BF16 stream");
    const bool swiglu = is_pair_epi(a->epi);
    MI355_CHECK_ARG(a->epi >= MI355_EPI_STORE && a->epi <= MI355_EPI_CLAMPGLU, MI355_E_ARG, "linear_gemm: bad epi");
    MI355_CHECK_ARG((a->epi != MI355_EPI_GEGLU && a->epi != MI355_EPI_CLAMPGLU) || (!q4 && f == nullptr), MI355_E_ARG, "linear_gemm: GEGLU and CLAMPGLU take the BF16 pair stream");
    MI355_CHECK_ARG(!(a->flags & MI355_LF_NORM_ONE) || !q4 || a->group_cols <= 0 || a->group_cols >= a->K, MI355_E_ARG,
                    "linear_gemm: no 1 + scale norm in front of grouped scales");
    MI355_CHECK_ARG(swiglu ? (a->R == 2 && (!q4 || (a->scales2 && a->zeros2)) && a->y_dtype == MI355_BF16) : a->R == 1, MI355_E_ARG,
                    "linear_gemm: STORE / ACCUM take the R = 1 stream, SWIGLU the interleaved R = 2 stream with bf16 output");
    MI355_CHECK_ARG(a->N % 4 == 0 && a->ldy % 4 == 0, MI355_E_SHAPE, "linear_gemm: N and ldy must be multiples of 4");
    auto two = [](int d) { return d == MI355_F32 || d == MI355_BF16; };
    MI355_CHECK_ARG(two(a->x_dtype) && two(a->y_dtype) && (!q4 || two(a->sz_dtype)), MI355_E_DTYPE, "linear_gemm: dtypes must be f32 or bf16");
    MI355_CHECK_ARG(a->norm_scale == nullptr || two(a->norm_dtype), MI355_E_DTYPE, "linear_gemm: norm scale dtype");
    MI355_CHECK_ARG(workspace_bytes >= mi355_linear_gemm_workspace_bytes(a->M, a->K) && (uintptr_t)workspace % 16 == 0,
                    MI355_E_SHAPE, "linear_gemm: workspace of %zu bytes is too small (need %zu)", workspace_bytes,
                    mi355_linear_gemm_workspace_bytes(a->M, a->K));
    hipStream_t s = (hipStream_t)stream;
    const int units = (a->K + 127) / 128, kp = units * 128;
    bf16_t* xb = (bf16_t*)workspace;
    float* rinv = (float*)((char*)workspace + (size_t)a->M * kp * 2);
    float* sx = rinv + a->M;
    int ksplit = 1;  // K-slices: gemm_cut(); grouped scales: here
    size_t tab_bytes = 0, sxt_bytes = 0;
    int n_groups = 0, tab_ld = 0;
    if (grouped) {
        n_groups = unit_sums ? 1 : (a->K + a->group_cols - 1) / a->group_cols;
        tab_ld = (a->N + 15) / 16 * 16;
        const TableBytes t = table_bytes(a->M, a->N, a->R, n_groups);
        tab_bytes = t.tables;
        sxt_bytes = t.sums;  // (of groups of whole units: in a place of their own)
        MI355_CHECK_ARG(tab_bytes + sxt_bytes <= kSplitBudget, MI355_E_SHAPE,
                        "linear_gemm: group tables of %zu B exceed the workspace region (%zu B)", tab_bytes + sxt_bytes, kSplitBudget);
        // (partial sums: at most half the region, the tables lie in the other)
        ksplit = unit_sums ? q4_cut(a->M, a->N, a->K, swiglu).ksplit : grouped_split(a->M, a->N, a->K, swiglu, a->group_cols);
    }
    int runs = 1, run_units = units;
    if (!grouped) {
        const GemmCut cut = gemm_cut(a->M, a->N, a->K, swiglu, !q4, f != nullptr, a->slice_rows != 0, streamed);
        ksplit = cut.ksplit;
        if (q4) gemm_runs(a->M, a->N, a->K, swiglu, cut, &runs, &run_units);
        MI355_CHECK_ARG(runs <= kMaxRuns && ksplit * runs <= kMaxSums, MI355_E_STATE, "linear_gemm: %d slices of %d runs (M=%d N=%d K=%d)", ksplit, runs, a->M, a->N, a->K);
    }
    // producer / consumer fusion (gemm_fuse.h): one scale per row, or groups of whole units — the caller plans with mi355_linear_gemm_plan or ..._grouped
    const bool fused = f != nullptr;
    const bool f_in = fused && f->prestaged;
    if (fused) {
        MI355_CHECK_ARG(!grouped || (a->group_cols >= 128 && (!f_in || f->tables != nullptr)), MI355_E_STATE,
                        "linear_gemm: fusion over a launch of small groups or without its tables (M=%d N=%d K=%d)", a->M, a->N, a->K);
        const bool produces = f->out_xb != nullptr || f->out_sx != nullptr || f->rope != nullptr;
        MI355_CHECK_ARG(!produces || a->N % 128 == 0, MI355_E_SHAPE, "linear_gemm: a producer of the fused chain has N %% 128 == 0 (N=%d)", a->N);
        MI355_CHECK_ARG(ksplit == 1 || !produces || a->epi == MI355_EPI_SWIGLU || a->y_dtype == MI355_F32, MI355_E_DTYPE,
                        "linear_gemm: the fused reduction of a K-split launch writes f32 rows (or the SwiGLU pair's bf16)");
        MI355_CHECK_ARG(!f_in || (ksplit == 1 && runs == 1 && !grouped) || (f->in_ppu >= 1 && (!grouped || f->in_ppu <= 2) && f->in_sx_n == units * f->in_ppu), MI355_E_ARG,
                        "linear_gemm: a consumer of K-slices, runs or groups needs %d x in_ppu partial operand sums (got %d, in_ppu %d)", units, f->in_sx_n, f->in_ppu);
        MI355_CHECK_ARG(!f_in || (a->x_dtype == MI355_BF16 && a->norm_scale == nullptr && a->K % 128 == 0 && a->ldx % 8 == 0 &&
                                  (uintptr_t)a->x % 16 == 0 && f->in_sx != nullptr && f->in_sx_n > 0 && (f->in_ss == nullptr || f->in_ss_n > 0)),
                        MI355_E_ARG, "linear_gemm: a pre-staged operand is bf16 [M, ldx] with K %% 128 == 0 and partial operand sums");
        MI355_CHECK_ARG(f->out_xb == nullptr || (a->epi == MI355_EPI_ACCUM && a->y_dtype == MI355_F32 && f->next_norm && f->out_ss &&
                                                 f->out_sx && f->out_ld % 4 == 0 && (void*)f->out_xb != a->x &&
                                                 (f_in || (void*)f->out_xb != workspace)),
                        MI355_E_ARG, "linear_gemm: the next operand is emitted by the f32 residual epilogue, next to its partial sums");
        MI355_CHECK_ARG(f->out_sx == nullptr || a->epi == MI355_EPI_SWIGLU || f->out_xb != nullptr, MI355_E_ARG,
                        "linear_gemm: partial operand sums come from the SwiGLU or the emitting residual epilogue");
        MI355_CHECK_ARG(f->rope == nullptr || (a->epi == MI355_EPI_STORE && f->pos && f->kcache && f->vcache && f->hs == 128 && f->S > 0 &&
                                               a->N == 3 * f->n_head * f->hs),
                        MI355_E_ARG, "linear_gemm: the K / V cache epilogue is c_attn's (N = 3 n_head x 128, STORE)");
    }
    float* part = (float*)((char*)(rinv + unit_sums_at(a->M) + (size_t)a->M * units) + 256);
    part = (float*)(((uintptr_t)part + 15) & ~(uintptr_t)15);
    // a bf16 operand in front of BF16 weights, whole units of it and no norm: multiplied where it lies
    const bool direct = !fused && !q4 && a->norm_scale == nullptr && a->x_dtype == MI355_BF16 && a->K % 128 == 0 && a->ldx % 8 == 0 &&
                        (uintptr_t)a->x % 16 == 0;
    const bool aligned = ((uintptr_t)a->x | (uintptr_t)a->norm_scale) % 16 == 0 && a->ldx % 4 == 0;
    GemmParams p;
    memset(&p, 0, sizeof(p));
    if (grouped) {
        // the group tables live in the split-K region of the workspace (its second half when the launch is split)
        const uint32_t* gtab = (uint32_t*)((char*)part + (ksplit > 1 ? kSplitBudget / 2 : 0));
        const int cols = unit_sums || a->group_cols >= 128 ? 128 : a->group_cols;
        const float* sxt = cols == 128 ? rinv + unit_sums_at(a->M) : (const float*)((const char*)gtab + tab_bytes);
        if (f_in) {
            gtab = f->tables;
            sxt = f->in_sx;
        } else {
            const GroupTables tables = group_tables(*a, unit_sums ? a->K : a->group_cols, (uint32_t*)gtab);
            hipLaunchKernelGGL(aligned ? stage_units_kernel<true> : stage_units_kernel<false>, dim3(a->M + tables.pieces()), dim3(256), 0, s, a->x, a->x_dtype, a->ldx,
                               a->norm_scale, a->norm_dtype, a->eps, a->K, xb, rinv, (float*)nullptr, 1, 1, units, 1.f, 0.f, (float*)sxt, a->M, cols, tables);
            MI355_LAUNCH_CHECK();
        }
        p.gtab = gtab;
        p.sxt = sxt;
        p.n_groups = n_groups;
        p.gq_shift = unit_sums ? 30 : a->group_cols >= 128 ? gq_shift - 2 : gq_shift;
        p.tab_ld = tab_ld;
    } else if (!f_in && !direct && aligned && a->K % 128 == 0 && units <= kStageLds - 32) {
        hipLaunchKernelGGL(stage_units_kernel<true>, dim3(a->M), dim3(256), 0, s, a->x, a->x_dtype, a->ldx, a->norm_scale, a->norm_dtype, a->eps, a->K, xb, rinv,
                           sx, ksplit, runs, run_units, a->alpha == 0.f ? 1.f : a->alpha, (a->flags & MI355_LF_NORM_ONE) ? 1.f : 0.f, (float*)nullptr, a->M, 128,
                           GroupTables{});
        MI355_LAUNCH_CHECK();
    } else if (!f_in && !direct) {
        hipLaunchKernelGGL(stage_rows_kernel, dim3(a->M), dim3(256), 0, s, a->x, a->x_dtype, a->ldx, a->norm_scale, a->norm_dtype,
                           a->eps, a->K, kp, xb, (int64_t)kp, rinv, sx, ksplit, runs, run_units, a->alpha == 0.f ? 1.f : a->alpha,
                           (a->flags & MI355_LF_NORM_ONE) ? 1.f : 0.f);
        MI355_LAUNCH_CHECK();
    }
    p.w = (const uint8_t*)a->w;
    {
        const size_t wb = mi355_packed_bytes(a->fmt, a->N, a->K, a->R, swiglu ? 1 : 0);
        MI355_CHECK_ARG(wb > 0 && wb < 0xFFFFFFF0ull, MI355_E_SHAPE, "linear_gemm: weight stream of %zu B", wb);
        p.w_bytes = (unsigned)wb;
    }
    MI355_CHECK_ARG((size_t)a->M * (f_in || direct ? (size_t)a->ldx : (size_t)kp) * 2 < 0xFFFFFFF0ull, MI355_E_SHAPE,
                    "linear_gemm: M x K too large for one launch");
    p.xb = f_in || direct ? (const bf16_t*)a->x : xb;
    p.ldxb = f_in || direct ? a->ldx : (int64_t)kp;
    p.rinv = direct ? nullptr : rinv;
    p.alpha = a->alpha == 0.f ? 1.f : a->alpha;
    p.limit = a->limit;
    p.bias = (const float*)a->bias;
    MI355_CHECK_ARG(a->slice_rows == 0 || (direct && a->epi == MI355_EPI_STORE && a->slice_rows > 0 && a->slice_rows % 256 == 0 &&
                                           a->N % a->slice_rows == 0 && a->slice_stride % 8 == 0),
                    MI355_E_ARG, "linear_gemm: operand slices take whole row blocks of a bf16 operand and the STORE epilogue");
    p.slice_blocks = a->slice_rows;
    p.slice_stride = a->slice_stride;
    p.sx = sx;
    p.scales = a->scales;
    p.zeros = a->zeros;
    p.scales2 = a->scales2;
    p.zeros2 = a->zeros2;
    p.streamed = streamed;
    p.relu2 = (a->flags & MI355_LF_RELU2) ? 1 : 0;
    MI355_CHECK_ARG(!p.relu2 || (a->epi == MI355_EPI_STORE && !fused), MI355_E_ARG, "linear_gemm: RELU2 belongs to the plain STORE epilogue");
    MI355_CHECK_ARG(!(grouped || f_in) || a->alpha == 0.f || a->alpha == 1.f, MI355_E_ARG, "linear_gemm: alpha needs the staging pass of per-row scales");
    p.y = a->y;
    p.ldy = a->ldy;
    p.M = a->M;
    p.N = a->N;
    p.K = a->K;
    p.units = units;
    p.n_tiles = (a->N + 15) / 16;
    p.sz_dtype = a->sz_dtype;
    p.y_dtype = a->y_dtype;
    p.ksplit = ksplit;
    p.runs = runs;
    p.run_units = run_units;
    p.part = part;
    if (norm != nullptr) {
        norm->done = ksplit > 1 && a->epi == MI355_EPI_ACCUM && a->y_dtype == MI355_F32 && a->N <= kNormHeld * 4096;
        p.rn = *norm;
    }
    if (grouped && !fused) return launch_gemm_grouped_epi<false>(p, a->epi, scale_groups && a->group_cols < 128, s);
    if (fused) {
        p.f_in = f_in ? 1 : 0;
        p.in_sx = f->in_sx;
        p.in_sx_n = f_in ? f->in_sx_n : 0;
        p.in_ppu = f_in ? f->in_ppu : 0;
        p.in_ss = f->in_ss;
        p.in_ss_n = f_in && f->in_ss != nullptr ? f->in_ss_n : 0;
        p.eps = a->eps;
        p.out_xb = f->out_xb;
        p.out_ld = f->out_ld;
        p.next_norm = f->next_norm;
        p.next_norm_dtype = f->next_norm_dtype;
        p.out_ss = f->out_ss;
        p.out_sx = f->out_sx;
        p.rope = f->rope;
        p.pos = f->pos;
        p.kcache = f->kcache;
        p.vcache = f->vcache;
        p.S = f->S;
        p.C = f->n_head * f->hs;
        p.rope_gathered = f->rope_gathered;
        p.q_scale = f->rope != nullptr ? f->q_scale : 0.f;
        if (grouped) return launch_gemm_grouped_epi<true>(p, a->epi, false, s);
        if (q4) return launch_gemm_epi<MI355_W_Q4, true>(p, a->epi, s);
        return launch_gemm_epi<MI355_W_BF16, true>(p, a->epi, s);
    }
    if (q4) return launch_gemm_epi<MI355_W_Q4, false>(p, a->epi, s);
    return launch_gemm_epi<MI355_W_BF16, false>(p, a->epi, s);
}
