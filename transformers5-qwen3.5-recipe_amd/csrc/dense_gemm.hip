// Dense launches (one row range, one weight matrix) as two passes: the packed weights are decoded once into a bf16 scratch
// laid out for the matrix cores, and a plain bf16 tile kernel multiplies with it.
//
// The kernels of mmq_tile.h decode every weight once per 256-row tile inside the matmul's step, where the decoding waves and
// the barrier per 64-wide step set the pace: 0.80-0.85 PFLOP/s at 4096 rows whatever the block format.  Decoding ahead costs
// one write and a few reads of 2 bytes per weight, which stay in the memory-side cache, and leaves a loop whose only work
// per step is LDS reads and MFMAs.
//
// Scratch layout ("panel"): weight rows in groups of eight, each group holding its k in blocks of 64:
//   panel[row / 8][k / 64][8 rows][64 elements], the eight 16-byte chunks of a row XOR-swizzled (panel_slot),
// so that one 1 KB request moves a group's block to LDS as it is.  Forward reads it as [output column][contraction] with
// 16-byte operand reads; grad-input reads the same panel as [contraction][output column] with transposing 8-byte reads
// (ds_read_b64_tr_b16).  The swizzle keeps both free of bank conflicts: sixteen consecutive rows at one chunk cover all
// bank groups, and four consecutive rows at an aligned pair of chunks cover four distinct 32-byte bank runs of each half.
#include <algorithm>
#include <type_traits>

#include "blocks.h"
#include "factor_grad.h"
#include "iq2xxs_grid.h"
#include "launch.h"
#include "mmq_host.h"

namespace ggq {

static __device__ const uint64_t d_iq2xxs_grid_dense[256] = GGQ_IQ2XXS_GRID_INIT;
static __device__ const uint4 d_zero16 = {0, 0, 0, 0};  // what a lane loads past the end of a contraction

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------------
// Decoding passes.  HBM-bound: packed bytes in, two bytes per weight out.

// What chunk index of row r is XOR-ed with (r mod 32 counts).
__device__ __forceinline__ int panel_swizzle(int r) { return ((((r >> 1) & 3) << 1) | ((r >> 3) & 1)) ^ (((r >> 4) & 1) << 2); }

template <int QT>
__device__ __forceinline__ const uint2* stage_tables(uint32_t* lds, int tid, int threads) {
    if constexpr (QT == kIQ2_XXS) {
        for (int i = tid; i < Fmt<kIQ2_XXS>::kTableWords; i += threads) lds[i] = Fmt<kIQ2_XXS>::table_word(i, i < 1024 ? d_iq2xxs_grid_dense[i >> 2] : 0ull);
        __syncthreads();
    }
    return (const uint2*)lds;
}

// One wave per (group of eight weight rows, 256 elements of k): lane (row lane / 8, run lane % 8) decodes one 32-element run;
// the eight lanes of a row read adjacent bytes.  The wave's 4 KB go through LDS and leave in whole 1 KB pieces.  The panel
// holds k0 .. k0 + kcols - 1 of every row; rows from n up to the next multiple of 64 are zeros (a contraction over the rows
// runs to there).
struct DecodeParams {
    const uint8_t* w;
    int64_t row_bytes;
    int n, k, k0, kcols;
    uint8_t* panel;
};
template <int QT>
struct DecodeLds {
    uint8_t out[4][4096];
    uint32_t tables[QT == kIQ2_XXS ? Fmt<kIQ2_XXS>::kTableWords : 1];
};
template <int QT>
__device__ __forceinline__ void decode_panel_body(const DecodeParams& p, int wg, DecodeLds<QT>& lds) {
    auto& out_lds = lds.out;
    const uint8_t* w = p.w;
    const int64_t row_bytes = p.row_bytes;
    const int n = p.n, k = p.k, k0 = p.k0, kcols = p.kcols;
    uint8_t* panel = p.panel;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint2* tab = stage_tables<QT>(lds.tables, threadIdx.x, 256);
    const int kblocks = (kcols + 255) >> 8, steps = kcols >> 6;
    const int64_t unit = (int64_t)wg * 4 + wave;
    const int group = (int)(unit / kblocks), kb = (int)(unit - (int64_t)group * kblocks);
    if (group * 8 >= ((n + 63) & ~63)) return;
    const int row = group * 8 + (lane >> 3), ksub = min((k0 >> 5) + kb * 8 + (lane & 7), (k >> 5) - 1);
    const int live_steps = min(4, steps - kb * 4);
    typename Fmt<QT>::Raw raw;
    uint32_t v[16];
    Fmt<QT>::load(raw, w + (int64_t)min(row, n - 1) * row_bytes, ksub);
    Fmt<QT>::decode(raw, ksub, v, tab);
    if (row >= n) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = 0u;
    }
    const int r8 = lane >> 3, sw = panel_swizzle(row), st = (lane & 7) >> 1, c0 = (lane & 1) * 4;
    uint8_t* mine = out_lds[wave] + st * 1024 + r8 * 128;
#pragma unroll
    for (int i = 0; i < 4; i++) *(uint4*)(mine + ((c0 + i) ^ sw) * 16) = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    // (LDS serves a wave in order; each wave reads back only what it wrote)
    uint8_t* dst = panel + ((int64_t)group * steps + kb * 4) * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint4 piece = *(const uint4*)(out_lds[wave] + i * 1024 + lane * 16);
        if (i < live_steps) *(uint4*)(dst + i * 1024) = piece;
    }
}

template <int QT>
__global__ __launch_bounds__(256) void decode_panel_kernel(DecodeParams p) {
    __shared__ __attribute__((aligned(16))) DecodeLds<QT> lds;
    decode_panel_body<QT>(p, blockIdx.x, lds);
}

// ---- out[m, 0..r_pad) = In[m, :] . F^T for sixteen rows: the four waves deal the contraction out in spans of 128 and add
// their sums in wave order.  F is [r][ldf] (contraction contiguous), or [contraction][r] (NATURAL): then a span of it goes
// through the wave's own LDS as [128][r_pad] and the operand is read back transposed.
// What bounds it is latency: a few dozen workgroups on part of the chip.  So DEPTH spans are in flight per wave, and no load
// stands behind a branch (there the compiler waits for every load before it): past the end of the contraction or of the rank
// a lane reads the last whole piece and drops it.  VEC: rows of F in whole pieces (NATURAL: r is a multiple of eight).  Without,
// a span of F is one run of pieces all the same, and its elements are taken apart behind LDS; one span less is in flight there,
// which leaves the kernel the registers of four workgroups per compute unit (three for ranks above 16).
// The launch with the decoding pass, forward / backward, before there was more than one span in flight and now (us): 512 rows, 2048 x
// 2048 Q8_0, rank 16 13.9 / 11.4 -> 11.0 / 9.6, rank 32 16.4 / 11.4 -> 11.8 / 9.0, rank 4 13.7 / 19.4 -> 10.2 / 9.9; 1021 rows, 512 x
// 2048 Q6_K, rank 8 9.5 / 7.0 -> 7.0 / 7.1; 4096 rows, 4096 x 2048 Q4_K, rank 16 13.7 / 19.2 -> 12.8 / 17.8 (there at the memory's
// rate), rank 20 17.7 / 60.4 -> 12.8 / 20.1.
template <int JB>
struct ThinLds {
    bf16_t f[4][128][JB * 16];
    f32x4_t red[4][JB][64];
};
typedef bf16_t __attribute__((may_alias)) aliasing_bf16_t;  // (read where 16-byte pieces were written)
__device__ __forceinline__ uint4 kept_if(bool keep, const uint4& v) { return make_uint4(keep ? v.x : 0u, keep ? v.y : 0u, keep ? v.z : 0u, keep ? v.w : 0u); }
template <int JB, bool NATURAL, bool VEC>
__device__ __forceinline__ void thin_product_body(const SkinnyNtParams& p, int wg, ThinLds<JB>& lds) {
    constexpr int DEPTH = 4 - JB - (NATURAL && !VEC);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lq = lane >> 4;
    const int m0 = wg * 16, spans = (p.c + 127) / 128;
    const bf16_t* in = p.in[0] + (int64_t)min(m0 + li, p.m - 1) * p.ld_in;
    f32x4_t acc[JB];
#pragma unroll
    for (int jb = 0; jb < JB; jb++) acc[jb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    uint4 x[DEPTH][4], f[DEPTH][JB][4];
    // NATURAL: piece (jb, i) of a span is contraction row ((4 jb + i) 64 + lane) / (2 JB), the lane's eight columns from j.  A rank that
    // is no multiple of eight has no such pieces: there it is the ((4 jb + i) 64 + lane)-th of the 16 r pieces of the span's rows,
    // one run that begins on a whole piece (the base is aligned, 128 rows are 256 r bytes) and ends on one (c is in eights).
    const int nat_j = lane % (2 * JB) * 8, nat_row = lane / (2 * JB);
    auto load = [&](int d, int span) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) x[d][i] = *(const uint4*)(in + min(span * 128 + 32 * i + 8 * lq, p.c - 8));
#pragma unroll
        for (int jb = 0; jb < JB; jb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (NATURAL) {
                    const int row = span * 128 + (4 * jb + i) * (32 / JB) + nat_row;
                    if constexpr (VEC) f[d][jb][i] = *(const uint4*)(p.f + (int64_t)min(row, p.c - 1) * p.r + min(nat_j, p.r - 8));
                    else f[d][jb][i] = *(const uint4*)(p.f + min((int64_t)span * 128 * p.r + 8 * min((4 * jb + i) * 64 + lane, 16 * p.r - 1), (int64_t)p.c * p.r - 8));
                } else {
                    f[d][jb][i] = *(const uint4*)(p.f + (int64_t)min(jb * 16 + li, p.r - 1) * p.ldf + min(span * 128 + 32 * i + 8 * lq, p.c - 8));
                }
            }
    };
    auto multiply = [&](int d, int span) __attribute__((always_inline)) {
        if (span * 128 + 128 > p.c) {  // the last, partial span
#pragma unroll
            for (int i = 0; i < 4; i++) {
                x[d][i] = kept_if(span * 128 + 32 * i + 8 * lq < p.c, x[d][i]);
#pragma unroll
                for (int jb = 0; VEC && jb < JB; jb++)
                    f[d][jb][i] = kept_if((NATURAL ? span * 128 + (4 * jb + i) * (32 / JB) + nat_row : span * 128 + 32 * i + 8 * lq) < p.c, f[d][jb][i]);
            }
        }
        bf16x8_t b[JB][4];
        if constexpr (NATURAL) {
            uint4* dst = (uint4*)&lds.f[wave][0][0];
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int i = 0; i < 4; i++) dst[(jb * 4 + i) * 64 + lane] = VEC ? kept_if(nat_j < p.r, f[d][jb][i]) : f[d][jb][i];
            // (LDS serves a wave in order, and no other wave uses this piece)
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (VEC) {
                        const bf16_t* src = &lds.f[wave][32 * i + 8 * lq + (li >> 2)][jb * 16 + (li & 3) * 4];
                        const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)src);
                        const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(src + 4 * JB * 16));
                        b[jb][i] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                    } else {  // rows of any rank start at any element: one at a time
                        const int row = 32 * i + 8 * lq, j = jb * 16 + li, r = (int)opaque((uint32_t)p.r);  // (else the addresses of all are kept through the loop)
                        const aliasing_bf16_t* src = (const aliasing_bf16_t*)&lds.f[wave][0][0] + row * r + min(j, r - 1);
                        uint32_t e[8];
#pragma unroll
                        for (int t = 0; t < 8; t++) e[t] = src[t * r];
                        b[jb][i] = __builtin_bit_cast(bf16x8_t, kept_if(j < r && span * 128 + row < p.c, make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16)));
                    }
                }
        } else {
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int i = 0; i < 4; i++) b[jb][i] = __builtin_bit_cast(bf16x8_t, kept_if(jb * 16 + li < p.r, f[d][jb][i]));
        }
#pragma unroll
        for (int jb = 0; jb < JB; jb++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[d][i]), b[jb][i], acc[jb], 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; d++) load(d, wave + 4 * d);
    int span = wave;
    for (; span + 4 * (DEPTH - 1) < spans; span += 4 * DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            multiply(d, span + 4 * d);
            load(d, span + 4 * (d + DEPTH));
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++)
        if (span + 4 * d < spans) multiply(d, span + 4 * d);
#pragma unroll
    for (int jb = 0; jb < JB; jb++) lds.red[wave][jb][lane] = acc[jb];
    __syncthreads();
    for (int jb = wave; jb < JB; jb += 4) {
        const f32x4_t sum = ((lds.red[0][jb][lane] + lds.red[1][jb][lane]) + lds.red[2][jb][lane]) + lds.red[3][jb][lane];
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (m0 + 4 * lq + v < p.m) p.out[(int64_t)(m0 + 4 * lq + v) * (JB * 16) + jb * 16 + li] = to_bf16(sum[v]);
    }
}

// The decoding pass together with the call's rank-sized work that does not read the panel: the thin product, and the gradient
// of B.  Each alone is a few microseconds of latency on part of the chip; at the sizes of one short sequence they and the gaps
// between their launches were half of a linear layer's step.  Workgroups are dealt in the order thin product (the longest
// chain), gradient, decoding.
struct SidePassParams {
    DecodeParams decode;
    SkinnyNtParams product;
    FactorGradParams gradient;
    int product_wgs, gradient_wgs;
};
template <int QT, int JB>
__global__ __launch_bounds__(256) void decode_side_kernel(SidePassParams p) {
    __shared__ __attribute__((aligned(16))) union {
        DecodeLds<QT> decode;
        ThinLds<JB> thin;
        FactorGradLds<JB, 1> narrow;
        FactorGradLds<JB, 2> wide;
    } lds;
    int wg = blockIdx.x;
    if (wg < p.product_wgs) {
        if (!p.product.f_natural) return thin_product_body<JB, false, true>(p.product, wg, lds.thin);
        if (p.product.r % 8 == 0) return thin_product_body<JB, true, true>(p.product, wg, lds.thin);
        return thin_product_body<JB, true, false>(p.product, wg, lds.thin);
    }
    wg -= p.product_wgs;
    if (wg < p.gradient_wgs) {
        if (p.gradient.c % 128 == 0) factor_grad_body<JB, 2>(p.gradient, wg, lds.wide);
        else factor_grad_body<JB, 1>(p.gradient, wg, lds.narrow);
        return;
    }
    decode_panel_body<QT>(p.decode, wg - p.gradient_wgs, lds.decode);
}

// ------------------------------------------------------------------------------------------------
// The tile kernel: C[m, col] = sum_t A[m, t] * W(col, t), plus scale * LA . LB when a LoRA term comes along.
struct DenseParams {
    const bf16_t* a;
    int64_t lda;
    int contraction;       // real length; steps = ceil / 64; past it A counts as zero
    const uint8_t* panel;
    int panel_steps;       // 64-element blocks of a panel row
    int m, cols;           // cols: columns of this launch
    void* c;               // bf16 [m][ldc], or fp32
    int64_t ldc;
    const float* row_scale;  // accumulate epilogue
    int splits;            // contraction dealt to this many workgroups (partial epilogue)
    int64_t split_stride;  // floats between two splits' partial sums
    // LoRA: la [m, r_pad]; lb [cols][rank], or (lb_k_major) [rank][lb_ld] with the columns contiguous
    const bf16_t *la, *lb;
    int r_pad, rank, lb_k_major;
    int64_t lb_ld;
    float lora_scale;
};
enum : int { kDenseStore = 0, kDenseAccum = 1, kDensePartial = 2 };

// Waves form a WM x WN grid, each owning RB x CB blocks of 16 x 16; NS stages of 64 contraction elements in LDS.
//
// What bounds it at a few thousand rows is power: on every compute unit at once the chip holds 1.7 to 2.0 GHz, and 16x16x32
// MFMAs get 2.05 PFLOP/s out of that (random operands in registers), 32x32x16 ones 1.83.
template <int WM, int WN, int RB, int CB, int NS>
struct DenseTile {
    static constexpr int kBM = WM * RB * 16, kBN = WN * CB * 16, kWaves = WM * WN, kThreadsWG = 64 * kWaves;
    static constexpr int kLoadsA = kBM / 8 / kWaves, kLoadsB = kBN / 8 / kWaves, kLoads = kLoadsA + kLoadsB;
    static constexpr int kStageA = kBM * 128, kStage = (kBM + kBN) * 128;
    static constexpr int kLdsBytes = NS * kStage;
    static constexpr int kOutPitch = CB * 32 + 16;  // bytes of a staged output row
    static_assert(kWaves * 32 * kOutPitch <= kLdsBytes, "output staging");
};

__device__ __forceinline__ void wait_loads(int n) {  // at most n of this wave's requests outstanding (n known at compile time after inlining)
    switch (n) {
        case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
        case 4: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
        case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
        case 8: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
        case 12: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    }
}

template <class T, int MODE, int WM, int WN, int RB, int CB, int NS, int EPI>
__device__ __forceinline__ void dense_body(const DenseParams& p, uint8_t* lds) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    // tile: every XCD takes a contiguous run of the tiles, ordered in stripes of four row tiles, so that the workgroups
    // running together on one XCD share row and column operands in its L2
    const int row_tiles = (p.m + T::kBM - 1) / T::kBM, col_tiles = (p.cols + T::kBN - 1) / T::kBN;
    const int total = row_tiles * col_tiles * p.splits, per_xcd = (total + 7) >> 3;
    int t = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || t >= total) return;
    const int split = t % p.splits;
    t /= p.splits;
    constexpr int kStripe = 4;
    const int stripe = t / (kStripe * col_tiles), in_stripe = t - stripe * kStripe * col_tiles;
    const int stripe_rows = min(kStripe, row_tiles - stripe * kStripe);
    const int row0 = (stripe * kStripe + in_stripe % stripe_rows) * T::kBM, col0 = (in_stripe / stripe_rows) * T::kBN;
    const int rows_valid = min(T::kBM, p.m - row0);

    const int all_steps = (p.contraction + 63) >> 6;
    const int per_split = (all_steps + p.splits - 1) / p.splits;
    const int s_begin = split * per_split, s_end = min(all_steps, s_begin + per_split), steps = s_end - s_begin;

    uint32_t a_off[T::kLoadsA];
    int a_chunk[T::kLoadsA];
#pragma unroll
    for (int j = 0; j < T::kLoadsA; j++) {
        const int r = 8 * (wave + T::kWaves * j) + (lane >> 3);
        a_chunk[j] = (lane & 7) ^ panel_swizzle(r);
        a_off[j] = ((uint32_t)min(r, rows_valid - 1) * (uint32_t)p.lda + (uint32_t)a_chunk[j] * 8u) * 2u;  // rows past the end repeat the last: never stored
    }
    const bf16_t* a_base = p.a + (int64_t)row0 * p.lda + (int64_t)s_begin * 64;
    // column operand requests: forward, eight columns (a row group) x 64 contraction elements each; grad-input, eight
    // contraction rows x 64 columns, block b of the tile's columns behind block b - 1 in LDS
    const uint8_t* b_src[T::kLoadsB];
    int64_t b_step;
    if (MODE == kModeNT) {
        b_step = 1024;
#pragma unroll
        for (int j = 0; j < T::kLoadsB; j++) b_src[j] = p.panel + ((int64_t)(col0 / 8 + wave + T::kWaves * j) * all_steps + s_begin) * 1024;
    } else {
        b_step = (int64_t)p.panel_steps * 8 * 1024;
#pragma unroll
        for (int j = 0; j < T::kLoadsB; j++) {
            const int u = wave + T::kWaves * j, block = min(col0 / 64 + (u >> 3), p.panel_steps - 1);  // (columns past the end are never stored)
            b_src[j] = p.panel + ((int64_t)(s_begin * 8 + (u & 7)) * p.panel_steps + block) * 1024;
        }
    }
    const int tail = p.contraction & 63;  // live elements of the last step, 0: all
    // request q of step s into its stage; whole: the step is known not to be the one the contraction ends in
    auto request = [&](int s, uint32_t stage_off, int q, bool whole) __attribute__((always_inline)) {
        const uint32_t dst = lds0 + stage_off + (q < T::kLoadsA ? (wave + T::kWaves * q) * 1024 : T::kStageA + (wave + T::kWaves * (q - T::kLoadsA)) * 1024);
        if (q >= T::kLoadsA) {
            load16_to_lds(dst, (uint32_t)lane * 16u, b_src[q - T::kLoadsA] + s * b_step);
        } else if (!whole && tail != 0 && s_begin + s == all_steps - 1) {
            const void* src = a_chunk[q] * 8 < tail ? (const void*)((const uint8_t*)(a_base + (int64_t)s * 64) + a_off[q]) : (const void*)&d_zero16;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(dst), "v"(src) : "memory");
        } else {
            load16_to_lds(dst, a_off[q], a_base + (int64_t)s * 64);
        }
    };

    f32x4_t acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    const int l16 = lane & 15, quarter = lane >> 4;
    if (p.la && split == 0) {  // scale * LA . LB first (operands straight from memory: one or two MFMAs per block and tile)
        for (int r0 = 0; r0 < p.r_pad; r0 += 32) {
            const int r = r0 + 8 * quarter;  // this lane's eight ranks (zeros past the rank in both operands)
            bf16x8_t lbv[CB];
#pragma unroll
            for (int j = 0; j < CB; j++) {
                const int col = min(col0 + (wn * CB + j) * 16 + l16, p.cols - 1);
                if (!p.lb_k_major) {
                    lbv[j] = __builtin_bit_cast(bf16x8_t, load8g(p.lb + (int64_t)col * p.rank + r, p.rank - r, (p.rank & 7) == 0));
                } else {
                    uint32_t e[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const uint32_t x = p.lb[(int64_t)min(r + i, p.rank - 1) * p.lb_ld + col];
                        e[i] = r + i < p.rank ? x : 0u;
                    }
                    lbv[j] = __builtin_bit_cast(bf16x8_t, make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)));
                }
            }
#pragma unroll
            for (int i = 0; i < RB; i++) {
                const int row = row0 + min((wm * RB + i) * 16 + l16, rows_valid - 1);
                const bf16x8_t lav = __builtin_bit_cast(bf16x8_t, r < p.r_pad ? *(const uint4*)(p.la + (int64_t)row * p.r_pad + r) : make_uint4(0, 0, 0, 0));
#pragma unroll
                for (int j = 0; j < CB; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lbv[j], lav, acc[i][j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int j = 0; j < CB; j++) acc[i][j] *= p.lora_scale;
    }

    // Main loop.  A step is two sub-steps of 32 contraction elements (chunks kk, 2 + kk, 4 + kk, 6 + kk of a row, one per lane
    // quarter: any order serves a sum, and these meet no bank conflict), each RB rows of CB MFMAs.  A row block's operand of
    // the next sub-step is read into the registers its row has just released, the last row's at the start of that sub-step; column
    // operands have two sets.  The step's one barrier stands kBarrierRow rows into the second sub-step, where every read of the
    // stage has returned: behind it the stage is refilled with step s + NS and the next stage's first operands are read, all
    // under MFMAs, so no wave meets the barrier with an idle matrix pipe behind it.
#pragma unroll
    for (int s = 0; s < NS; s++)
        if (s < steps)
#pragma unroll
            for (int q = 0; q < T::kLoads; q++) request(s, s * T::kStage, q, false);
    // LDS offsets of this lane's operand chunks, by sub-step: rows (and forward's columns) of even and odd blocks of sixteen;
    // grad-input: lane s of sixteen points at row s / 4 of four contraction rows, columns 4 (s % 4) .. + 3
    uint32_t ra[2][2], rb[2][MODE == kModeNT ? 2 : 2 * CB];
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int odd = 0; odd < 2; odd++) {
            const uint32_t slot = (uint32_t)((2 * quarter + kk) ^ panel_swizzle(16 * odd + l16)) * 16u;
            ra[kk][odd] = (uint32_t)(wm * RB * 16 + l16) * 128u + slot;
            if (MODE == kModeNT) rb[kk][odd] = (uint32_t)T::kStageA + (uint32_t)(wn * CB * 16 + l16) * 128u + slot;
        }
    if (MODE == kModeNN) {
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                // chunk (2 j + x) ^ swizzle of the row: j only meets the swizzle's upper two bits, so a block's offset is the
                // first one's with two address bits flipped
                const int row = 8 * (2 * quarter + kk) + 4 * t + (l16 >> 2), sw = panel_swizzle(row) ^ ((l16 & 3) >> 1);
                const uint32_t first = (uint32_t)T::kStageA + (uint32_t)row * 128u + (uint32_t)sw * 16u + (uint32_t)(l16 & 1) * 8u;
#pragma unroll
                for (int j = 0; j < CB; j++) {
                    const int col = (wn * CB + j) * 16;
                    rb[kk][2 * j + t] = (first ^ (uint32_t)((col & 63) * 2)) + (uint32_t)(col >> 6) * 8192u;
                }
            }
    }
    constexpr int kSets = RB <= 4 ? 2 : 1;  // row operand sets
    bf16x8_t fa[kSets][RB], fb[2][CB];
    auto read_a = [&](int i, uint32_t stage_off, int kk) __attribute__((always_inline)) {
        fa[kk & (kSets - 1)][i] = *(const bf16x8_t*)(lds + stage_off + ra[kk][(wm * RB + i) & 1] + i * 2048);
    };
    auto read_b = [&](int set, int j, uint32_t stage_off, int kk) __attribute__((always_inline)) {
        if constexpr (MODE == kModeNT) {
            fb[set][j] = *(const bf16x8_t*)(lds + stage_off + rb[kk][(wn * CB + j) & 1] + j * 2048);
        } else {
            const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(lds + stage_off + rb[kk][2 * j]));
            const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(lds + stage_off + rb[kk][2 * j + 1]));
            fb[set][j] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };
    if (steps > 0) {
        if (steps >= NS) wait_loads((NS - 1) * T::kLoads);
        else wait_loads(0);
        lds_barrier();
#pragma unroll
        for (int j = 0; j < CB; j++) read_b(0, j, 0, 0);
#pragma unroll
        for (int i = 0; i < (kSets == 2 ? RB : RB - 1); i++) read_a(i, 0, 0);
        uint32_t cur = 0;
        static_assert(RB % 2 == 0 && CB % 2 == 0, "blocks of sixteen alternate between two read offsets");
        constexpr int kBarrierRow = kSets == 2 ? 0 : RB / 4;
        // one step; WHOLE: step s + NS exists and is not the contraction's last
        auto step = [&](int s, auto whole_tag) __attribute__((always_inline)) {
            constexpr bool WHOLE = decltype(whole_tag)::value;
            const uint32_t nxt = cur == (NS - 1) * T::kStage ? 0u : cur + T::kStage;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const uint32_t from = kk == 1 ? nxt : cur;  // where the next sub-step's operands are
                constexpr int kFirst[2] = {kSets == 2 ? 0 : 1, kBarrierRow};  // the row from which on they are read
                const int first = kFirst[kk];
#pragma unroll
                for (int i = 0; i < RB; i++) {
                    if (kk == 1 && i == kBarrierRow) {
                        // step s + 1 has landed when only the requests of the steps after it are outstanding
                        if (WHOLE || s + NS - 1 < steps) wait_loads((NS - 2) * T::kLoads);
                        else wait_loads(0);
                        lds_barrier();
                    }
                    if (kSets == 1 && i == 0) read_a(RB - 1, cur, kk);
                    if constexpr (kSets == 2) {  // all of the next sub-step's operands, in the first half of the rows
                        constexpr int kPer = (RB + CB + RB / 2 - 1) / (RB / 2);
#pragma unroll
                        for (int q = i * kPer; q < (i + 1) * kPer && q < RB + CB; q++) {
                            if (q < CB) read_b(kk ^ 1, q, from, kk ^ 1);
                            else read_a(q - CB, from, kk ^ 1);
                        }
                    } else if (i >= first) {  // column operands first, then the operands of the rows done so far
                        const int u = i - first;
#pragma unroll
                        for (int j = u * 2; j < (u + 1) * 2 && j < CB; j++) read_b(kk ^ 1, j, from, kk ^ 1);
                        const int lo = u == 0 ? 0 : kk == 0 ? i - 1 : min(i - 1, 2 * u - 1), hi = kk == 0 ? i : min(i, 2 * u + 1);
#pragma unroll
                        for (int r = lo; r < hi; r++) read_a(r, from, kk ^ 1);
                    }
                    if (kk == 1 && i >= kBarrierRow && (WHOLE || s + NS < steps)) {
                        constexpr int kRows = RB - kBarrierRow;
#pragma unroll
                        for (int q = (i - kBarrierRow) * T::kLoads / kRows; q < (i - kBarrierRow + 1) * T::kLoads / kRows; q++) request(s + NS, cur, q, WHOLE);
                    }
#pragma unroll
                    for (int j = 0; j < CB; j++) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kk][j], fa[kk & (kSets - 1)][i], acc[i][j], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            cur = nxt;
        };
        int s = 0;
        for (; s + NS < steps - 1; s++) step(s, std::true_type{});
        for (; s < steps; s++) step(s, std::false_type{});
    }

    // acc[i][j][v]: row 16 (wm RB + i) + lane % 16, column 16 (wn CB + j) + 4 (lane / 16) + v
    if constexpr (EPI == kDenseStore) {
        __syncthreads();  // every wave is done with the stages; the (surplus) operand reads have returned
        uint8_t* stage = lds + wave * 32 * T::kOutPitch;
        constexpr int kLanesPerRow = CB * 2, kRowsPerStore = 64 / kLanesPerRow;
        const int cw = col0 + wn * CB * 16;
        const bool whole = (p.ldc & 7) == 0 && (((uintptr_t)p.c) & 15) == 0;
#pragma unroll
        for (int i = 0; i < RB; i += 2) {  // 32 rows at a time
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < CB; j++)
                    *(uint2*)(stage + (16 * h + l16) * T::kOutPitch + j * 32 + quarter * 8) =
                        make_uint2(pack_bf16(acc[i + h][j][0], acc[i + h][j][1]), pack_bf16(acc[i + h][j][2], acc[i + h][j][3]));
            const int ch = lane % kLanesPerRow;
#pragma unroll
            for (int u = 0; u < 32 / kRowsPerStore; u++) {
                const int rl = u * kRowsPerStore + lane / kLanesPerRow;
                const uint4 piece = *(const uint4*)(stage + rl * T::kOutPitch + ch * 16);
                const int row = (wm * RB + i) * 16 + rl, col = cw + ch * 8;
                if (row < rows_valid) {
                    bf16_t* dst = (bf16_t*)p.c + (int64_t)(row0 + row) * p.ldc + col;
                    if (whole && col + 8 <= p.cols) {
                        *(uint4*)dst = piece;
                    } else {
                        const uint32_t wds[4] = {piece.x, piece.y, piece.z, piece.w};
#pragma unroll
                        for (int e = 0; e < 8; e++)
                            if (col + e < p.cols) dst[e] = (bf16_t)((e & 1) ? wds[e >> 1] >> 16 : wds[e >> 1] & 0xFFFFu);
                    }
                }
            }
        }
    } else {
        float* c = (float*)p.c + (EPI == kDensePartial ? (int64_t)split * p.split_stride : 0);
#pragma unroll
        for (int i = 0; i < RB; i++) {
            const int row = (wm * RB + i) * 16 + l16;
            if (row >= rows_valid) continue;
            const float rs = EPI == kDenseAccum && p.row_scale ? p.row_scale[row0 + row] : 1.0f;
            float* dst_row = c + (int64_t)(row0 + row) * p.ldc;
#pragma unroll
            for (int j = 0; j < CB; j++) {
                const int col = col0 + (wn * CB + j) * 16 + quarter * 4;
                if (col >= p.cols) continue;  // (fp32 outputs have a multiple of four columns)
                float4* dst = (float4*)(dst_row + col);
                float4 o = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
                if (EPI == kDenseAccum) {
                    const float4 old = *dst;
                    o.x = fmaf(old.x, rs, o.x), o.y = fmaf(old.y, rs, o.y), o.z = fmaf(old.z, rs, o.z), o.w = fmaf(old.w, rs, o.w);
                }
                *dst = o;
            }
        }
    }
}

template <int MODE, int WM, int WN, int RB, int CB, int NS, int EPI>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2, 2))) void dense_gemm_kernel(DenseParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dense_lds[];
    dense_body<DenseTile<WM, WN, RB, CB, NS>, MODE, WM, WN, RB, CB, NS, EPI>(p, dense_lds);
}

// Split partial sums, added in split order, into an fp32 accumulator: c = c * row_scale + sum (replace: c = sum).
__global__ __launch_bounds__(256) void dense_reduce_accum_kernel(const float* partial, int64_t split_stride, int splits, int64_t m, int64_t cols, float* c, int64_t ldc,
                                                                 const float* row_scale, int replace) {
    const int64_t quads = cols / 4, total = m * quads;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / quads, q = i - row * quads;
        float4 s = ((const float4*)(partial + row * cols))[q];
        for (int k = 1; k < splits; k++) {
            const float4 t = ((const float4*)(partial + k * split_stride + row * cols))[q];
            s.x += t.x, s.y += t.y, s.z += t.z, s.w += t.w;
        }
        float4* dst = (float4*)(c + row * ldc) + q;
        if (!replace) {
            const float rs = row_scale ? row_scale[row] : 1.0f;
            const float4 old = *dst;
            s.x = fmaf(old.x, rs, s.x), s.y = fmaf(old.y, rs, s.y), s.z = fmaf(old.z, rs, s.z), s.w = fmaf(old.w, rs, s.w);
        }
        *dst = s;
    }
}

// bf16 result of split partial sums, added in split order.
__global__ __launch_bounds__(256) void dense_reduce_kernel(const float* partial, int64_t split_stride, int splits, int64_t m, int64_t cols, bf16_t* c, int64_t ldc) {
    const int64_t quads = cols / 4, total = m * quads;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / quads, q = i - row * quads;
        float4 s = ((const float4*)(partial + row * cols))[q];
        for (int k = 1; k < splits; k++) {
            const float4 t = ((const float4*)(partial + k * split_stride + row * cols))[q];
            s.x += t.x, s.y += t.y, s.z += t.z, s.w += t.w;
        }
        *(uint2*)(c + row * ldc + q * 4) = make_uint2(pack_bf16(s.x, s.y), pack_bf16(s.z, s.w));
    }
}

// ------------------------------------------------------------------------------------------------
template <int MODE, int WM, int WN, int RB, int CB, int NS, int EPI>
static int launch_tile(const DenseParams& p, hipStream_t s) {
    using T = DenseTile<WM, WN, RB, CB, NS>;
    const int64_t tiles = (int64_t)((p.m + T::kBM - 1) / T::kBM) * ((p.cols + T::kBN - 1) / T::kBN) * p.splits;
    const int64_t grid = (tiles + 7) / 8 * 8;
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "dense_gemm: too many tiles for one launch");
    static LdsLimit lim;
    if (int rc = raise_lds_limit(lim, (const void*)dense_gemm_kernel<MODE, WM, WN, RB, CB, NS, EPI>, T::kLdsBytes, "dense_gemm")) return rc;
    hipLaunchKernelGGL((dense_gemm_kernel<MODE, WM, WN, RB, CB, NS, EPI>), dim3((unsigned)grid), dim3(T::kThreadsWG), T::kLdsBytes, s, p);
    return check_launch("dense_gemm");
}
template <int MODE, int EPI>
static int launch_shape_mode(int shape, const DenseParams& p, hipStream_t s) {
    switch (shape) {
        case 0: return launch_tile<MODE, 2, 4, 8, 4, 2, EPI>(p, s);   // 256 x 256
        case 1: return launch_tile<MODE, 2, 2, 4, 4, 2, EPI>(p, s);   // 128 x 128, two workgroups per compute unit
        case 2: return launch_tile<MODE, 2, 2, 2, 2, 4, EPI>(p, s);   // 64 x 64, two workgroups per compute unit
        case 3: return launch_tile<MODE, 2, 4, 4, 4, 3, EPI>(p, s);   // 128 x 256
    }
    return set_error(GGQ_ERR_SHAPE, "dense_gemm: unknown tile shape");
}
template <int EPI>
static int launch_shape(int mode, int shape, const DenseParams& p, hipStream_t s) {
    return mode == kModeNT ? launch_shape_mode<kModeNT, EPI>(shape, p, s) : launch_shape_mode<kModeNN, EPI>(shape, p, s);
}

template <int QT>
static int launch_decode_panel(const DecodeParams& d, const DenseSide* side, hipStream_t s) {
    const int64_t units = (int64_t)((d.n + 63) / 64 * 8) * ((d.kcols + 255) / 256), wgs = (units + 3) / 4;
    if (!side) {
        hipLaunchKernelGGL(decode_panel_kernel<QT>, dim3((unsigned)wgs), dim3(256), 0, s, d);
        return check_launch("decode_panel");
    }
    SidePassParams p{};
    p.decode = d;
    if (side->product) p.product = *side->product, p.product_wgs = (p.product.m + 15) / 16;
    if (side->gradient) {
        p.gradient_wgs = (int)factor_grad_plan(*side->gradient, side->r_pad, 1);
        p.gradient = *side->gradient;
    }
    const dim3 grid((unsigned)(wgs + p.product_wgs + p.gradient_wgs));
    if (side->r_pad == 16) hipLaunchKernelGGL((decode_side_kernel<QT, 1>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((decode_side_kernel<QT, 2>), grid, dim3(256), 0, s, p);
    return check_launch("decode_side");
}
static int decode_panel(int qt, const DecodeParams& d, const DenseSide* side, hipStream_t s) {
    switch (qt) {
        case kQ8_0: return launch_decode_panel<kQ8_0>(d, side, s);
        case kQ2_K: return launch_decode_panel<kQ2_K>(d, side, s);
        case kQ3_K: return launch_decode_panel<kQ3_K>(d, side, s);
        case kQ4_K: return launch_decode_panel<kQ4_K>(d, side, s);
        case kQ5_K: return launch_decode_panel<kQ5_K>(d, side, s);
        case kQ6_K: return launch_decode_panel<kQ6_K>(d, side, s);
        case kIQ2_XXS: return launch_decode_panel<kIQ2_XXS>(d, side, s);
    }
    return set_error(GGQ_ERR_QTYPE, "unsupported GGML type id %d", qt);
}

// Aligned rows in eights, one segment without an index, rank up to kDenseSideMaxRank.  (A natural factor is aligned: the entry points refuse
// others.)
bool dense_side_takes(const DenseSide& side) {
    if (side.r_pad > kDenseSideMaxRank) return false;
    if (const SkinnyNtParams* q = side.product)
        if (q->nseg != 1 || q->in_rows.on() || q->c % 8 || q->ld_in % 8 || ((uintptr_t)q->in[0] & 15) || (!q->f_natural && (q->ldf % 8 || ((uintptr_t)q->f & 15)))) return false;
    return true;
}

// ------------------------------------------------------------------------------------------------
// Panels of at most this many bytes are decoded at a time: small enough to be read back out of the 256 MB memory-side cache,
// large enough that a slab's launch fills the chip.  Larger matrices go in slabs of output columns.
constexpr int64_t kPanelBytes = 128ll << 20;
constexpr int kMaxSplits = 16;

static int64_t slab_columns(int64_t cols, int64_t contraction) {
    const int64_t steps = (contraction + 63) / 64, fit = kPanelBytes / (steps * 128) / 256 * 256;
    const int64_t padded = (cols + 255) / 256 * 256;
    return std::min(padded, std::max<int64_t>(fit, 256));
}

// Whether both directions of an [n, k] matrix run over one panel of all of it.
bool dense_panel_whole(int64_t n, int64_t k) { return slab_columns(n, k) >= n && slab_columns(k, n) >= k; }

// Tile shape and number of contraction splits for an [m, cols] output: the smallest estimate of the launch, plus the pass that
// adds split partial sums.  A tile's 64-wide step slows down with the share of the chip that is busy (clock and L2), by shape
// from `idle` to `full` microseconds; measured at one tile, a quarter, a half and all of the slots, within 10 % of the estimate:
//   256 x 256, one per compute unit:  1.07 / 1.08 / 1.13 / 1.40     128 x 256, one: 0.52 / 0.56 / 0.65 / 0.80
//   128 x 128, two:                   0.37 / 0.55 / 0.62 / 0.90      64 x 64, two: 0.12 / 0.14 / 0.16 / 0.30
// A larger tile reads less per output: 256 x 256 wins where it fills the chip in whole rounds or by splits (4096 x 8192 over
// 2048: 119 us against 128 with 128 x 128), 128 x 256 where it would leave a half of it idle (4096 x 2048 over 8192: 113 us
// against 154, and 122 with 128 x 128), the smaller ones for short sequences.
std::atomic<int> g_dense_shape{-1}, g_dense_splits{0};  // ggq_debug_force_dense_tile (a test aid): the automatic choice

// max_splits: what the output's alignment and the workspace allow (with none, the shape chosen for ten splits can leave most of the
// chip idle: 701 x 2048 over 32768, 577 us against 207 with the shape for one).
static void pick_tile(int64_t m, int64_t cols, int64_t steps, int64_t max_splits, int& shape, int& splits) {
    static const struct { int rows, cols, slots; double idle, full, fixed; } kShape[4] = {
        {256, 256, 256, 1.05, 1.40, 6.0}, {128, 128, 512, 0.36, 0.90, 2.5}, {64, 64, 512, 0.11, 0.30, 2.5}, {128, 256, 256, 0.50, 0.80, 5.0}};  // (fixed: a tile's start and end)
    double best = 1e30;
    const int only_shape = g_dense_shape.load(std::memory_order_relaxed), only_splits = g_dense_splits.load(std::memory_order_relaxed);
    shape = std::max(only_shape, 0), splits = 1;
    for (int sh = 0; sh < 4; sh++) {
        if (only_shape >= 0 && sh != only_shape) continue;
        const auto& t = kShape[sh];
        const int64_t tiles = ((m + t.rows - 1) / t.rows) * ((cols + t.cols - 1) / t.cols);
        for (int sp = 1; sp <= max_splits; sp++) {
            const int64_t per = (steps + sp - 1) / sp;
            if (sp > 1 && (per < 4 || (sp - 1) * per >= steps)) continue;
            if (only_splits > 0 && sp != std::min<int64_t>(only_splits, max_splits)) continue;
            const int64_t units = tiles * sp, rounds = units / t.slots, rest = units % t.slots;
            const double load = (double)rest / t.slots, slow = sh == 0 ? load * load : load;
            double est = 3.0 + rounds * (per * t.full + t.fixed) + (rest ? per * (t.idle + (t.full - t.idle) * slow) + t.fixed : 0.0);
            if (sp > 1) est += 3.0 + (double)m * cols * 4.0 * (1.5 * sp) / 5e6;
            if (est < best * 0.999) best = est, shape = sh, splits = sp;
        }
    }
}

static int64_t splits_with_room(int64_t bytes, int64_t m, int64_t cols) { return std::min<int64_t>(kMaxSplits, std::max<int64_t>(1, bytes / (m * cols * 4))); }

void dense_plan(int mode, int64_t m, int64_t n, int64_t k, int64_t ws_bytes, int& shape, int& splits) {
    const int64_t cols = mode == kModeNT ? n : k, contraction = mode == kModeNT ? k : n, steps = (contraction + 63) / 64;
    const int64_t slab = slab_columns(cols, contraction), panel_bytes = (slab * steps * 128 + 255) / 256 * 256, cn = std::min(cols, slab);
    pick_tile(m, cn, steps, cn % 4 == 0 ? splits_with_room(ws_bytes - panel_bytes, m, cn) : 1, shape, splits);
}

int64_t dense_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    if (m < kDenseMinRows || n <= 0 || k <= 0) return 0;
    const int64_t nt = slab_columns(n, k) * ((k + 63) / 64) * 128, nn = slab_columns(k, n) * ((n + 63) / 64) * 128;
    int64_t partial = 0;
    for (int mode = 0; mode < 2; mode++) {
        const int64_t cols = mode == kModeNT ? n : k, c = mode == kModeNT ? k : n;
        const int64_t slab = std::min(cols, slab_columns(cols, c));
        int shape, splits;
        pick_tile(m, slab, (c + 63) / 64, slab % 4 == 0 ? kMaxSplits : 1, shape, splits);
        if (splits > 1) partial = std::max(partial, (int64_t)splits * m * slab * 4);
    }
    return (std::max(nt, nn) + 255) / 256 * 256 + (partial + 255) / 256 * 256;
}

bool dense_takes(int mode, int64_t m, int64_t n, int64_t k, const void* a, int64_t lda, bool a_zero_padded) {
    const int64_t cols = mode == kModeNT ? n : k, contraction = mode == kModeNT ? k : n;
    return m >= kDenseMinRows && ((uintptr_t)a & 15) == 0 && lda % 8 == 0 && (contraction % 8 == 0 || a_zero_padded) && 256 * lda < (1ll << 30) && cols > 0;
}

int dense_mmq(const DenseCall& q, void* ws, int64_t ws_bytes, hipStream_t s, const DenseSide* side) {
    const int64_t cols = q.mode == kModeNT ? q.n : q.k, contraction = q.mode == kModeNT ? q.k : q.n, steps = (contraction + 63) / 64;
    if (!block_multiple(q.qt, q.k) || q.k % 64) return set_error(GGQ_ERR_SHAPE, "dense_gemm: K=%lld must be a multiple of 64 and of the block size of type %d", (long long)q.k, q.qt);
    const int64_t slab = slab_columns(cols, contraction), panel_bytes = (slab * steps * 128 + 255) / 256 * 256;
    if (!ws || ws_bytes < panel_bytes) return set_error(GGQ_ERR_WORKSPACE, "dense_gemm: workspace too small");
    if (q.accumulate && (q.mode != kModeNN || !q.fp32)) return set_error(GGQ_ERR_SHAPE, "dense_gemm: only the fp32 grad-input accumulates");
    const int64_t row_bytes = packed_row_bytes(q.qt, q.k);
    uint8_t* panel = (uint8_t*)ws;
    TimedScope timed(q.qt, q.mode, q.fp32 ? kEpiAccumF32 : kEpiStore, kShapePanels, s);
    for (int64_t c0 = 0; c0 < cols; c0 += slab) {
        const int64_t cn = std::min(slab, cols - c0);
        const uint8_t* w = (const uint8_t*)q.w + (q.mode == kModeNT ? c0 * row_bytes : 0);
        const int kcols = (int)(q.mode == kModeNT ? q.k : cn);
        if (!q.panel_ready)
            if (int rc = decode_panel(q.qt, DecodeParams{w, row_bytes, (int)(q.mode == kModeNT ? cn : q.n), (int)q.k, (int)(q.mode == kModeNT ? 0 : c0), kcols, panel},
                                      c0 == 0 ? side : nullptr, s)) return rc;
        DenseParams p{};
        p.a = (const bf16_t*)q.a, p.lda = q.lda, p.contraction = (int)(q.a_zero_padded ? steps * 64 : contraction);
        p.panel = panel, p.panel_steps = kcols / 64, p.m = (int)q.m, p.cols = (int)cn, p.ldc = q.ldc, p.row_scale = q.row_scale;
        if (q.la) {
            p.la = (const bf16_t*)q.la, p.r_pad = q.r_pad, p.rank = q.rank, p.lora_scale = q.lora_scale, p.lb_k_major = q.mode == kModeNN, p.lb_ld = q.k;
            p.lb = (const bf16_t*)q.lb + (q.mode == kModeNT ? c0 * q.rank : c0);
        }
        int shape, splits;
        const bool can_split = cn % 4 == 0 && q.ldc % 4 == 0 && ((uintptr_t)q.c & 7) == 0;
        pick_tile(q.m, cn, steps, can_split ? splits_with_room(ws_bytes - panel_bytes, q.m, cn) : 1, shape, splits);
        p.splits = splits;
        if (splits > 1) {
            float* partial = (float*)(panel + panel_bytes);
            p.c = partial, p.ldc = cn, p.split_stride = q.m * cn;
            if (int rc = launch_shape<kDensePartial>(q.mode, shape, p, s)) return rc;
            const int64_t work = q.m * (cn / 4);
            if (q.fp32)
                hipLaunchKernelGGL(dense_reduce_accum_kernel, dim3((unsigned)std::min<int64_t>((work + 255) / 256, 4096)), dim3(256), 0, s, partial, p.split_stride, splits, q.m,
                                   cn, (float*)q.c + c0, q.ldc, q.row_scale, q.accumulate ? 0 : 1);
            else hipLaunchKernelGGL(dense_reduce_kernel, dim3((unsigned)std::min<int64_t>((work + 255) / 256, 4096)), dim3(256), 0, s, partial, p.split_stride, splits, q.m, cn,
                               (bf16_t*)q.c + c0, q.ldc);
            if (int rc = check_launch("dense_reduce")) return rc;
        } else if (q.fp32) {
            p.c = (float*)q.c + c0;
            if (int rc = q.accumulate ? launch_shape_mode<kModeNN, kDenseAccum>(shape, p, s) : launch_shape<kDensePartial>(q.mode, shape, p, s)) return rc;
        } else {
            p.c = (bf16_t*)q.c + c0;
            if (int rc = launch_shape<kDenseStore>(q.mode, shape, p, s)) return rc;
        }
    }
    return GGQ_OK;
}

}  // namespace ggq
