// The factor-gradient product, as a device function that several launches share.
#pragma once
#include "common.h"
#include "mmq_host.h"

namespace ggq {

typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16_t* lds_v4i16_ptr;

__device__ __forceinline__ uint4 load8g(const bf16_t* p, int valid, bool vec) {
    if (valid >= 8 && vec) return *(const uint4*)p;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (valid <= 0) return v;
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 8; i++) e[i] = i < valid ? (uint32_t)p[i] : 0u;
    v.x = e[0] | (e[1] << 16), v.y = e[2] | (e[3] << 16), v.z = e[4] | (e[5] << 16), v.w = e[6] | (e[7] << 16);
    return v;
}

// ---- G[e][c, j] = s * sum_m In[m, c] * S[m, j] over the rows of expert e.  One workgroup per
// (expert, 64 * CB columns); each wave owns CB blocks of 16 columns; rows are consumed 32 at a time
// through LDS, where the operands of the contraction over m are read with transposing loads.  The loads
// of four 32-row slices are issued together (of rows in place; a slice of rows behind an index waits for its
// indices and the loads before them, one with routing weights for its weights) and the slices then go through
// two alternating LDS buffers, one barrier each.  Experts without rows get zeros.
template <int JB, int CB>
struct FactorGradLds {
    static constexpr int kPitch = 64 * CB + 32, kSPitch = JB * 16 + 8;
    bf16_t in_t[2][32][kPitch];
    bf16_t s_t[2][32][kSPitch];
    bf16_t g_t[4][16][JB * 16];
};
template <int JB, int CB>
__device__ __forceinline__ void factor_grad_body(const FactorGradParams& p, int unit, FactorGradLds<JB, CB>& lds) {
    // rows are contraction rows m; the operands are read with transposing 8-byte LDS reads (lane L of a
    // 16-lane group gets element L % 4 of the 8 bytes addressed by lanes L / 4 + 4 t), so the tiles stay as
    // loaded; the row pitches keep four consecutive rows' 32-byte pieces on distinct banks
    constexpr int kCols = 64 * CB, kPitch = FactorGradLds<JB, CB>::kPitch, kSPitch = FactorGradLds<JB, CB>::kSPitch;
    auto& in_t = lds.in_t;
    auto& s_t = lds.s_t;
    auto& g_t = lds.g_t;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int blocks_per_seg = (p.c + kCols - 1) / kCols;
    const int col_blocks = p.nseg * blocks_per_seg;
    const int splits = p.row_splits > 1 ? p.row_splits : 1;
    const int split = unit % splits, ucb = unit / splits;
    const int experts = p.units / (col_blocks * splits);
    const int e = p.blocks_outer ? ucb % experts : ucb / col_blocks, cblk = p.blocks_outer ? ucb / experts : ucb - e * col_blocks;
    const int seg = cblk / blocks_per_seg;
    const int c0 = (cblk - seg * blocks_per_seg) * kCols;
    int row_begin = 0, row_end = p.m;
    if (p.ranges) {
        row_begin = p.ranges[2 * e];
        row_end = p.ranges[2 * e + 1];
    } else if (splits > 1) {  // this workgroup's share of the rows, in whole 32-row slices
        const int share = (((p.m + splits - 1) / splits) + 31) & ~31;
        row_begin = min(p.m, split * share);
        row_end = min(p.m, row_begin + share);
    }
    const bf16_t* in = p.in[seg];
    const bool vec = ((p.ld_in & 7) == 0) && (((uintptr_t)in & 15) == 0);
    const int li = lane & 15, lq = lane >> 4;
    f32x4_t acc[CB][JB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int jb = 0; jb < JB; jb++) acc[cb][jb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    constexpr int rp = JB * 16;
    const int tr = threadIdx.x >> 3, tch = threadIdx.x & 7;           // In slice: 32 rows x CB x 8 chunks of 8
    const int sr = threadIdx.x / (rp / 8), sch = threadIdx.x % (rp / 8);  // S slice: 32 rows x rp/8 chunks
    int buf = 0;
    for (int m0 = row_begin; m0 < row_end; m0 += 128) {
        uint4 vin[4][CB], vs[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int r = m0 + 32 * u + tr;
            const int src = r < row_end ? p.in_rows.source(r) : 0;
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                const int tcc = c0 + cb * 64 + tch * 8;
                vin[u][cb] = load8g(in + (int64_t)src * p.ld_in + tcc, r < row_end ? p.c - tcc : 0, vec);
            }
            vs[u] = make_uint4(0, 0, 0, 0);
            if (sr < 32 && m0 + 32 * u + sr < row_end) {
                const int64_t row = m0 + 32 * u + sr;
                vs[u] = *(const uint4*)(p.s + row * rp + sch * 8);
                if (p.s_weights) {
                    const int64_t wi = p.s_weight_index[row];
                    // (routing weights act at bf16 precision everywhere on the path)
                    const float w = p.s_weights_are_bf16 ? bf16_to_f32(((const bf16_t*)p.s_weights)[wi]) : bf16_to_f32(to_bf16(((const float*)p.s_weights)[wi]));
                    vs[u] = make_uint4(pack_bf16(bf16_lo(vs[u].x) * w, bf16_hi(vs[u].x) * w), pack_bf16(bf16_lo(vs[u].y) * w, bf16_hi(vs[u].y) * w),
                                       pack_bf16(bf16_lo(vs[u].z) * w, bf16_hi(vs[u].z) * w), pack_bf16(bf16_lo(vs[u].w) * w, bf16_hi(vs[u].w) * w));
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (m0 + 32 * u >= row_end) break;  // uniform over the workgroup
#pragma unroll
            for (int cb = 0; cb < CB; cb++) *(uint4*)&in_t[buf][tr][cb * 64 + tch * 8] = vin[u][cb];
            if (sr < 32) *(uint4*)&s_t[buf][sr][sch * 8] = vs[u];
            // one barrier per slice: the slice after the next reuses this buffer, and every wave passes the
            // next barrier only after its reads of this one
            __syncthreads();
            // B operand (n = factor column j, contraction m): source lane s = li points at contraction row
            // 8*lq + s/4 (+4 for the second read), factor columns 4*(s%4) .. +3 of the block's 16
            bf16x8_t b[JB];
#pragma unroll
            for (int jb = 0; jb < JB; jb++) {
                const bf16_t* b_src = &s_t[buf][8 * lq + (li >> 2)][jb * 16 + (li & 3) * 4];
                const v4i16_t b_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)b_src);
                const v4i16_t b_hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(b_src + 4 * kSPitch));
                b[jb] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(b_lo, b_hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
            // A operand (row = column c, contraction m): the same pattern over the wave's 16 columns of block cb
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                const bf16_t* a_src = &in_t[buf][8 * lq + (li >> 2)][cb * 64 + wave * 16 + (li & 3) * 4];
                const v4i16_t a_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)a_src);
                const v4i16_t a_hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(a_src + 4 * kPitch));
                const bf16x8_t a = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a_lo, a_hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                for (int jb = 0; jb < JB; jb++) acc[cb][jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[jb], acc[cb][jb], 0, 0, 0);
            }
            buf ^= 1;
        }
    }
    // acc[cb][jb][v]: c = c0 + 64*cb + wave*16 + 4*lq + v, j = 16*jb + li
    const int64_t ctot = (int64_t)p.nseg * p.c;
    if (splits > 1) {  // unscaled fp32 partial sums [split][column][r_pad]; factor_reduce_kernel finishes
        float* part = p.partials + (int64_t)split * ctot * rp;
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int c = c0 + 64 * cb + wave * 16 + 4 * lq + v;
                    if (c < p.c) part[((int64_t)seg * p.c + c) * rp + jb * 16 + li] = acc[cb][jb][v];
                }
        return;
    }
    bf16_t* out = p.out + (int64_t)e * p.out_expert_elems;
    const bool vec4 = (ctot & 3) == 0 && (((uintptr_t)out & 7) == 0);
    const bool vec8 = (p.r & 7) == 0 && (((uintptr_t)out & 15) == 0);
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        const int cw0 = c0 + 64 * cb + wave * 16;  // first column of this wave's block
        if (p.out_j_major) {
            // [r][columns]: a lane holds four consecutive columns of factor row j: one 8-byte store
#pragma unroll
            for (int jb = 0; jb < JB; jb++) {
                const int j = jb * 16 + li, c = cw0 + 4 * lq;
                if (j >= p.r) continue;
                bf16_t* dst = out + (int64_t)j * ctot + (int64_t)seg * p.c + c;
                if (vec4 && c + 3 < p.c) {
                    *(uint2*)dst = make_uint2(pack_bf16(acc[cb][jb][0] * p.scale, acc[cb][jb][1] * p.scale), pack_bf16(acc[cb][jb][2] * p.scale, acc[cb][jb][3] * p.scale));
                } else {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (c + v < p.c) dst[v] = to_bf16(acc[cb][jb][v] * p.scale);
                }
            }
        } else if (vec8) {
            // [columns][r]: the wave's 16 columns x r are one contiguous run; transpose through LDS (each wave
            // reads back only what it wrote; LDS serves a wave in order) and store 16 bytes per lane
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int v = 0; v < 4; v++) g_t[wave][4 * lq + v][jb * 16 + li] = to_bf16(acc[cb][jb][v] * p.scale);
            const int chunks_per_row = p.r >> 3;
            bf16_t* dst = out + ((int64_t)seg * p.c + cw0) * p.r;
            for (int id = lane; id < 16 * chunks_per_row; id += 64) {
                const int row = id / chunks_per_row, ch = id - row * chunks_per_row;
                const uint4 piece = *(const uint4*)&g_t[wave][row][ch * 8];
                if (cw0 + row < p.c) *(uint4*)(dst + (int64_t)id * 8) = piece;
            }
        } else {
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int c = cw0 + 4 * lq + v, j = jb * 16 + li;
                    if (c < p.c && j < p.r) out[((int64_t)seg * p.c + c) * p.r + j] = to_bf16(acc[cb][jb][v] * p.scale);
                }
        }
    }
}


// Columns of a workgroup, workgroups and row splits of a launch (set in p); false when it is empty.
inline int factor_grad_col_blocks(const FactorGradParams& p) {
    const int cols = p.c % 128 == 0 ? 128 : 64;  // wide column blocks (256 contiguous bytes per row and workgroup) when they divide the segment
    return p.nseg * ((p.c + cols - 1) / cols);
}
inline int64_t factor_grad_plan(FactorGradParams& p, int r_pad, int64_t experts) {
    const int col_blocks = factor_grad_col_blocks(p);
    // One row range for everything (a dense layer) leaves only the column blocks to spread over the compute units: deal
    // the rows out as well, enough to give every unit a workgroup, in shares of at least 128 rows.
    p.row_splits = 1;
    if (!p.ranges && experts == 1 && p.partials && col_blocks < 256 && p.m >= 256) {
        const int64_t want = (256 + col_blocks - 1) / col_blocks;
        const int64_t fit = p.partials_bytes / ((int64_t)p.nseg * p.c * r_pad * 4);
        int64_t splits = want < p.m / 128 ? want : p.m / 128;
        splits = splits < fit ? splits : fit;
        p.row_splits = (int)(splits < 1 ? 1 : splits > 64 ? 64 : splits);
    }
    // Units go to the XCDs in contiguous runs.  An expert's column blocks follow one another, so that one L2 sees whole rows; but
    // rows gathered through an index are read once per route of a token, and a matrix that exceeds an L2 (4 MB) then comes
    // through the fabric that many times.  There the experts follow one another, block after block: an XCD reads a column block
    // once and finds it in its L2 for the other routes.  4096 x 2048, 8 routes a token, both gradients: 72.2 -> 66.8 us; 2048 x
    // 4096: 80.5 -> 74.7; a matrix of 4 MB loses, 36.9 -> 39.6.
    p.blocks_outer = p.in_rows.on() && (int64_t)p.in_rows.index_rows * p.c * 2 > (6 << 20);
    const int64_t units = experts * col_blocks * p.row_splits;
    p.units = (int)units;
    return units;
}

}  // namespace ggq
