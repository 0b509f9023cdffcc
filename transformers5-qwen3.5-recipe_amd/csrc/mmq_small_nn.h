// Q4_K grad-input ("NN") of expert groups of a few dozen rows:
//
//   C[m, k] = sum_seg sum_n A_seg[m, n] * W_seg[n, k]  (+ s * LA[m, :] . LB[:, k])
//
// The kernel of mmq_direct8_nn.h turns every decoded block through LDS (a lane decodes a weight row, an MFMA operand holds
// eight rows of one column): 8 KB in and out per wave and step of 64 x 32 weights, which 16 to 64 activation rows cannot pay
// for.  Here no decoded weight touches LDS.  A lane holds four adjacent packed bytes of EIGHT weight rows, so it has eight
// contraction rows of four columns and, in the high nibbles, of four more: the two halves of an operand register are two rows
// of one column, and one v_cvt_pk_bf16_f32 that has to be spent anyway puts them together.  The sixteen columns of a
// 16x16x32 MFMA are then every fourth column: lane c = lane % 16 has byte column 4 c + j for operand j, a wave 128 columns
// (half a block's 128 quant bytes, both nibbles), and the quarter lane / 16 takes contraction rows 8 q .. 8 q + 7.
//
// A workgroup is four waves = 512 columns = two adjacent blocks of every weight row (288 contiguous bytes), up to 64 activation
// rows, two of them on a compute unit (210 registers; 168, for a third, spill).  Larger groups are several tiles, each a
// workgroup of its own.  Per step of 32 weight rows
//   * the packed rows and the A tile [64][32] go global -> LDS directly, two steps ahead, through a ring of three stages;
//   * every lane works out one (sub-block scale, min) pair of pairs (one row, one quant group) for all four waves;
//   * a wave reads its dwords and scales, forms its eight operands and issues 8 x (row blocks of 16) MFMAs.
// The LDS layouts are permuted so that all of these reads are free of bank conflicts (raw_chunk, scale_slot, a_slot32).  Sums and
// roundings are those of mmq_direct8_nn.h, in the same order (LoRA ranks up to 32): the same bits.
//
// What bounds it: the packed bytes (302 MB, 50 us) and, at 32 rows and more, the instructions of a step; with all packed rows in
// L2 74 / 87 / 102 us at 16 / 32 / 48 rows.  The call (with dY . B, 9 us) for 256 experts of 5 / 16 / 32 / 48 / 64 rows each: 2 x 512
// rows of W, k 2048: 83 / 86 / 96 / 116 / 130 us, against 126 / 134 / 129 / 159 / 160 on mmq_direct8_nn.h; 2048 rows of W, k 512,
// where it has one workgroup per compute unit: 59 / 60 / 66 / 77 / 84 against 69 / 70 / 70 / 82 / 86.
#pragma once
#include "mmq_direct.h"

namespace ggq {

struct SmallNN {
    static constexpr int kWaves = 4, kThreadsWG = 64 * kWaves;
    static constexpr int kRows = 64, kCols = 512;      // of a tile
    static constexpr int kStages = 3;
    static constexpr int kRawBytes = 32 * 288, kABytes = kRows * 64;
    static constexpr int kScaleBase = kStages * (kRawBytes + kABytes);
    static constexpr int kLdsBytes = kScaleBase + 32 * 8 * 16;  // 43 KB

    // Chunk (16 bytes) of a raw stage that holds piece (0..17) of weight row 8 q + i: rows 8 q + i, q = 0..3, side by side, their
    // pieces turned by two per q, so that the same piece of the four rows falls on four different quarters of the banks.
    static __device__ __forceinline__ int raw_chunk(int i, int q, int piece) {
        const int t = piece + 2 * q;
        return (i * 4 + q) * 18 + (t >= 18 ? t - 18 : t);
    }
    // 16-byte slot of the scales of (weight row r, part = 4 * block + quant group)
    static __device__ __forceinline__ int scale_slot(int r, int part) { return r * 8 + ((part + 2 * (r >> 3)) & 7); }
    // 16-byte slot of contraction chunk q of activation row m: sixteen rows at one chunk cover all banks, and so do four rows each at
    // different chunks
    static __device__ __forceinline__ int a_slot32(int m, int q) { return m * 4 + (q ^ ((0x78 >> (2 * ((m >> 2) & 3))) & 3)); }

    template <int RB>  // blocks of sixteen activation rows
    static __device__ __forceinline__ void work(const MmqParams& p, int64_t expert, int row_begin, int rows_valid, int col_block) {
        extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int l16 = lane & 15, q = lane >> 4;
        const int sps = 2 * p.steps_per_seg, steps = p.nseg * sps;  // steps of 32 weight rows
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem_raw;
        // Requests of a stage, four per wave: its 144 chunks of the raw rows (64 + 64 + 16 lanes) and 16 RB chunks of the A tile
        uint32_t w_voff[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int chunk = 144 * wave + (j < 2 ? 64 * j + lane : 128 + l16), pos = chunk / 18, qq = pos & 3;
            int piece = chunk - 18 * pos - 2 * qq;
            piece += piece < 0 ? 18 : 0;
            w_voff[j] = (uint32_t)(8 * qq + (pos >> 2)) * (uint32_t)p.w_row_bytes + 16u * piece;
        }
        uint32_t a_voff;
        {
            const int chunk = 16 * RB * wave + min(lane, 16 * RB - 1), m = chunk >> 2;
            const int kc = (chunk & 3) ^ ((0x78 >> (2 * ((m >> 2) & 3))) & 3);
            const int rr = m < rows_valid ? m : min(m - rows_valid, rows_valid - 1);  // (rows past the end: never stored)
            const int src = p.a_rows.on() ? p.a_rows.source(row_begin + rr) : rr;
            a_voff = (uint32_t)(((int64_t)src * p.lda + kc * 8) * 2);
        }
        const int64_t a_row0 = p.a_rows.on() ? 0 : (int64_t)row_begin * p.lda;
        const bf16_t* a_src = p.a[0] + a_row0;
        const uint8_t* const w_plane[2] = {p.w[0] + expert * p.w_expert_bytes, p.nseg > 1 ? p.w[1] + expert * p.w_expert_bytes : nullptr};
        const uint8_t* w_src = w_plane[0] + col_block * 144;
        const int64_t w_step = 32 * p.w_row_bytes;
        int left = sps, seg = 0, wr = 0;
        auto request = [&]() __attribute__((always_inline)) {  // the next step's stage (past the last step: the last one again)
            const uint32_t dst = lds_base + wr * (kRawBytes + kABytes);
            load16_to_lds(dst + wave * 2304, w_voff[0], w_src);
            load16_to_lds(dst + wave * 2304 + 1024, w_voff[1], w_src);
            if (lane < 16) load16_to_lds(dst + wave * 2304 + 2048, w_voff[2], w_src);
            if (lane < 16 * RB) load16_to_lds(dst + kRawBytes + wave * (256 * RB), a_voff, a_src);
            wr = wr == kStages - 1 ? 0 : wr + 1;
            if (left > 1) left--, w_src += w_step, a_src += 32;
            else if (seg + 1 < p.nseg) left = sps, seg++, w_src = w_plane[1] + col_block * 144, a_src = p.a[1] + a_row0;
        };
        f32x4_t acc[8][RB];
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++) acc[s][rb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        // LDS addresses: this lane's dword of weight row 8 q + i (+ 1152 i), its scales (+ 128 i), its A operand (+ 1024 rb); the
        // header it takes apart and where its scales go
        const int blk = wave >> 1, half = wave & 1;
        const int raw_at = raw_chunk(0, q, 9 * blk + 1 + 4 * half + (l16 >> 2)) * 16 + (l16 & 3) * 4;
        const uint8_t* const scale_at = smem_raw + kScaleBase + scale_slot(8 * q, 4 * blk + 2 * half + (l16 >> 3)) * 16;
        const int a_at = kRawBytes + a_slot32(l16, q) * 16;
        const int hrow = tid >> 3, part = tid & 7;
        const int hdr_at = raw_chunk(hrow & 7, hrow >> 3, 9 * (part >> 2)) * 16;
        uint8_t* const scale_to = smem_raw + kScaleBase + scale_slot(hrow, part) * 16;
        const int grp_sh = 16 * (part & 1);
        const bool grp_hi = (part & 2) != 0;

        request();
        request();
        int rd = 0;
        for (int st = 0; st < steps; st++) {
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  // all but the newest stage's requests: this step's rows have landed
            lds_barrier();
            request();  // into the stage every wave has just finished with
            const uint8_t* const stage = smem_raw + rd * (kRawBytes + kABytes);
            rd = rd == kStages - 1 ? 0 : rd + 1;
            {   // (scale * 2^24, -min) of the two sub-blocks of one quant group; the odd one's nibbles are read at bits 4..7
                const u32x4_t hdr = *(const u32x4_t*)(stage + hdr_at);
                const float d = half_bits_to_f32(hdr.x & 0xFFFFu) * kMixScale, dmin = -half_bits_to_f32(hdr.x >> 16);
                const uint32_t lo_s = hdr.y & 0x3F3F3F3Fu, lo_m = hdr.z & 0x3F3F3F3Fu;
                const uint32_t hi_s = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u), hi_m = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
                const uint32_t sc = opaque((grp_hi ? hi_s : lo_s) >> grp_sh), mn = opaque((grp_hi ? hi_m : lo_m) >> grp_sh);
                const float4 v = make_float4(d * ubyte0(sc), dmin * ubyte0(mn), d * (1.0f / 16.0f) * ubyte1(sc), dmin * ubyte1(mn));
                *(float4*)scale_to = v;
            }
            uint32_t w[8];
#pragma unroll
            for (int i = 0; i < 8; i++) w[i] = *(const uint32_t*)(stage + raw_at + 1152 * i);
            bf16x8_t a[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++) a[rb] = *(const bf16x8_t*)(stage + a_at + 1024 * rb);
            lds_barrier();  // the scales of all four waves
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                float dl[8], nm[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float2 s = *(const float2*)(scale_at + 128 * i + 8 * hi);
                    dl[i] = s.x, nm[i] = s.y;
                }
#pragma unroll
                for (int odd = 0; odd < 2; odd++) {
                    uint32_t x[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) x[i] = (odd ? w[i] >> 8 : w[i]) & (hi ? 0x00F000F0u : 0x000F000Fu);
                    // byte columns `odd` and `odd` + 2
                    uint32_t o[2][4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        o[0][i] = pack_bf16(mix_lo(x[2 * i], dl[2 * i], nm[2 * i]), mix_lo(x[2 * i + 1], dl[2 * i + 1], nm[2 * i + 1]));
                        o[1][i] = pack_bf16(mix_hi(x[2 * i], dl[2 * i], nm[2 * i]), mix_hi(x[2 * i + 1], dl[2 * i + 1], nm[2 * i + 1]));
                    }
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        const bf16x8_t b = Direct::as_operand(o[u]);
#pragma unroll
                        for (int rb = 0; rb < RB; rb++) acc[4 * hi + odd + 2 * u][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[rb], acc[4 * hi + odd + 2 * u][rb], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);  // (one pair of operands at a time: fewer registers)
                }
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may land in LDS after the workgroup has gone

        // acc[4 hi + j][rb][v]: row 16 rb + l16, column 256 blk + 64 (2 half + q / 2) + 32 hi + 16 (q % 2) + 4 v + j of the tile
        const int col0 = col_block * 256 + 256 * blk + 128 * half;
        if (p.r_pad > 0) {
            const bf16_t* const factor = p.lb + expert * p.lb_expert_elems;  // [rank][k]
            const int c8 = l16 >> 3, cl = (4 * l16) & 31;                     // operand column c of set (hi, j): 64 c8 + 32 hi + cl + j
            const int r = 8 * q;  // this lane's eight ranks of 32
            bf16x8_t la[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                la[rb] = __builtin_bit_cast(bf16x8_t, r < p.r_pad ? *(const uint4*)(p.la + (int64_t)(row_begin + min(16 * rb + l16, rows_valid - 1)) * p.r_pad + r) : make_uint4(0, 0, 0, 0));
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                uint2 f[8];  // four columns of eight ranks (zeros past the rank)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    f[i] = *(const uint2*)(factor + (int64_t)min(r + i, p.lora_rank - 1) * p.k + col0 + 64 * c8 + 32 * hi + cl);
                    if (r + i >= p.lora_rank) f[i] = make_uint2(0, 0);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    uint32_t o[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t e0 = j < 2 ? f[2 * i].x : f[2 * i].y, e1 = j < 2 ? f[2 * i + 1].x : f[2 * i + 1].y;
                        o[i] = (j & 1) ? (e0 >> 16) | (e1 & 0xFFFF0000u) : (e0 & 0xFFFFu) | (e1 << 16);
                    }
#pragma unroll
                    for (int rb = 0; rb < RB; rb++) {
                        const f32x4_t t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Direct::as_operand(o), la[rb], (f32x4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[4 * hi + j][rb][v] = __builtin_fmaf(p.lora_scale, t[v], acc[4 * hi + j][rb][v]);
                    }
                }
            }
        }
        bf16_t* const cbase = (bf16_t*)p.c[0];
        const bool vec = (p.ldc & 7) == 0 && (((uintptr_t)cbase) & 15) == 0;
        const int col = col0 + 64 * (q >> 1) + 16 * (q & 1);  // + 32 hi: this lane's sixteen columns
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const int row = 16 * rb + l16;
            if (row >= rows_valid) continue;
            bf16_t* const dst = cbase + (int64_t)(row_begin + row) * p.ldc + col;
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                uint32_t o[8];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    o[2 * v] = pack_bf16(acc[4 * hi][rb][v], acc[4 * hi + 1][rb][v]);
                    o[2 * v + 1] = pack_bf16(acc[4 * hi + 2][rb][v], acc[4 * hi + 3][rb][v]);
                }
                if (vec) {
                    *(uint4*)(dst + 32 * hi) = make_uint4(o[0], o[1], o[2], o[3]);
                    *(uint4*)(dst + 32 * hi + 8) = make_uint4(o[4], o[5], o[6], o[7]);
                } else {
#pragma unroll
                    for (int e = 0; e < 16; e++) dst[32 * hi + e] = (bf16_t)((e & 1) ? o[e >> 1] >> 16 : o[e >> 1] & 0xFFFFu);
                }
            }
        }
    }

    // A unit is 512 columns of one entry of the row-tile table, of at most 64 rows.
    static __device__ __forceinline__ void run(const MmqParams& p) {
        const int chunks = p.col_tiles_per_seg / 2;
        const int row_tiles = min(*p.num_tiles, p.max_row_tiles);
        const int slot = (int)(blockIdx.x >> 3);
        const int row_tile = (slot / chunks) * 8 + (int)(blockIdx.x & 7), col_block = 2 * (slot % chunks);
        if (row_tile >= row_tiles) return;
        const TileDesc t = p.tiles[row_tile];
        const int rows = min(t.row_end - t.row_begin, kRows);
        if (rows <= 0) return;
        if (rows <= 16) work<1>(p, t.expert, t.row_begin, rows, col_block);
        else if (rows <= 32) work<2>(p, t.expert, t.row_begin, rows, col_block);
        else if (rows <= 48) work<3>(p, t.expert, t.row_begin, rows, col_block);
        else work<4>(p, t.expert, t.row_begin, rows, col_block);
    }
};

__global__ __launch_bounds__(SmallNN::kThreadsWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void mmq_small_nn_q4k_kernel(const MmqParams p) {
    SmallNN::run(p);
}

}  // namespace ggq
