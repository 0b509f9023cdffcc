// IQ2_XXS grad-input ("NN") of expert groups of a few dozen rows, the counterpart of mmq_small_iq2.h:
//
//   C[m, k] = sum_seg sum_n A_seg[m, n] * W_seg[n, k]  (+ s * LA[m, :] . LB[:, k])
//
// As in mmq_small_nn.h no decoded weight touches LDS.  A lane decodes one group of eight columns of EIGHT weight rows: two rows'
// pairs of columns (one byte selection and one sign flip each, as in the forward kernel) become two operand words of one column
// by two more byte selections.  Operand j of a 16x16x32 MFMA has column 32 (c % 4) + 8 (c / 4) + j in its slot c = lane % 16, the quarter lane / 16
// takes contraction rows 8 q .. 8 q + 7: a wave covers 128 columns, half a block.
//
// A workgroup is four waves = 512 columns = two adjacent blocks of every weight row (132 bytes), up to 80 activation rows, two of
// them on a compute unit (256 registers: 160 of accumulators).  The sums are those of the tile kernel (mmq_tile.h) in the same
// order, the LoRA term first: bit for bit the same results (with the term last, 0.03 % of the norm apart).  Per step of 32 weight rows
//   * the packed rows (as the 16-byte chunks that cover them) go global -> LDS four steps ahead, the A tile two steps ahead;
//   * every lane makes two records of the step after the next, one per (row, sub-block of 32): the magnitudes 8, 25, 43 times its
//     scale as bf16, the codebook indexes, the sign fields;
//   * a wave reads its records two pairs of rows ahead, the selectors and signs they name one pair ahead, and issues eight MFMAs per
//     sixteen rows.
//
// What bounds it: LDS (the codebook reads are random: 15 cycles for 64 lanes' 16 bytes, which is why a group's signs are one word,
// doubled from pair to pair, instead of four words of a table: 8 % less at 16 rows) and, beside it, the instructions of two waves per
// SIMD; sixty-four columns per wave and four waves per SIMD take 1.4 times as long.  256 experts, 2 x 2048 rows of W, k 4096: 541 / 660 / 743 /
// 823 us at 16 / 48 / 64 / 72 rows per expert, against 834 / 973 / 991 / 1083 of the tile kernel (with rank 16, the call with dY . B: 569 /
// 685 / 778 / 855 against 866 / 1015 / 1037 / 1128); 4096 rows of W, k 2048: 284 / 335 / 383 / 418 against 423 / 493 / 504 / 549.  Groups of
// more than 80 rows stay there.
#pragma once
#include "mmq_small_iq2.h"

namespace ggq {

struct SmallNNIq2 {
    static constexpr int kWaves = 4, kThreadsWG = 64 * kWaves;
    static constexpr int kBlocks = 5, kRows = 16 * kBlocks, kCols = 512;  // of a tile
    static_assert(kRows == kSmallNNIq2Rows, "table entries");
    static constexpr int kStages = 4;
    static constexpr int kTableBytes = 256 * 16 + 128 * 4;                         // the selectors of Fmt<kIQ2_XXS>, then a word of signs per seven-bit field
    static constexpr int kRawPitch = 144, kRawBytes = 32 * kRawPitch;             // the 16-byte chunks that cover a row's 132 bytes
    static constexpr int kRecBytes = 32 * 16 * 16, kABytes = kRows * 64;
    static constexpr int kRecBase = kTableBytes, kRawBase = kRecBase + kStages * kRecBytes, kABase = kRawBase + kStages * kRawBytes;
    static constexpr int kLdsBytes = kABase + kStages * kABytes;                  // 4.5 + 32 + 18 + 20 KB: two workgroups on a compute unit

    // 16-byte slot of the record of (weight row r, sub-block sb of sixteen): the same sub-blocks of rows r, r + 8, r + 16, r + 24
    // fall on different banks
    static __device__ __forceinline__ int rec_slot(int r, int sb) { return r * 16 + ((sb + 4 * (r >> 3)) & 15); }
    static __device__ __forceinline__ int a_slot32(int m, int q) { return m * 4 + (q ^ ((0x78 >> (2 * ((m >> 2) & 3))) & 3)); }

    // LDS by its address (the workgroup's allocation starts at 0: constant parts of an address become the instruction's offset)
    template <class T>
    static __device__ __forceinline__ __attribute__((address_space(3))) T* lds(uint32_t address) {
        return (__attribute__((address_space(3))) T*)(uintptr_t)address;
    }
    // load16_to_lds of the first LANES lanes (the whole wave is active around it)
    template <int LANES>
    static __device__ __forceinline__ void load16_to_lds_first(uint32_t dst, uint32_t voff, const void* sbase) {
        if constexpr (LANES >= 64) load16_to_lds(dst, voff, sbase);
        else
            asm volatile("s_mov_b32 m0, %0\n\ts_bfm_b64 exec, %3, 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                         : : "s"(dst), "v"(voff), "s"(sbase), "n"(LANES) : "memory");
    }

    template <int RB>  // blocks of sixteen activation rows
    static __device__ __forceinline__ void work(const MmqParams& p, int64_t expert, int row_begin, int rows_valid, int col_block) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int l16 = lane & 15, q = lane >> 4;
        const int groups_per_seg = p.n / 128, groups = p.nseg * groups_per_seg;  // groups of four steps of 32 weight rows
        // Requests of a step: 72 chunks of the packed rows per wave (64 + 8 lanes) and 16 RB chunks of the A tile
        const uint32_t row_bytes = (uint32_t)p.w_row_bytes, piece = 66u * col_block;
        uint32_t w_voff[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int chunk = 72 * wave + (j == 0 ? lane : 64 + (lane & 7)), row = chunk / 9;
            w_voff[j] = (((uint32_t)row * row_bytes + piece) & ~15u) + 16u * (chunk - 9 * row);
        }
        constexpr int NA = (16 * RB + 63) / 64;  // requests
        uint32_t a_voff[NA];
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int chunk = 16 * RB * wave + min(64 * i + lane, 16 * RB - 1), m = chunk >> 2;
            const int kc = (chunk & 3) ^ ((0x78 >> (2 * ((m >> 2) & 3))) & 3);
            const int rr = m < rows_valid ? m : min(m - rows_valid, rows_valid - 1);  // (rows past the end: never stored)
            const int src = p.a_rows.on() ? p.a_rows.source(row_begin + rr) : rr;
            a_voff[i] = (uint32_t)(((int64_t)src * p.lda + kc * 8) * 2);
        }
        const int64_t a_row0 = p.a_rows.on() ? 0 : (int64_t)row_begin * p.lda;
        const uint8_t* const w_plane[2] = {p.w[0] + expert * p.w_expert_bytes, p.nseg > 1 ? p.w[1] + expert * p.w_expert_bytes : nullptr};
        const int64_t w_step = 32 * p.w_row_bytes;
        // cursors of a group's packed rows and of its A columns (past the last group: the last one again)
        struct Cursor {
            const uint8_t* w;
            const bf16_t* a;
            int left, seg;
        };
        auto next_group = [&](Cursor& c) __attribute__((always_inline)) {
            if (c.left > 1) c.left--, c.w += 4 * w_step, c.a += 128;
            else if (c.seg + 1 < p.nseg) c.left = groups_per_seg, c.seg++, c.w = w_plane[1], c.a = p.a[1] + a_row0;
        };
        auto request_w = [&](const uint8_t* src, int slot) __attribute__((always_inline)) {
            const uint32_t dst = kRawBase + slot * kRawBytes + wave * 1152;
            load16_to_lds(dst, w_voff[0], src);
            load16_to_lds_first<8>(dst + 1024, w_voff[1], src);
        };
        auto request_a = [&](const bf16_t* src, int slot) __attribute__((always_inline)) {
            const uint32_t dst = kABase + slot * kABytes + wave * (256 * RB);
            if constexpr (RB < 4) load16_to_lds_first<16 * RB>(dst, a_voff[0], src);
            else {
                load16_to_lds(dst, a_voff[0], src);
                if constexpr (RB > 4) load16_to_lds_first<16 * (RB - 4)>(dst + 1024, a_voff[1], src);
            }
        };
        // This thread's two records of a step: rows 8 wave + q and + 4, sub-block l16.  A run starts two bytes into a dword in the first
        // block of a piece and at a dword in the second.
        uint32_t raw_blk[2], rec_to[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t row = 8 * wave + 4 * j + q;
            raw_blk[j] = opaque(kRawBase + row * kRawPitch + ((row * row_bytes + piece) & 15u) + 66 * (l16 >> 3));
            rec_to[j] = opaque(kRecBase + rec_slot(row, l16) * 16);
        }
        const uint32_t run_shift = l16 < 8 ? 2 : 0;
        const uint32_t run_at[2] = {opaque(raw_blk[0] + 8 * (l16 & 7) + (l16 < 8 ? 0 : 2)), opaque(raw_blk[1] + 8 * (l16 & 7) + (l16 < 8 ? 0 : 2))};
        uint32_t rw[2][4];  // a run's three dwords and its block's scale
        auto read_raw = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int i = 0; i < 3; i++) rw[j][i] = *lds<const volatile uint32_t>(run_at[j] + slot * kRawBytes + 4 * i);  // (volatile: a paired read has no room for the slot's offset)
                rw[j][3] = *lds<const volatile uint16_t>(raw_blk[j] + slot * kRawBytes);
            }
        };
        auto write_records = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t idx = __builtin_amdgcn_alignbyte(rw[j][1], rw[j][0], run_shift), aux = __builtin_amdgcn_alignbyte(rw[j][2], rw[j][1], run_shift);
                const float db = half_bits_to_f32(rw[j][3]) * __builtin_fmaf((float)(aux >> 28), 0.25f, 0.125f);
                const u32x4_t rec = {pack_bf16(db * 8.0f, db * 25.0f), pack_bf16(db * 43.0f, 0.0f), idx, aux};
                *lds<u32x4_t>(rec_to[j] + slot * kRecBytes) = rec;
            }
        };
        f32x4_t acc[8][RB];
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++) acc[s][rb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        // this lane's records: weight rows 8 q + i (+ 256 i bytes), sub-block 4 wave + l16 % 4, of it group l16 / 4 (in this order the four
        // lanes of a row store 64 contiguous bytes: 2 % of the launch at 64 rows)
        const uint32_t rec_at = opaque(kRecBase + rec_slot(8 * q, 4 * wave + (l16 & 3)) * 16);
        const uint32_t idx_rot = (8 * (l16 >> 2) + 28) & 31, sgn_rot = (7 * (l16 >> 2) + 30) & 31;  // (the byte ends up at bit 4, the seven bits at bit 2: entries of 16 and of 4 bytes)
        const uint32_t a_at = opaque(kABase + a_slot32(l16, q) * 16);

        Cursor cw{w_plane[0], p.a[0] + a_row0, groups_per_seg, 0}, ca = cw;
#pragma unroll
        for (int i = 0; i < 3; i++) request_w(cw.w + i * w_step, i);
        request_a(ca.a, 0);
        // acc[j][rb][v]: row 16 rb + l16, column 32 v + 8 q + j of the wave's 128
        const int col0 = col_block * 256 + 128 * wave;
        if (p.r_pad > 0) {  // the LoRA term ahead of the products, as in the tile kernel: the same sums in the same order
            const bf16_t* const factor = p.lb + expert * p.lb_expert_elems + col0 + 32 * (l16 & 3) + 8 * (l16 >> 2);  // [rank][k]; operand column l16 of set 0
#pragma unroll 1
            for (int r0 = 0; r0 < p.r_pad; r0 += 32) {
                const int r = r0 + 8 * q;
                bf16x8_t la[RB];
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
                    la[rb] = __builtin_bit_cast(bf16x8_t, r < p.r_pad ? *(const uint4*)(p.la + (int64_t)(row_begin + min(16 * rb + l16, rows_valid - 1)) * p.r_pad + r) : make_uint4(0, 0, 0, 0));
                uint4 f[8];  // eight columns of eight ranks (zeros past the rank)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    f[i] = *(const uint4*)(factor + (int64_t)min(r + i, p.lora_rank - 1) * p.k);
                    if (r + i >= p.lora_rank) f[i] = make_uint4(0, 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    uint32_t o[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint4 &f0 = f[2 * i], &f1 = f[2 * i + 1];
                        const uint32_t e0 = j < 2 ? f0.x : j < 4 ? f0.y : j < 6 ? f0.z : f0.w, e1 = j < 2 ? f1.x : j < 4 ? f1.y : j < 6 ? f1.z : f1.w;
                        o[i] = __builtin_amdgcn_perm(e1, e0, (j & 1) ? 0x07060302u : 0x05040100u);
                    }
#pragma unroll
                    for (int rb = 0; rb < RB; rb++) acc[j][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Direct::as_operand(o), la[rb], acc[j][rb], 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int rb = 0; rb < RB; rb++) acc[j][rb] *= p.lora_scale;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        read_raw(0);
        write_records(0);
        read_raw(1);
        write_records(1);
        lds_barrier();
        request_w(cw.w + 3 * w_step, 3);
        request_a(ca.a + 32, 1);
        next_group(cw);  // (the packed rows are asked for four steps ahead)
        // Two rows' records; the selectors and sign words they name, one pair of rows ahead of their use
        u32x4_t rec[2], sel[2][2];
        uint32_t lo[2][2], hi[2][2], flips[2][2];
        auto ask_records = [&](int slot, int i2) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 2; r++) rec[r] = *lds<const u32x4_t>(rec_at + slot * kRecBytes + 256 * (2 * i2 + r));
        };
        auto ask_words = [&](int b) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                sel[b][r] = *lds<const u32x4_t>(__builtin_amdgcn_alignbit(rec[r].z, rec[r].z, idx_rot) & 0xFF0u);
                flips[b][r] = *lds<const uint32_t>((__builtin_amdgcn_alignbit(rec[r].w, rec[r].w, sgn_rot) & 0x1FCu) + 4096);
                lo[b][r] = rec[r].x, hi[b][r] = rec[r].y;
            }
        };
        ask_records(0, 0);
        ask_words(0);
        ask_records(0, 1);
        for (int g = 0; g < groups; g++) {
            auto step = [&](int S) __attribute__((always_inline)) {
                // All but the requests of the step before: this step's A tile and the packed rows of the step after the next have
                // landed, in every wave behind the barrier.
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA + 2) : "memory");
                lds_barrier();
                // into stages every wave is done with
                if (S == 2) next_group(ca);
                request_w(cw.w + S * w_step, S);
                request_a(ca.a + 32 * ((S + 2) & 3), (S + 2) & 3);
                read_raw((S + 2) & 3);
                bf16x8_t a[2];
                uint32_t o[8][4];
#pragma unroll
                for (int i2 = 0; i2 < 4; i2++) {
                    const int b = i2 & 1;
                    if (i2 < 3) ask_words(b ^ 1);
                    if (i2 < 2) ask_records(S, i2 + 2);
                    else if (i2 == 2) ask_records((S + 1) & 3, 0);
                    if (i2 == 3) {
#pragma unroll
                        for (int rb = 0; rb < RB && rb < 2; rb++) a[rb] = *lds<const bf16x8_t>(a_at + S * kABytes + 1024 * rb);
                    }
                    uint32_t f0 = flips[b][0], f1 = flips[b][1];
#pragma unroll
                    for (int c = 0; c < 4; c++) {  // two rows of one column side by side
                        const uint32_t w0 = Iq2Signs::flip(__builtin_amdgcn_perm(hi[b][0], lo[b][0], sel[b][0][c]), f0);
                        const uint32_t w1 = Iq2Signs::flip(__builtin_amdgcn_perm(hi[b][1], lo[b][1], sel[b][1][c]), f1);
                        o[2 * c][i2] = __builtin_amdgcn_perm(w1, w0, 0x05040100u);
                        o[2 * c + 1][i2] = __builtin_amdgcn_perm(w1, w0, 0x07060302u);
                        if (c < 3) f0 = Iq2Signs::twice(f0), f1 = Iq2Signs::twice(f1);
                    }
                    if (i2 == 1) write_records((S + 2) & 3);  // of the step after the next
                    __builtin_amdgcn_sched_barrier(0);
                }
                ask_words(0);  // of the next step
                ask_records((S + 1) & 3, 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
#pragma unroll
                    for (int j = 0; j < 8; j++) acc[j][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Direct::as_operand(o[j]), a[rb & 1], acc[j][rb], 0, 0, 0);
                    if (rb + 2 < RB) a[rb & 1] = *lds<const bf16x8_t>(a_at + S * kABytes + 1024 * (rb + 2));
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            if constexpr (RB > 3) {  // (unrolled, the accumulators no longer stay in registers)
#pragma unroll 1
                for (int S = 0; S < 4; S++) step(S);
            } else {
                step(0);
                step(1);
                step(2);
                step(3);
            }
            next_group(cw);
        }
        // (the records and words past the last step; their readers are gone)
        asm volatile("" ::"v"(rec[0].x), "v"(rec[1].x));
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may land in LDS after the workgroup has gone

        bf16_t* const cbase = (bf16_t*)p.c[0];
        const bool vec = (p.ldc & 7) == 0 && (((uintptr_t)cbase) & 15) == 0;
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const int row = 16 * rb + l16;
            if (row >= rows_valid) continue;
            bf16_t* const dst = cbase + (int64_t)(row_begin + row) * p.ldc + col0 + 8 * q;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                uint32_t o[4];
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] = pack_bf16(acc[2 * c][rb][v], acc[2 * c + 1][rb][v]);
                if (vec) *(uint4*)(dst + 32 * v) = make_uint4(o[0], o[1], o[2], o[3]);
                else {
#pragma unroll
                    for (int e = 0; e < 8; e++) dst[32 * v + e] = (bf16_t)((e & 1) ? o[e >> 1] >> 16 : o[e >> 1] & 0xFFFFu);
                }
            }
        }
    }

    // A unit is 512 columns of one entry of the row-tile table, of at most 80 rows.
    static __device__ __forceinline__ void run(const MmqParams& p) {
        const int chunks = p.k / kCols;
        const int row_tiles = min(*p.num_tiles, p.max_row_tiles);
        const int slot = (int)(blockIdx.x >> 3);
        const int row_tile = (slot / chunks) * 8 + (int)(blockIdx.x & 7), col_block = 2 * (slot % chunks);
        if (row_tile >= row_tiles) return;
        for (int i = threadIdx.x; i < 1024 + 128; i += kThreadsWG) *lds<uint32_t>(4 * i) = i < 1024 ? Fmt<kIQ2_XXS>::table_word(i, d_iq2xxs_grid_mm[i >> 2]) : Iq2Signs::word(i - 1024);
        const TileDesc t = p.tiles[row_tile];
        const int rows = min(t.row_end - t.row_begin, kRows);
        if (rows <= 0) return;
        if (rows <= 16) work<1>(p, t.expert, t.row_begin, rows, col_block);
        else if (rows <= 32) work<2>(p, t.expert, t.row_begin, rows, col_block);
        else if (rows <= 48) work<3>(p, t.expert, t.row_begin, rows, col_block);
        else if (rows <= 64) work<4>(p, t.expert, t.row_begin, rows, col_block);
        else work<5>(p, t.expert, t.row_begin, rows, col_block);
    }
};

__global__ __launch_bounds__(SmallNNIq2::kThreadsWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void mmq_small_nn_iq2xxs_kernel(const MmqParams p) {
    SmallNNIq2::run(p);
}

}  // namespace ggq
