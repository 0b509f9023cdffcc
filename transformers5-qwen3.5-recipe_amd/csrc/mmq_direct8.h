// Q4_K forward ("NT") tile kernel in which the waves that issue the MFMAs decode the packed weights themselves.
//
//   C[m, n] = sum_k A[m, k] * W[n, k]  (+ s * LA[m, :] . LB[n, :])
//
// A workgroup is 512 lanes = eight waves, two per SIMD with 256 registers each, and computes tiles of up to 192 rows x
// 256 columns; wave w owns the 32 columns at 32 w of every row: up to six 32-row blocks of MFMA 32x32x16 accumulators.
// The kernel is instantiated per number of live 32-row blocks, so an expert group of any size up to 192 rows is one row
// tile and issues no MFMA on empty blocks.  Per contraction step of 64
//   * the A tile goes global -> LDS directly (no registers), three steps ahead, through a ring of four stages; rows are
//     unpadded with XOR-swizzled 16-byte slots (a_slot), every wave reads all of them;
//   * the packed blocks go global -> LDS directly as well, the whole 144-byte blocks (header and quant bytes, four steps)
//     of the wave's 32 columns at a time, nine adjacent lanes per row, into two wave-private buffers;
//   * a lane reads its 16 quant bytes of the step, and once per block its header, from its wave's buffer and decodes them
//     in registers into the operands of the step's four MFMA sub-steps (mmq_direct.h).  No decoded weight ever touches LDS.
// A single wave issues at most one instruction per four to five cycles, whatever its kind, so a step's decode
// arithmetic, LDS reads, requests and waits (about eight instructions per MFMA) cannot hide behind that wave's own
// MFMAs; with two waves per SIMD one wave's MFMAs run while the other decodes, reads and waits.
// The weights are the MFMA's first operand, so a lane's accumulator registers hold four consecutive columns of one row;
// a finished row block goes through a wave-private LDS block and leaves as 64-byte row pieces.  The LoRA term is added
// there.  A workgroup takes a run of column tiles of its row tile and treats their steps as one stream, so the requests
// of a tile's first steps are in flight while the tile before it finishes.  The requests are inline-asm loads the
// compiler does not track; the step waits for them with exact counts (vector memory operations complete in issue order).
//
// What bounds it: the clock the matrix cores leave (1.9 GHz at 128 rows and more), plus what does not overlap them: 256
// experts, 2 x 512 columns, k 2048 take 88 us at 32 rows each and 22 us for every 32 rows more (302 MB of packed weights: 58
// us at 5.2 TB/s).  Whole-block requests, staging of its own, and cursors that only add: 102 / 88 / 107 / 153 / 182 / 204 us
// at 16 / 32 / 64 / 128 / 160 / 192 rows, before 109 / 95 / 114 / 160 / 187 / 209.
#pragma once
#include "mmq_direct.h"

namespace ggq {

struct Direct8 {
    static constexpr int kTM = kDirectBM, kTN = kDirectBN;
    static constexpr int kWaves = 8;
    static constexpr int kThreadsWG = 64 * kWaves;
    // Packed weights: per wave two buffers of 32 rows x 144 bytes, a block of each of the wave's 32 columns (a row pitch of
    // 144 bytes spreads the lane-per-row reads over all banks); then per wave 2 KB in which a finished row block's output is
    // staged; then the row tile's LA rows (rank <= 16), 32 bytes each; then the A ring.  Six row blocks leave no room for
    // staging: they stage in the packed buffer just read, and request its next contents only behind the store path.
    static constexpr int kWBufBytes = 32 * 144;
    static constexpr int kOutBase = kWaves * 2 * kWBufBytes;               // 72 KB
    static constexpr int kLdsBytes = 160 * 1024 - 4096;  // 156 KB
    template <int LIVE>
    struct Layout {
        static constexpr int kStages = LIVE <= 4 ? 4 : 3;
        static constexpr bool kOwnStaging = LIVE <= 5;
        static constexpr int kLaBase = kOutBase + (kOwnStaging ? kWaves * 2048 : 0), kABase = kLaBase + LIVE * 1024;
    };
    static_assert(kOutBase + kWaves * 2048 + 4 * (1024 + 4 * 4096) <= kLdsBytes && kOutBase + kWaves * 2048 + 5 * (1024 + 3 * 4096) <= kLdsBytes && kOutBase + 6 * (1024 + 3 * 4096) <= kLdsBytes, "LDS");
    using Scales = Direct::Scales;
    using RowCtx = Direct::RowCtx;

    template <int LIVE>
    static __device__ __forceinline__ void work(const MmqParams& p, const RowCtx& c, int ct0, int ct1) {
        extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
        using L = Layout<LIVE>;
        constexpr int kStages = L::kStages, kLaBase = L::kLaBase, kABase = L::kABase;
        constexpr int NI = (LIVE + 1) / 2;       // direct-to-LDS instructions per A stage and wave (the last of an odd block count: half its lanes)
        constexpr int kStageBytes = LIVE * 4096;
        constexpr int kStores = 2 * LIVE - 1;    // 16-byte store instructions a tile certainly issues per wave (two per full row block, one for the last)
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int lane_c = lane & 31, lane_h = lane >> 5;
        const int steps = p.steps_per_seg, blocks = steps >> 2;
        const int out_cols = p.n;
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem_raw;
        // A tile loads: instruction i fills slots 512 i + tid: tile row 64 i + tid / 8, slot tid % 8; the last instruction of
        // an odd block count has half the rows, 32 lanes of every wave.  Rows past the group's end repeat its first rows
        // (their results are never stored; one row repeated by all of them cost 2 % of a launch of 16-row groups).  With a
        // row index the lane offsets carry the whole stored row (the host keeps the matrix under 4 GiB).
        const bf16_t* a_src = p.a[0] + (p.a_rows.on() ? 0 : (int64_t)c.row_begin * p.lda);
        uint32_t a_voff[NI];
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int r = 64 * i + (2 * i + 1 < LIVE ? tid >> 3 : 4 * wave + (lane_c >> 3)), s = tid & 7;
            const int kc = s ^ ((r >> 1) & 7);
            const int rr = r < c.rows_valid ? r : min(r - c.rows_valid, c.rows_valid - 1);
            const int src = p.a_rows.on() ? p.a_rows.source(c.row_begin + rr) : rr;
            a_voff[i] = (uint32_t)(((int64_t)src * p.lda + kc * 8) * 2);
        }
        auto tile_origin = [&](int ct, int& seg, int& col0) __attribute__((always_inline)) {
            seg = ct / p.col_tiles_per_seg;
            col0 = (ct - seg * p.col_tiles_per_seg) * kTN;
        };
        // The A cursor: the next step to request; it only moves the contraction offset, the same way for every column tile.
        const bf16_t* a_next = a_src;
        int a_left = steps;
        int a_wr = 0;  // byte offset of the stage the next request fills
        uint32_t ph_dst;  // the open phase's A stage and source
        const bf16_t* ph_src;
        auto phase_open = [&]() __attribute__((always_inline)) {
            ph_dst = lds_base + kABase + a_wr;
            ph_src = a_next;
            a_wr = a_wr == (kStages - 1) * kStageBytes ? 0 : a_wr + kStageBytes;
            a_next += 64;
            if (--a_left == 0) a_left = steps, a_next = a_src;
        };
        auto request_a = [&](auto i_c) __attribute__((always_inline)) {
            constexpr int I = decltype(i_c)::value;
            if constexpr (2 * I + 1 < LIVE) load16_to_lds(ph_dst + I * 8192 + wave * 1024, a_voff[I], ph_src);
            else if constexpr (2 * I < LIVE) {
                if (lane_h == 0) load16_to_lds(ph_dst + I * 8192 + wave * 512, a_voff[I], ph_src);
            }
        };
        // The W cursor: (column tile, 256-wide block) of the next block to request.  Whole blocks go global -> LDS directly:
        // the 288 16-byte chunks of the wave's 32 blocks in row order, chunk 64 j + lane by instruction j (the fifth moves
        // 32).  What a request costs is the cache lines it touches: a step's blocks as separate headers and quant halves,
        // 16 rows x 64 bytes each, kept the vector cache busy for 204 ns (L2 hits), as whole blocks for 88.
        int w_tile_i = ct0, w_blk = 0;
        const uint8_t* w_next;  // packed row of the cursor tile's first column (scalar)
        uint32_t w_voff[5];     // this lane's byte offset from the cursor's block there in instruction j
        auto w_cursor_rows = [&]() __attribute__((always_inline)) {
            int seg, col0;
            tile_origin(w_tile_i, seg, col0);
            w_next = (seg ? p.w[1] : p.w[0]) + c.expert * p.w_expert_bytes + (int64_t)col0 * p.w_row_bytes;
#pragma unroll
            for (int j = 0; j < 5; j++) {
                const int chunk = j < 4 ? 64 * j + lane : 256 + lane_c, row = chunk / 9;
                w_voff[j] = (uint32_t)min(32 * wave + row, out_cols - 1 - col0) * (uint32_t)p.w_row_bytes + 16u * (chunk - 9 * row);
            }
        };
        w_cursor_rows();
        int w_wr = 0;  // byte offset (inside the wave's pair) of the buffer the open block's requests fill
        const uint32_t w_lds = lds_base + wave * (2 * kWBufBytes);
        auto request_w = [&](auto j_c) __attribute__((always_inline)) {
            constexpr int J = decltype(j_c)::value;
            if constexpr (J < 4) load16_to_lds(w_lds + w_wr + J * 1024, w_voff[J], w_next + w_blk * 144);
            else if (lane_h == 0) load16_to_lds(w_lds + w_wr + J * 1024, w_voff[J], w_next + w_blk * 144);
        };
        auto w_cursor_advance = [&]() __attribute__((always_inline)) {  // past the last block of the last tile the cursor stays
            w_wr ^= kWBufBytes;
            if (w_blk + 1 < blocks) w_blk++;
            else if (w_tile_i + 1 < ct1) w_tile_i++, w_blk = 0, w_cursor_rows();
        };

        f32x16_t acc[LIVE];
        // LDS read addresses: block rb is tile rows 32 rb + lane_c; sub-step I reads chunk 4 (I / 2) + 2 h + (I % 2)
        const uint8_t* a_row = smem_raw + kABase + lane_c * kARowBytes;
        int a_koff[4];
#pragma unroll
        for (int i = 0; i < 4; i++) a_koff[i] = a_slot(lane_c, 4 * (i >> 1) + 2 * lane_h + (i & 1)) * 16;
        bf16x8_t ao[LIVE];
        const uint8_t* const w_row = smem_raw + wave * (2 * kWBufBytes) + lane_c * 144;  // this lane's block (+ 16 + 32 S + 16 h: its quant bytes of step S)
        const int w_q = 16 + 16 * lane_h;
        int w_rd = 0;  // byte offset of the buffer of the current block
        int a_rd = 0;  // byte offset of the A stage of the current step

        u32x4_t qc, qn;  // quant bytes of the current / next step
        u32x4_t hc, hn;  // headers of the current / next block
        auto request_w_block = [&]() __attribute__((always_inline)) {
            request_w(std::integral_constant<int, 0>{}), request_w(std::integral_constant<int, 1>{}), request_w(std::integral_constant<int, 2>{});
            request_w(std::integral_constant<int, 3>{}), request_w(std::integral_constant<int, 4>{});
            w_cursor_advance();
        };
        request_w_block();
#pragma unroll
        for (int i = 0; i < kStages - 1; i++) {
            phase_open();
            request_a(std::integral_constant<int, 0>{}), request_a(std::integral_constant<int, 1>{}), request_a(std::integral_constant<int, 2>{});
        }
        // the first 16 rank columns of the row tile's LA rows stay in LDS for all the column tiles of this workgroup: the
        // epilogue then reads them with LDS reads, which no pending store or request stands in front of
        if (p.r_pad > 0) {
            for (int id = tid; id < LIVE * 64; id += kThreadsWG) {
                const int row = id >> 1, half = id & 1;
                *(uint4*)(smem_raw + kLaBase + row * 32 + half * 16) = *(const uint4*)(p.la + (int64_t)(c.row_begin + min(row, c.rows_valid - 1)) * p.r_pad + half * 8);
            }
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 2) * NI) : "memory");  // the first blocks and the first step's A stage have landed
        lds_barrier();
        hc = *(const u32x4_t*)w_row;
        // Phase p = the last sub-step of step p - 1 and the first three of step p: it reads A stage p only, and its
        // requests (behind the barrier that opens it) fill the stage of step p - 1.  A phase's first A instruction goes
        // out in its first sub-step, the others in the next step's first two.
        request_w_block();  // phase 0: block 1, A of step kStages - 1
        phase_open();
        request_a(std::integral_constant<int, 0>{});
        qc = *(const u32x4_t*)(w_row + w_q);
        Scales sc;
        uint32_t bx[4], by[4];  // B operands of the current / next sub-step
        sc = Direct::chunk_scales<0>(hc);
        Direct::decode_half<0, 0>(qc, sc, bx);
        Direct::decode_half<0, 1>(qc, sc, bx);
#pragma unroll
        for (int rb = 0; rb < LIVE; rb++) ao[rb] = *(const bf16x8_t*)(a_row + a_koff[0] + rb * 32 * kARowBytes);
        // One sub-step, row block by row block: the block's MFMA, then its operand of the following sub-step is read
        // into the registers it has just released, then a half of the decode of the next B operand.
        auto sub_step = [&](const uint32_t* b, int next_stage_off, int next_i, auto&& piece, auto&& request) __attribute__((always_inline)) {
            const uint8_t* src = a_row + next_stage_off + a_koff[next_i];
            const bf16x8_t b0 = Direct::as_operand(b);
#pragma unroll
            for (int rb = 0; rb < LIVE; rb++) {
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b0, ao[rb], acc[rb], 0, 0, 0);
                if (rb == 0) request();  // this sub-step's share of the step's memory requests, behind its first MFMA
                ao[rb] = *(const bf16x8_t*)(src + rb * 32 * kARowBytes);
                if (0 * LIVE / 2 == rb) piece(std::integral_constant<int, 0>{});
                if (1 * LIVE / 2 == rb) piece(std::integral_constant<int, 1>{});
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        bool stores_behind = false;  // the tile before this one went out through the staged store path
        for (int ct = ct0; ct < ct1; ct++) {
#pragma unroll
            for (int i = 0; i < LIVE; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][e] = 0.0f;
            // This lane's row of the LoRA factor B (first 16 of the rank), requested ahead of the tile's steps with a load of
            // the same untracked kind as the other requests (without a LoRA term: 16 bytes of the packed weights, unused).
            // A load the compiler tracks would be waited for at its use in the epilogue with vmcnt(0): behind the next
            // tile's first requests, and behind the stores of the row blocks before it, one round trip each.
            u32x4_t lb0_raw;
            {
                int seg0, colz;
                tile_origin(ct, seg0, colz);
                const void* src = p.r_pad > 0 ? (const void*)(p.lb + c.expert * p.lb_expert_elems + ((int64_t)seg0 * out_cols + min(colz + 32 * wave + lane_c, out_cols - 1)) * p.r_pad + lane_h * 8)
                                              : (const void*)(p.w[0] + c.expert * p.w_expert_bytes);
                asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(lb0_raw) : "v"(src) : "memory");
            }
            if (!L::kOwnStaging && ct > ct0) request_w_block();
            auto block = [&](auto first_c, bool last) __attribute__((always_inline)) {
                constexpr bool FIRST = decltype(first_c)::value;
                // Requests per phase P (= step index % 4): an A stage [NI]; P = 3 and 0: the next block but one, into the buffer
                // whose last quant bytes step 2 has read [3 + 2] (staging in that buffer: behind a tile's last block all of it
                // in phase 0, behind the store path).
                auto step = [&](auto s_c) __attribute__((always_inline)) {
                    constexpr int S = decltype(s_c)::value;
                    // the quant bytes of the next step: of this block, or the first of the next one, with its header
                    if (S == 3) w_rd ^= kWBufBytes;
                    qn = *(const u32x4_t*)(w_row + w_rd + w_q + 32 * ((S + 1) & 3));
                    if (S == 3) hn = *(const u32x4_t*)(w_row + w_rd);
                    const int a_rd_next = a_rd == (kStages - 1) * kStageBytes ? 0 : a_rd + kStageBytes;
                    __builtin_amdgcn_sched_barrier(0);
                    sub_step(bx, a_rd, 1, [&](auto k_c) __attribute__((always_inline)) { Direct::decode_half<1, decltype(k_c)::value>(qc, sc, by); },
                             [&]() __attribute__((always_inline)) { request_a(std::integral_constant<int, 1>{}); });
                    sub_step(by, a_rd, 2, [&](auto k_c) __attribute__((always_inline)) { Direct::decode_half<2, decltype(k_c)::value>(qc, sc, bx); },
                             [&]() __attribute__((always_inline)) { request_a(std::integral_constant<int, 2>{}); });
                    sub_step(bx, a_rd, 3, [&](auto k_c) __attribute__((always_inline)) { Direct::decode_half<3, decltype(k_c)::value>(qc, sc, by); },
                             [&]() __attribute__((always_inline)) {});
                    // End of phase S.  All but the requests of this phase and the one before it have landed: this wave's
                    // part of A stage S + 1 (requested two phases ago) and every packed byte requested before that.  Behind
                    // the barrier every wave's part has, and every wave is done reading stage S, which the next phase's
                    // requests overwrite.  Requests complete in order, so the distance matters: packed bytes come from
                    // HBM, and a wait that covered requests only one step old stalled on them.
                    // (Three stages: A stages are requested one phase later, and only this phase's requests may be outstanding.)
                    // A tile's phase 0 also holds the tile before's stores and the request of the LoRA factor row.
                    constexpr int kTwo = kStages - 3;  // 1: the phase before this one counts, 0: it does not
                    constexpr int kLate = L::kOwnStaging ? 0 : 3;  // packed requests of phase 3 that come in phase 0 at a tile's end
                    constexpr int kGroup[4] = {NI + 2 + (FIRST ? 1 + kLate : 0), NI, NI, NI + 3}, kLastOfTile = NI + 3 - kLate;
                    constexpr int kBehind = kGroup[S] + kTwo * (S == 0 && FIRST ? kLastOfTile : kGroup[(S + 3) & 3]);
                    if (FIRST && (S == 0 || (S == 1 && kTwo))) {
                        if (stores_behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kBehind + kStores) : "memory");
                        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kBehind) : "memory");
                    } else if (S == 3 && kLate && last) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kBehind - kLate) : "memory");
                    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kBehind) : "memory");
                    lds_barrier();
                    phase_open();
                    // behind the last sub-step's MFMAs: the first operand of the next step (of the next tile behind a
                    // tile's last step), with the scales of its quant group
                    sub_step(by, a_rd_next, 0, [&](auto k_c) __attribute__((always_inline)) {
                        constexpr int K = decltype(k_c)::value;
                        if (K == 0) sc = Direct::chunk_scales<(S + 1) & 3>(S == 3 ? hn : hc);
                        Direct::decode_half<0, K>(qn, sc, bx);
                    }, [&]() __attribute__((always_inline)) {
                        const bool here = L::kOwnStaging || !last;
                        if (S == 2 && here) request_w(std::integral_constant<int, 0>{}), request_w(std::integral_constant<int, 1>{}), request_w(std::integral_constant<int, 2>{});
                        if (S == 3 && here) request_w(std::integral_constant<int, 3>{}), request_w(std::integral_constant<int, 4>{}), w_cursor_advance();
                        request_a(std::integral_constant<int, 0>{});
                    });
                    qc = qn;
                    a_rd = a_rd_next;
                };
                step(std::integral_constant<int, 0>{});
                step(std::integral_constant<int, 1>{});
                step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{});
                hc = hn;
            };
            block(std::true_type{}, blocks == 1);
            for (int kb = 1; kb < blocks; kb++) block(std::false_type{}, kb + 1 == blocks);
            // ---- LoRA term and store.  A lane holds four consecutive columns of one row: acc[rb][i] is tile row
            // 32 rb + lane_c, column 32 wave + 8 (i / 4) + 4 h + (i % 4): a row block goes out as 64-byte row pieces.
            // (own, opaque copies of the lane coordinates: none of this part's address arithmetic may be hoisted in
            // front of the tile loop, where it would sit in registers through every main loop)
            int lane_e = lane;
            asm volatile("" : "+v"(lane_e));
            const int lane_ce = lane_e & 31, lane_he = lane_e >> 5;
            int seg, col0;
            tile_origin(ct, seg, col0);
            const int64_t ldc = p.ldc;
            bf16_t* const cbase = (bf16_t*)(seg ? p.c[1] : p.c[0]);
            const int rows_valid = c.rows_valid;
            const int col_quad = col0 + 32 * wave + 4 * lane_he;  // first column of this lane's quad at i / 4 = 0
            const bool vec = ((ldc & 7) == 0) && ((((uintptr_t)cbase) & 15) == 0) && col0 + kTN <= out_cols;
            stores_behind = vec;
            const int nl = p.r_pad >> 4;  // LoRA sub-steps (0: no LoRA)
            const float ls = nl > 0 ? p.lora_scale : 0.0f;
            const bf16_t* const lb_lane = p.lb + c.expert * p.lb_expert_elems + ((int64_t)seg * out_cols + min(col0 + 32 * wave + lane_ce, out_cols - 1)) * p.r_pad + lane_he * 8;
            // (the factor row landed long ago: every step's wait leaves only the requests of two phases outstanding)
            asm volatile("" : "+v"(lb0_raw));
            const bf16x8_t lb0 = __builtin_bit_cast(bf16x8_t, lb0_raw);
            bf16x8_t la0[LIVE];
            if (nl > 0) {
#pragma unroll
                for (int rb = 0; rb < LIVE; rb++)
                    la0[rb] = *(const bf16x8_t*)(smem_raw + kLaBase + (32 * rb + lane_ce) * 32 + lane_he * 16);
            }
            uint8_t* const stage = smem_raw + (L::kOwnStaging ? kOutBase + wave * 2048 : wave * (2 * kWBufBytes) + (w_rd ^ kWBufBytes));
#pragma unroll
            for (int rb = 0; rb < LIVE; rb++) {
                const int row = 32 * rb + lane_ce;
                f32x16_t t;  // LB . LA^T for this row block
#pragma unroll
                for (int e = 0; e < 16; e++) t[e] = 0.0f;
                if (nl > 0) {
                    t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lb0, la0[rb], t, 0, 0, 0);
                    const bf16_t* la = p.la + (int64_t)(c.row_begin + min(row, rows_valid - 1)) * p.r_pad + lane_he * 8;
#pragma nounroll
                    for (int kk = 1; kk < nl; kk++)
                        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8_t*)(lb_lane + kk * 16), *(const bf16x8_t*)(la + kk * 16), t, 0, 0, 0);
                }
                if (vec) {
                    // 8-byte pieces in (the 16-byte chunk g of a row sits at position g ^ (row / 4) % 4), 64-byte row pieces
                    // out; LDS accesses of one wave execute in order, so no wait is needed between the two
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        float o[4];
#pragma unroll
                        for (int j = 0; j < 4; j++) o[j] = __builtin_fmaf(ls, t[4 * g + j], acc[rb][4 * g + j]);
                        *(uint2*)(stage + lane_ce * 64 + ((g ^ ((lane_ce >> 2) & 3)) * 16) + 8 * lane_he) = make_uint2(pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]));
                    }
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int r = 16 * i + (lane_e >> 2), ch = (lane_e & 3) ^ ((r >> 2) & 3);
                        const uint4 v = *(const uint4*)(stage + r * 64 + (lane_e & 3) * 16);
                        if (32 * rb + r < rows_valid) *(uint4*)(cbase + (int64_t)(c.row_begin + 32 * rb + r) * ldc + col0 + 32 * wave + ch * 8) = v;
                    }
                } else if (rb < LIVE - 1 || row < rows_valid) {  // only the last live block can be partial
                    bf16_t* const crow = cbase + (int64_t)(c.row_begin + row) * ldc;
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int col = col_quad + 8 * (i >> 2) + (i & 3);
                        if (col < out_cols) crow[col] = to_bf16(__builtin_fmaf(ls, t[i], acc[rb][i]));
                    }
                }
                __builtin_amdgcn_sched_barrier(0);  // one row block at a time: keeps the register need of this part small
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may land in LDS after the workgroup has gone
    }

    // Work assignment as in the four-wave kernel: a unit is a run of up to col_tiles_per_wg column tiles of one row
    // tile; consecutive units (which share an A tile) stay on one XCD.
    static __device__ __forceinline__ void run(const MmqParams& p) {
        const int col_tiles = p.nseg * p.col_tiles_per_seg;
        const int chunks = (col_tiles + p.col_tiles_per_wg - 1) / p.col_tiles_per_wg;
        const int row_tiles = p.tiles ? min(*p.num_tiles, p.max_row_tiles) : p.max_row_tiles;
        // Row tile rt runs on XCD rt % 8 (the table lists the tiles with the most rows first: every XCD gets its
        // share of them, and takes its own in that order); the column-tile runs of a row tile follow one another there.
        const int slot = (int)(blockIdx.x >> 3);
        const int row_tile = (slot / chunks) * 8 + (int)(blockIdx.x & 7), chunk = slot % chunks;
        if (row_tile >= row_tiles) return;
        RowCtx c;
        int row_end;
        if (p.tiles) {
            const TileDesc t = p.tiles[row_tile];
            c.row_begin = t.row_begin, row_end = t.row_end, c.expert = t.expert;
        } else {
            c.row_begin = row_tile * kTM;
            row_end = min(p.m, c.row_begin + kTM);
            c.expert = 0;
        }
        c.rows_valid = row_end - c.row_begin;
        if (c.rows_valid <= 0) return;  // (the table builders emit no empty tile; a descriptor that is one must not index row -1)
        const int ct0 = chunk * p.col_tiles_per_wg, ct1 = min(col_tiles, ct0 + p.col_tiles_per_wg);
        switch ((c.rows_valid + 31) >> 5) {
            case 1: work<1>(p, c, ct0, ct1); break;
            case 2: work<2>(p, c, ct0, ct1); break;
            case 3: work<3>(p, c, ct0, ct1); break;
            case 4: work<4>(p, c, ct0, ct1); break;
            case 5: work<5>(p, c, ct0, ct1); break;
            default: work<6>(p, c, ct0, ct1); break;
        }
    }
};

__global__ __launch_bounds__(Direct8::kThreadsWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void mmq_direct8_q4k_kernel(const MmqParams p) {
    Direct8::run(p);
}

}  // namespace ggq
