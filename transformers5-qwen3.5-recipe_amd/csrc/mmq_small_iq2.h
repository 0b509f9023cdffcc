// IQ2_XXS forward ("NT") kernel for expert groups of a few dozen rows, in which the waves that issue the MFMAs decode the
// packed weights themselves.
//
//   C[m, n] = sum_k A[m, k] * W[n, k]  (+ s * LA[m, :] . LB[n, :])
//
// With 64 rows per expert a decoded weight feeds two 32-row MFMA blocks: there is too little matrix work per weight to hide
// a producer / consumer pipeline behind (decode -> LDS store -> barrier -> LDS read), and that chain paces the tile kernel.
// Here a workgroup is 512 lanes = eight waves and computes tiles of up to 128 rows x 256 columns; wave w owns the 32 columns
// at 32 w.  Per contraction step of 64
//   * the A tile (rows x 128 bytes) goes global -> LDS directly, three steps ahead (two for 97 rows and more), through a ring of
//     four (three) stages (rows unpadded with XOR-swizzled 16-byte slots, a_slot);
//   * once per block (four steps) a wave asks for the 66 bytes of each of its 32 columns, as the five aligned 16-byte chunks that cover
//     them, into its own part of LDS; a step before the block begins a lane (column lane % 32, half h = lane / 32) takes its runs
//     2 step + h and the block's scale out of it into registers, and the next block is asked for into the same place;
//   * a lane decodes its run's 32 weights in registers (selectors of Fmt<kIQ2_XXS> and words of signs in LDS, read two groups of 8
//     weights ahead of their use) and feeds group i of the run to MFMA i of the step: an MFMA sums its 16 contraction slots in any
//     order, so the lane half reads the matching 16-byte slot (4 h + i) of the A row.  No decoded weight touches LDS.
// All requests of the loop are inline-asm loads the compiler does not track, in a fixed order, waited for with exact counts (vector
// memory operations complete in issue order).
// The workgroup keeps 77 KB of LDS (73 KB dynamic, the tables static) and at most 128 registers per lane (the rest, 364 bytes per lane,
// is spilled outside the contraction loops), so two workgroups share a compute unit and cover each other's barriers.  The weights are
// the MFMA's first operand, so a lane's accumulator registers hold four consecutive columns of one row; a finished row block goes
// through a wave-private LDS block (in the ring, idle by then) and leaves as 64-byte row pieces, the LoRA term added there.
//
// What bounds it: requests, decoding and MFMAs add up rather than overlap.  256 experts, 2 x 2048 rows of W, k 4096, 64 rows each:
// 740 us; with eight bytes per lane and step asked for straight into registers (a request of 32 cache lines) 797, with four words
// of signs per group read from a table besides 810.  4096 rows of W, k 2048: 413, 465, 471.
#pragma once
#include "mmq_direct.h"

namespace ggq {

// The signs of a group of eight weights as ONE word, from the seven-bit field that codes them (the eighth is the parity of the other
// seven): pair j's two are at bits 15 and 31 after j doublings.
struct Iq2Signs {
    static __device__ __forceinline__ uint32_t word(uint32_t s7) {
        const uint32_t s = s7 | ((uint32_t)(__builtin_popcount(s7) & 1) << 7);
        uint32_t w = 0;
        for (int j = 0; j < 4; j++) w |= ((s >> (2 * j)) & 1u) << (15 - j) | ((s >> (2 * j + 1)) & 1u) << (31 - j);
        return w;
    }
    // (instructions of full rate: a left shift and v_and_or take twice as long)
    static __device__ __forceinline__ uint32_t flip(uint32_t x, uint32_t flips) {  // x ^ (flips & 0x80008000)
        uint32_t o;
        asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x78" : "=v"(o) : "v"(x), "v"(flips), "s"(0x80008000u));
        return o;
    }
    static __device__ __forceinline__ uint32_t twice(uint32_t x) {
        uint32_t o;
        asm("v_add_u32 %0, %1, %1" : "=v"(o) : "v"(x));
        return o;
    }
};

struct SmallIq2 {
    static constexpr int kTableWords = 256 * 4 + 128;  // the selectors of Fmt<kIQ2_XXS>, then Iq2Signs::word of every field
    static constexpr int kTM = kSmallBM, kTN = kSmallBN;
    static constexpr int kWaves = 8;
    static constexpr int kThreadsWG = 64 * kWaves;
    static constexpr int kRingBytes = 48 * 1024;                                    // A: 4 stages of up to 96 rows or 3 of 128, 128 bytes each
    static constexpr int kLaBase = kRingBytes;                                      // then the row tile's LA rows, 32 bytes each
    static constexpr int kPackedBase = kLaBase + kTM * 32;                          // then a block of every column per wave, as five 16-byte chunks
    static constexpr int kPackedPitch = 80, kPackedBytes = 32 * kPackedPitch;
    static constexpr int kLdsBytes = kPackedBase + kWaves * kPackedBytes + 16;      // 48 + 4 + 20 = 72 KB of dynamic LDS (a run's third dword may lie past the last block)
    // (the decoder's tables, 4.5 KB, are a static array: it sits at LDS address 0, which the compiler then folds into the lookups)
    static constexpr int kOutBase = 0;  // eight 2 KB staging blocks of the epilogue: over the ring, which a finished tile no longer needs

    using RowCtx = Direct::RowCtx;

    template <int LIVE>
    static __device__ __forceinline__ void work(const MmqParams& p, const RowCtx& c, int ct0, int ct1, uint32_t* table_words) {
        extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int lane_c = lane & 31, lane_h = lane >> 5;
        const int steps = p.steps_per_seg;  // a multiple of 4: the contraction is a whole number of 256-wide blocks
        const int out_cols = p.n;
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem_raw;
        for (int i = tid; i < kTableWords; i += kThreadsWG) table_words[i] = i < 1024 ? Fmt<kIQ2_XXS>::table_word(i, d_iq2xxs_grid_mm[i >> 2]) : Iq2Signs::word(i - 1024);
        // the first 16 rank columns of the row tile's LA rows stay in LDS for all the column tiles of this workgroup
        if (p.r_pad > 0) {
            for (int id = tid; id < LIVE * 64; id += kThreadsWG) {
                const int row = id >> 1, half = id & 1;
                *(uint4*)(smem_raw + kLaBase + row * 32 + half * 16) = *(const uint4*)(p.la + (int64_t)(c.row_begin + min(row, c.rows_valid - 1)) * p.r_pad + half * 8);
            }
        }
        __syncthreads();
        // A tile loads: the workgroup's one instruction fills slots tid: tile row tid / 8, slot tid % 8.  Rows past the
        // group's end repeat its last row (their results are never stored).  With a row index the lane offsets carry the
        // whole stored row (the host keeps the matrix under 4 GiB).
        const bf16_t* const a_base = p.a[0] + (p.a_rows.on() ? 0 : (int64_t)c.row_begin * p.lda);
        constexpr int NA = (LIVE + 1) / 2;  // instructions per step: 64 rows each, the last of an odd number of row blocks 32
        constexpr int kStages = LIVE < 4 ? 4 : 3, D = kStages - 1, kStageBytes = LIVE * 4096;  // (D steps ahead)
        static_assert(kStages * kStageBytes <= kRingBytes, "");
        uint32_t a_voff[NA];
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const bool half = 2 * i + 1 >= LIVE;
            const int r = 64 * i + (half ? 4 * wave + ((lane & 31) >> 3) : tid >> 3), s = tid & 7;
            const int kc = s ^ ((r >> 1) & 7);
            const int rr = min(r, c.rows_valid - 1);
            const int src = p.a_rows.on() ? p.a_rows.source(c.row_begin + rr) : rr;
            a_voff[i] = (uint32_t)(((int64_t)src * p.lda + kc * 8) * 2);
        }
        auto issue_a = [&](int step, int stage) __attribute__((always_inline)) {
            const uint32_t dst = lds_base + stage * kStageBytes;
#pragma unroll
            for (int i = 0; i < NA; i++) {
                if (2 * i + 1 < LIVE) load16_to_lds(dst + i * 8192 + wave * 1024, a_voff[i], a_base + min(step, steps - 1) * 64);
                else if (lane_h == 0) load16_to_lds(dst + i * 8192 + wave * 512, a_voff[i], a_base + min(step, steps - 1) * 64);
            }
        };
        auto tile_origin = [&](int ct, int& seg, int& col0) __attribute__((always_inline)) {
            seg = ct / p.col_tiles_per_seg;
            col0 = (ct - seg * p.col_tiles_per_seg) * kTN;
        };
        // LDS read addresses: block rb is tile rows 32 rb + lane_c; MFMA i of a step reads contraction elements
        // 32 h + 8 i .. + 7 of the step: chunk 4 h + i
        const uint8_t* const a_row = smem_raw + lane_c * 128;
        const int a_koff0 = a_slot(lane_c, 4 * lane_h) * 16;  // chunk 4 h + i sits at this offset ^ 16 i

        f32x16_t acc[LIVE];
        for (int ct = ct0; ct < ct1; ct++) {
#pragma unroll
            for (int i = 0; i < LIVE; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][e] = 0.0f;
            int seg, col0;
            tile_origin(ct, seg, col0);
            // The packed rows: a block (66 bytes, at any even address) of each of the wave's 32 columns, as the five aligned chunks that
            // cover it, into the wave's own part of LDS (columns past the end repeat the last one; their results are never stored)
            const uint8_t* const plane = (seg ? p.w[1] : p.w[0]) + c.expert * p.w_expert_bytes;
            const uint32_t lead = (uint32_t)((uintptr_t)plane & 15);
            const uint8_t* const w_base = plane - lead;
            const int blocks = steps >> 2;
            auto column = [&](int r) __attribute__((always_inline)) { return lead + (uint32_t)min(col0 + 32 * wave + r, out_cols - 1) * (uint32_t)p.w_row_bytes; };  // (unsigned: a weight plane may pass 2 GiB)
            uint32_t w_voff[3];
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const int chunk = 64 * j + (j < 2 ? lane : lane & 31), row = chunk / 5;
                w_voff[j] = column(row) + 16 * (chunk - 5 * row);
            }
            auto issue_w = [&](int block) __attribute__((always_inline)) {
                const uint32_t at = 66u * min(block, blocks - 1), dst = lds_base + kPackedBase + wave * kPackedBytes;
                load16_to_lds(dst, (w_voff[0] + at) & ~15u, w_base);
                load16_to_lds(dst + 1024, (w_voff[1] + at) & ~15u, w_base);
                if (lane_h == 0) load16_to_lds(dst + 2048, (w_voff[2] + at) & ~15u, w_base);
            };
            // this lane's runs 2 s + h of its column's block, and the block's scale: they leave LDS a step before the block begins
            const uint32_t own_column = column(lane_c);
            uint32_t q[4][2], d_cur = 0, d_next;
            auto read_block = [&](int block) __attribute__((always_inline)) {
                const uint32_t at = kPackedBase + wave * kPackedBytes + lane_c * kPackedPitch + ((own_column + 66u * min(block, blocks - 1)) & 15u);
                const uint32_t run = at + 2 + 8 * lane_h;
                const uint32_t* const words = (const uint32_t*)(smem_raw + (run & ~3u));
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const uint32_t w0 = words[4 * s], w1 = words[4 * s + 1], w2 = words[4 * s + 2];
                    q[s][0] = __builtin_amdgcn_alignbyte(w1, w0, run), q[s][1] = __builtin_amdgcn_alignbyte(w2, w1, run);  // (its low two bits: 0 or 2)
                }
                d_next = *(const uint16_t*)(smem_raw + at);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the block's bytes are in registers: the next may land
            };
            // The order every step keeps: [A of step t + D], and the last step of a block then asks for the block after the next.  The
            // requests ahead of the loop follow the same order.
            issue_w(0);
#pragma unroll
            for (int t = 0; t < D; t++) issue_a(t, t);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D * NA) : "memory");
            read_block(0);
            issue_w(1);
            // Table reads run two groups of 8 weights ahead of the MFMAs, over the step boundaries too: the selectors and sign
            // words of the first two groups of step 0 are asked for here.
            const uint4* const sel = (const uint4*)table_words;
            const uint32_t* const signs = table_words + 1024;
            uint32_t cur_idx = q[0][0], cur_aux = q[0][1];
            uint4 e[2];     // selectors and signs of the next two groups
            uint32_t f[2];
            auto ask = [&](int slot, int l) __attribute__((always_inline)) {
                e[slot] = sel[(cur_idx >> (8 * l)) & 0xFFu], f[slot] = signs[(cur_aux >> (7 * l)) & 127u];
            };
            ask(0, 0);
            ask(1, 1);
            int rd = 0;  // (three stages: the step's)
            for (int t0 = 0; t0 < steps; t0 += 4) {
                auto step = [&](auto s_c) __attribute__((always_inline)) {
                    constexpr int S = decltype(s_c)::value;
                    // A step needs its A stage, requested D steps back: the A requests of the D - 1 steps since may still be on their
                    // way, and the packed block's three if one of the last D steps ended a block.  Behind the barrier every wave's
                    // part of the stage has landed, and every wave is done reading the stage of the step before, which this step's
                    // request overwrites.  In the last step of a block the next one's packed bytes, requested four steps back, have
                    // landed with it.
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * NA + (S < (D == 3 ? 3 : 2) ? 3 : 0)) : "memory");
                    lds_barrier();
                    const int stage = kStages == 4 ? S : rd;
                    issue_a(t0 + S + D, kStages == 4 ? (S + D) & 3 : rd == 0 ? 2 : rd - 1);
                    if (kStages == 3) rd = rd == 2 ? 0 : rd + 1;
                    if (S == 0) d_cur = d_next;
                    if (S == 3) {
                        read_block((t0 >> 2) + 1);
                        issue_w((t0 >> 2) + 2);
                    }
                    const float db = half_bits_to_f32(d_cur & 0xFFFFu) * (0.5f + (float)(cur_aux >> 28)) * 0.25f;
                    // the three products a weight can be, as bf16: bytes 0..5 of {hi : lo}
                    const uint32_t lo = pack_bf16(db * 8.0f, db * 25.0f), hi = pack_bf16(db * 43.0f, 0.0f);
                    const uint8_t* src = a_row + stage * kStageBytes;
                    // the step's scale leaves cur_aux here: group 2 below moves the next run's words in
                    constexpr int kFirst = LIVE < 4 ? LIVE : 2;  // (four row blocks: the A operands come in two halves, for registers)
                    constexpr bool kAhead = LIVE <= 2;           // (few row blocks: the A operands of a group are read during the group before)
                    bf16x8_t a[kFirst], a_next[kFirst];
                    if (kAhead) {
#pragma unroll
                        for (int rb = 0; rb < kFirst; rb++) a_next[rb] = *(const bf16x8_t*)(src + a_koff0 + rb * 32 * 128);
                    }
#pragma unroll
                    for (int l = 0; l < 4; l++) {
                        if (kAhead) {
#pragma unroll
                            for (int rb = 0; rb < kFirst; rb++) a[rb] = a_next[rb];
                            if (l < 3) {
#pragma unroll
                                for (int rb = 0; rb < kFirst; rb++) a_next[rb] = *(const bf16x8_t*)(src + (a_koff0 ^ (16 * (l + 1))) + rb * 32 * 128);
                            }
                        } else {
#pragma unroll
                            for (int rb = 0; rb < kFirst; rb++) a[rb] = *(const bf16x8_t*)(src + (a_koff0 ^ (16 * l)) + rb * 32 * 128);
                        }
                        u32x4_t w;
                        uint32_t flips = f[l & 1];
                        w[0] = Iq2Signs::flip(__builtin_amdgcn_perm(hi, lo, e[l & 1].x), flips);
                        flips = Iq2Signs::twice(flips);
                        w[1] = Iq2Signs::flip(__builtin_amdgcn_perm(hi, lo, e[l & 1].y), flips);
                        flips = Iq2Signs::twice(flips);
                        w[2] = Iq2Signs::flip(__builtin_amdgcn_perm(hi, lo, e[l & 1].z), flips);
                        flips = Iq2Signs::twice(flips);
                        w[3] = Iq2Signs::flip(__builtin_amdgcn_perm(hi, lo, e[l & 1].w), flips);
                        // the slot is free: the group two ahead, which from group 2 on belongs to the next step's run
                        if (l == 2) cur_idx = q[(S + 1) & 3][0], cur_aux = q[(S + 1) & 3][1];
                        ask(l & 1, (l + 2) & 3);
                        const bf16x8_t b = __builtin_bit_cast(bf16x8_t, w);
#pragma unroll
                        for (int rb = 0; rb < kFirst; rb++) acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a[rb], acc[rb], 0, 0, 0);
                        if (LIVE == 4) {
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int rb = 0; rb < 2; rb++) a[rb] = *(const bf16x8_t*)(src + (a_koff0 ^ (16 * l)) + (rb + 2) * 32 * 128);
#pragma unroll
                            for (int rb = 0; rb < 2; rb++) acc[rb + 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a[rb], acc[rb + 2], 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                step(std::integral_constant<int, 0>{});
                step(std::integral_constant<int, 1>{});
                step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{});
            }
            asm volatile("" ::"v"(e[0].x), "v"(f[0]), "v"(e[1].x), "v"(f[1]));  // (the table reads past the last step)
            // every request has landed (the ones past the last step repeat it); every wave is done with the ring
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            lds_barrier();
            // ---- LoRA term and store.  A lane holds four consecutive columns of one row: acc[rb][i] is tile row
            // 32 rb + lane_c, column 32 wave + 8 (i / 4) + 4 h + (i % 4): a row block goes out as 64-byte row pieces.
            const int64_t ldc = p.ldc;
            bf16_t* const cbase = (bf16_t*)(seg ? p.c[1] : p.c[0]);
            const int rows_valid = c.rows_valid;
            const int col_quad = col0 + 32 * wave + 4 * lane_h;  // first column of this lane's quad at i / 4 = 0
            const bool vec = ((ldc & 7) == 0) && ((((uintptr_t)cbase) & 15) == 0) && col0 + kTN <= out_cols;
            const int nl = p.r_pad >> 4;  // LoRA sub-steps (0: no LoRA)
            const float ls = nl > 0 ? p.lora_scale : 0.0f;
            const bf16_t* const lb_lane = p.lb + c.expert * p.lb_expert_elems + ((int64_t)seg * out_cols + min(col0 + 32 * wave + lane_c, out_cols - 1)) * p.r_pad + lane_h * 8;
            bf16x8_t lb0;  // this lane's row of the LoRA factor B (first 16 of the rank)
            if (nl > 0) lb0 = *(const bf16x8_t*)lb_lane;
            uint8_t* const stage = smem_raw + kOutBase + wave * 2048;
#pragma unroll
            for (int rb = 0; rb < LIVE; rb++) {
                const int row = 32 * rb + lane_c;
                f32x16_t t;  // LB . LA^T for this row block
#pragma unroll
                for (int e = 0; e < 16; e++) t[e] = 0.0f;
                if (nl > 0) {
                    const bf16_t* la = p.la + (int64_t)(c.row_begin + min(row, rows_valid - 1)) * p.r_pad + lane_h * 8;
                    const bf16x8_t la0 = *(const bf16x8_t*)(smem_raw + kLaBase + row * 32 + lane_h * 16);
                    t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lb0, la0, t, 0, 0, 0);
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
                        *(uint2*)(stage + lane_c * 64 + ((g ^ ((lane_c >> 2) & 3)) * 16) + 8 * lane_h) = make_uint2(pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]));
                    }
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int r = 16 * i + (lane >> 2), ch = (lane & 3) ^ ((r >> 2) & 3);
                        const uint4 v = *(const uint4*)(stage + r * 64 + (lane & 3) * 16);
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
                __builtin_amdgcn_sched_barrier(0);
            }
            // the stores count among the outstanding vector memory operations: gone before the next tile's requests are
            // counted; and every wave is done with its staging block before the next tile's requests land in the ring
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (ct + 1 < ct1) lds_barrier();
        }
    }

    // Work assignment: a unit is a run of up to col_tiles_per_wg column tiles of one row tile; the units of a row tile
    // (which share its A rows) follow one another on one XCD.
    static __device__ __forceinline__ void run(const MmqParams& p) {
        const int col_tiles = p.nseg * p.col_tiles_per_seg;
        const int chunks = (col_tiles + p.col_tiles_per_wg - 1) / p.col_tiles_per_wg;
        const int row_tiles = p.tiles ? min(*p.num_tiles, p.max_row_tiles) : p.max_row_tiles;
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
        // the decoder's tables: the kernel's one static LDS array, so it sits at LDS address 0 and the lookups need no base
        __shared__ __attribute__((aligned(16))) uint32_t table_words[kTableWords];
        switch ((c.rows_valid + 31) >> 5) {
            case 1: work<1>(p, c, ct0, ct1, table_words); break;
            case 2: work<2>(p, c, ct0, ct1, table_words); break;
            case 3: work<3>(p, c, ct0, ct1, table_words); break;
            default: work<4>(p, c, ct0, ct1, table_words); break;
        }
    }
};

__global__ __launch_bounds__(SmallIq2::kThreadsWG) __attribute__((amdgpu_waves_per_eu(4, 4))) void mmq_small_iq2xxs_kernel(const MmqParams p) {
    SmallIq2::run(p);
}

}  // namespace ggq
