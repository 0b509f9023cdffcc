// Rank-r LoRA side kernels (r <= 64) around the packed-weight tile kernel.  All are HBM-bound streams
// over the activations; they use the 16x16x32 bf16 MFMA so the arithmetic never shows.
//
//   skinny_nt      out[m, j]  = sum_c In[m, c] * F[e][j, c]          (x A^T,  dY B via B^T)
//   factor_grad    G[e][c, j] = s * sum_{m in group e} In[m, c] * S[m, j]   (dB, dA; fixed order, no atomics)
//   pad / transpose helpers that lay the factors out [cols][r_pad] for the tile kernel.
#include <algorithm>
#include "factor_grad.h"
#include "launch.h"
#include "mmq_host.h"

namespace ggq {

// ---- out[m, 0..r_pad) = In[m, :] . F[e][0..r, :]^T.  One workgroup per 16 rows; its four waves deal the
// contraction out in 128-wide trips (trip t to wave t % 4), so a 64-row tile keeps sixteen waves of loads
// in flight, and add their partial sums through LDS in wave order (fixed order: deterministic).
// In may be two column segments (pair): contraction runs over seg 0 then seg 1, F rows are [r][nseg*C].
template <int JB>  // JB = r_pad / 16
__global__ __launch_bounds__(256) void skinny_nt_kernel(SkinnyNtParams p) {
    __shared__ float red[3][JB][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // Workgroup ids go round-robin over the eight XCDs; give every XCD a contiguous run of units, so the
    // workgroups that share one expert's factor rows share an L2 as well.
    const int units = 4 * (p.tiles ? *p.num_tiles : (int)(gridDim.x >> 2));
    const int per_xcd = (units + 7) >> 3;
    const int slot = blockIdx.x >> 3;
    if (slot >= per_xcd) return;
    const int unit = (blockIdx.x & 7) * per_xcd + slot;
    if (unit >= units) return;
    const int tile = unit >> 2, sub = unit & 3;
    int group = 0, row_begin, row_end;
    if (p.tiles) {
        const TileDesc t = p.tiles[tile];
        group = t.group, row_begin = t.row_begin, row_end = t.row_end;
    } else {
        row_begin = tile * 64;
        row_end = min(p.m, row_begin + 64);
    }
    const int64_t expert = p.expert_ids ? p.expert_ids[group] : 0;
    const int m0 = row_begin + sub * 16;
    if (m0 >= row_end) return;  // uniform over the workgroup
    const int li = lane & 15, lq = lane >> 4;
    const int row = m0 + li;
    const bool row_ok = row < row_end;
    const int src_row = row_ok ? p.in_rows.source(row) : 0;  // stored row of segment 0 (an index comes with one segment)
    const bf16_t* f = p.f + expert * p.f_expert_elems;  // [r][ldf]
    f32x4_t acc[JB];
#pragma unroll
    for (int jb = 0; jb < JB; jb++) acc[jb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const bool fvec = ((p.ldf & 7) == 0) && ((p.c & 7) == 0) && (((uintptr_t)p.f & 15) == 0);
    bool vec = (p.ld_in & 7) == 0;
    for (int seg = 0; seg < p.nseg; seg++) vec = vec && (((uintptr_t)p.in[seg] & 15) == 0);
    // aligned operands: 128-wide trips, every load of a trip issued ahead of its MFMAs
    const int trips_per_seg = (vec && fvec) ? p.c / 128 : 0;
    for (int t = wave; t < trips_per_seg * p.nseg; t += 4) {
        const int seg = t / trips_per_seg, c0 = (t - seg * trips_per_seg) * 128;
        const bf16_t* in = p.in[seg] + (int64_t)src_row * p.ld_in;
        uint4 av[4], bv[JB][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int cc = c0 + 32 * u + lq * 8;
            av[u] = row_ok ? *(const uint4*)(in + cc) : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int jb = 0; jb < JB; jb++) {
                const int j = jb * 16 + li;
                bv[jb][u] = j < p.r ? *(const uint4*)(f + (int64_t)j * p.ldf + seg * p.c + cc) : make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
                acc[jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av[u]), __builtin_bit_cast(bf16x8_t, bv[jb][u]), acc[jb], 0, 0, 0);
    }
    // what the trips leave (and everything, for unaligned operands): 32-wide steps dealt the same way
    int step = 0;
    for (int seg = 0; seg < p.nseg; seg++) {
        const bf16_t* in = p.in[seg] + (int64_t)src_row * p.ld_in;
        for (int c0 = trips_per_seg * 128; c0 < p.c; c0 += 32, step++) {
            if ((step & 3) != wave) continue;
            const int cc = c0 + lq * 8;
            const uint4 av = load8g(in + cc, row_ok ? p.c - cc : 0, vec);
            const bf16x8_t a = __builtin_bit_cast(bf16x8_t, av);
#pragma unroll
            for (int jb = 0; jb < JB; jb++) {
                const int j = jb * 16 + li;
                const uint4 bv = load8g(f + (int64_t)j * p.ldf + seg * p.c + cc, j < p.r ? p.c - cc : 0, fvec);
                acc[jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8_t, bv), acc[jb], 0, 0, 0);
            }
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int jb = 0; jb < JB; jb++)
#pragma unroll
            for (int v = 0; v < 4; v++) red[wave - 1][jb][v][lane] = acc[jb][v];
    }
    __syncthreads();
    if (wave > 0) return;
    // acc[jb][v]: row = m0 + 4*lq + v, col = 16*jb + li
#pragma unroll
    for (int jb = 0; jb < JB; jb++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float sum = ((acc[jb][v] + red[0][jb][v][lane]) + red[1][jb][v][lane]) + red[2][jb][v][lane];
            const int r = m0 + 4 * lq + v;
            if (r < row_end) p.out[(int64_t)r * (JB * 16) + jb * 16 + li] = to_bf16(sum);
        }
}

// ---- The same product for aligned operands with a contraction that is a multiple of 64: every byte
// goes global -> LDS directly in whole 128-byte row pieces (a lane-per-row register load of the MFMA
// operand layout costs the vector cache one access per lane; these loads cost one per 64 bytes), and the
// operands are read back from LDS.  One workgroup per 64-row tile; wave w owns rows 32*(w&1)..+31 and
// every second 64-wide contraction step (parity w>>1), with a two-stage ring of its own: no workgroup
// barrier inside the loop.  Rows keep their 16-byte chunks XOR-swizzled (a_slot) so both the 1 KB writes
// and the operand reads are bank-conflict free.
// FNAT: the factor is given as [contraction][r] (r a multiple of 8, the natural layout of B for dY . B): a
// 64-wide step of it is one contiguous run, copied as it is; the operand reads transpose it on the way out
// of LDS (ds_read_b64_tr_b16: within 16 lanes, lane L gets element L % 4 of the 8 bytes addressed by lanes
// L / 4 + 4 t, t = 0..3, so source lane s points at contraction row s / 4, factor columns 4 (s % 4) .. +3).
template <int JB, bool FNAT>
__global__ __launch_bounds__(256) void skinny_nt_direct_kernel(SkinnyNtParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t sk_lds[];
    constexpr int kInBytes = 32 * 128, kFBytes = JB * 16 * 128, kStage = kInBytes + kFBytes;
    const int f_loads = FNAT ? p.r >> 3 : 2 * JB;  // 1 KB direct-to-LDS instructions per stage of the factor
    const int loads = 4 + f_loads;                 // ... and of the stage
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int units = p.tiles ? *p.num_tiles : (p.m + 63) / 64;
    const int per_xcd = (units + 7) >> 3;
    const int slot = blockIdx.x >> 3;
    if (slot >= per_xcd) return;
    const int unit = (blockIdx.x & 7) * per_xcd + slot;
    if (unit >= units) return;
    int group = 0, row_begin, row_end;
    if (p.tiles) {
        const TileDesc t = p.tiles[unit];
        group = t.group, row_begin = t.row_begin, row_end = t.row_end;
    } else {
        row_begin = unit * 64;
        row_end = min(p.m, row_begin + 64);
    }
    const int64_t expert = p.expert_ids ? p.expert_ids[group] : 0;
    const int half = wave & 1, parity = wave >> 1;
    const int r0 = row_begin + 32 * half;
    const int rows_valid = row_end - r0;  // <= 0: this wave only joins the final barrier
    const bf16_t* f = p.f + expert * p.f_expert_elems;  // [r][ldf], or [nseg*C][r] (FNAT)
    uint8_t* my = sk_lds + wave * 2 * kStage;
    const uint32_t my_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)my;
    // lane's 16 bytes in each 8-row load: row lane/8 of the load, the chunk that belongs in slot lane%8
    uint32_t in_off[4], f_off[2 * JB];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int rl = 8 * q + (lane >> 3);
        int row = min(rl, rows_valid - 1);  // rows past the tile are copies of its last row, never stored
        if (p.in_rows.on()) row = rows_valid > 0 ? p.in_rows.source(r0 + row) : 0;  // the whole stored row (matrix under 4 GiB)
        in_off[q] = ((uint32_t)row * (uint32_t)p.ld_in + (uint32_t)(a_slot(rl, lane & 7) * 8)) * 2u;
    }
#pragma unroll
    for (int q = 0; q < 2 * JB; q++) {
        if (FNAT) {
            f_off[q] = (uint32_t)(q * 64 + lane) * 16u;  // a straight copy
        } else {
            const int jl = 8 * q + (lane >> 3);
            const int j = min(jl, p.r - 1);  // factor rows past the rank are masked when the operand is read
            f_off[q] = ((uint32_t)j * (uint32_t)p.ldf + (uint32_t)(a_slot(jl, lane & 7) * 8)) * 2u;
        }
    }
    const int steps_per_seg = p.c / 64, steps = steps_per_seg * p.nseg;
    auto issue = [&](int step, int stage) {
        const int seg = step / steps_per_seg, c0 = (step - seg * steps_per_seg) * 64;
        const bf16_t* in_base = p.in[seg] + (p.in_rows.on() ? 0 : (int64_t)r0 * p.ld_in) + c0;
        const bf16_t* f_base = FNAT ? f + ((int64_t)seg * p.c + c0) * p.r : f + seg * p.c + c0;
        const uint32_t lds = my_lds + stage * kStage;
#pragma unroll
        for (int q = 0; q < 4; q++) load16_to_lds(lds + q * 1024, in_off[q], in_base);
#pragma unroll
        for (int q = 0; q < 2 * JB; q++)
            if (q < f_loads) load16_to_lds(lds + kInBytes + q * 1024, f_off[q], f_base);
    };
    const int li = lane & 15, lq = lane >> 4;
    f32x4_t acc[2][JB];
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int jb = 0; jb < JB; jb++) acc[rb][jb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (rows_valid > 0) {
        if (parity < steps) issue(parity, 0);
        int stage = 0;
        for (int step = parity; step < steps; step += 2, stage ^= 1) {
            if (step + 2 < steps) {
                issue(step + 2, stage ^ 1);
                wait_loads_at_most(loads);
            } else {
                wait_loads_at_most(0);
            }
            const uint8_t* st = my + stage * kStage;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                uint4 b[JB];
#pragma unroll
                for (int jb = 0; jb < JB; jb++) {
                    const int j = jb * 16 + li;
                    if (FNAT) {
                        const uint8_t* src = st + kInBytes + (kk * 32 + 8 * lq + (li >> 2)) * (p.r * 2) + jb * 32 + (li & 3) * 8;
                        const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)src);
                        const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(src + 4 * (p.r * 2)));
                        b[jb] = __builtin_bit_cast(uint4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                    } else {
                        b[jb] = *(const uint4*)(st + kInBytes + j * 128 + a_slot(j, kk * 4 + lq) * 16);
                    }
                    if (j >= p.r) b[jb] = make_uint4(0, 0, 0, 0);
                }
#pragma unroll
                for (int rb = 0; rb < 2; rb++) {
                    const int rl = rb * 16 + li;
                    const uint4 a = *(const uint4*)(st + rl * 128 + a_slot(rl, kk * 4 + lq) * 16);
#pragma unroll
                    for (int jb = 0; jb < JB; jb++)
                        acc[rb][jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b[jb]), acc[rb][jb], 0, 0, 0);
                }
            }
            // the next trip's loads overwrite the other stage only; this stage is rewritten one trip later,
            // after these reads have returned (the MFMAs above waited for them)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    }
    // the odd-parity waves hand their sums to the even ones through the (now idle) ring
    __syncthreads();
    float* red = (float*)(sk_lds + (wave & 1) * 2 * kStage);  // the ring of wave (w&1): its loads are done
    if (parity == 1) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int jb = 0; jb < JB; jb++)
#pragma unroll
                for (int v = 0; v < 4; v++) red[((rb * JB + jb) * 4 + v) * 64 + lane] = acc[rb][jb][v];
    }
    __syncthreads();
    if (parity == 1) return;
    // acc[rb][jb][v]: row = r0 + 16*rb + 4*lq + v, col = 16*jb + li
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int jb = 0; jb < JB; jb++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float sum = acc[rb][jb][v] + red[((rb * JB + jb) * 4 + v) * 64 + lane];
                const int r = r0 + 16 * rb + 4 * lq + v;
                if (r < row_end) p.out[(int64_t)r * (JB * 16) + jb * 16 + li] = to_bf16(sum);
            }
}

template <int JB, int CB>
__global__ __launch_bounds__(256) void factor_grad_kernel(FactorGradParams p) {
    __shared__ __attribute__((aligned(16))) FactorGradLds<JB, CB> lds;
    // contiguous runs of (expert, column block) units per XCD: one L2 sees whole rows of an expert
    const int per_xcd = ((int)gridDim.x + 7) >> 3;
    const int unit = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || unit >= p.units) return;
    factor_grad_body<JB, CB>(p, unit, lds);
}

// out = bf16(scale * sum over the row splits, in split order) of the partial sums of split factor_grad launches, one or two of
// them (blockIdx.y).  One lane per (column, j < r_pad); lanes of a wave run along j, then columns: contiguous reads.
struct FactorReduceParams {
    const float* partials[2];
    bf16_t* out[2];
    int64_t ctot[2];
    int splits[2], out_j_major[2];
    int r, r_pad;
    float scale;
};
__global__ __launch_bounds__(256) void factor_reduce_kernel(FactorReduceParams p) {
    const int w = blockIdx.y;
    const int64_t total = p.ctot[w] * p.r_pad;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t c = i / p.r_pad;
        const int j = (int)(i - c * p.r_pad);
        if (j >= p.r) continue;
        float sum = 0.f;
        for (int sp = 0; sp < p.splits[w]; sp++) sum += p.partials[w][(int64_t)sp * total + i];
        p.out[w][p.out_j_major[w] ? (int64_t)j * p.ctot[w] + c : c * p.r + j] = to_bf16(sum * p.scale);
    }
}

// dst[e][c][0..r_pad) = src[e][c][0..r) zero padded   (transpose = false, src [E][C][r])
// dst[e][c][0..r_pad) = src[e][0..r)[c] zero padded   (transpose = true,  src [E][r][C])
// One lane per (e, c): its r_pad outputs are contiguous (16-byte stores); with transpose the reads of a
// wave are 64 consecutive columns of one factor row.
__global__ __launch_bounds__(256) void pad_factor_kernel(const bf16_t* src, bf16_t* dst, int64_t experts, int c, int r, int r_pad, int transpose) {
    const int64_t total = experts * c;
    for (int64_t ec = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; ec < total; ec += (int64_t)gridDim.x * blockDim.x) {
        const int cc = (int)(ec % c);
        const int64_t e = ec / c;
        for (int j0 = 0; j0 < r_pad; j0 += 8) {
            uint32_t v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int j = j0 + i;
                v[i] = j < r ? (uint32_t)(transpose ? src[(e * r + j) * c + cc] : src[ec * r + j]) : 0u;
            }
            *(uint4*)(dst + ec * r_pad + j0) = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
        }
    }
}

// dst[e][j][c] = src[e][c][j]  for j < r  (B [E][C][r] -> B^T [E][r][C]).  One lane per (e, c): it reads
// its r contiguous inputs and a wave writes 64 consecutive columns of each output row.
__global__ __launch_bounds__(256) void transpose_factor_kernel(const bf16_t* src, bf16_t* dst, int64_t experts, int c, int r) {
    const int64_t total = experts * c;
    const bool vec = (r & 7) == 0 && (((uintptr_t)src & 15) == 0);
    for (int64_t ec = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; ec < total; ec += (int64_t)gridDim.x * blockDim.x) {
        const int cc = (int)(ec % c);
        const int64_t e = ec / c;
        for (int j0 = 0; j0 < r; j0 += 8) {
            uint32_t w[4] = {0u, 0u, 0u, 0u};
            if (vec) {
                const uint4 q = *(const uint4*)(src + ec * r + j0);
                w[0] = q.x, w[1] = q.y, w[2] = q.z, w[3] = q.w;
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (j0 + i < r) w[i >> 1] |= (uint32_t)src[ec * r + j0 + i] << (16 * (i & 1));
            }
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (j0 + i < r) dst[(e * r + j0 + i) * c + cc] = (bf16_t)(w[i >> 1] >> (16 * (i & 1)));
        }
    }
}

static inline unsigned grid_for(int64_t total, int block) {
    int64_t g = (total + block - 1) / block;
    return (unsigned)(g < 1 ? 1 : (g > 65535 * 16 ? 65535 * 16 : g));
}

int pad_factor(const bf16_t* src, bf16_t* dst, int64_t experts, int c, int r, int r_pad, bool transpose, hipStream_t s) {
    const int64_t total = experts * c;
    if (total == 0) return 0;
    hipLaunchKernelGGL(pad_factor_kernel, dim3(grid_for(total, 256)), dim3(256), 0, s, src, dst, experts, c, r, r_pad, transpose ? 1 : 0);
    return check_launch("pad_factor");
}

int transpose_factor(const bf16_t* src, bf16_t* dst, int64_t experts, int c, int r, hipStream_t s) {
    const int64_t total = experts * c;
    if (total == 0) return 0;
    hipLaunchKernelGGL(transpose_factor_kernel, dim3(grid_for(total, 256)), dim3(256), 0, s, src, dst, experts, c, r);
    return check_launch("transpose_factor");
}

template <int JB, bool FNAT>
static int launch_skinny_direct(const SkinnyNtParams& p, int grid_tiles, hipStream_t s) {
    constexpr int kSmem = 4 * 2 * (32 * 128 + JB * 16 * 128);
    static LdsLimit lds_limit;  // per instantiation
    if (int rc = raise_lds_limit(lds_limit, (const void*)skinny_nt_direct_kernel<JB, FNAT>, kSmem, "skinny_nt")) return rc;
    hipLaunchKernelGGL((skinny_nt_direct_kernel<JB, FNAT>), dim3(((unsigned)grid_tiles + 7u) & ~7u), dim3(256), kSmem, s, p);
    return check_launch("skinny_nt_direct");
}

// The factor may be handed over as [contraction][r] (f_natural) when this holds; otherwise the caller
// passes it transposed, [r][contraction].
bool skinny_nt_takes_natural_factor(const SkinnyNtParams& p) {
    bool ok = (p.r & 7) == 0 && (p.ld_in & 7) == 0 && (p.c & 63) == 0 && ((uintptr_t)p.f & 15) == 0 && (p.f_expert_elems & 7) == 0 &&
              (uint64_t)64 * (uint64_t)p.ld_in * 2 < (1ull << 31);
    for (int seg = 0; seg < p.nseg; seg++) ok = ok && ((uintptr_t)p.in[seg] & 15) == 0;
    return ok;
}

int skinny_nt(const SkinnyNtParams& p, int r_pad, int grid_tiles, hipStream_t s) {
    if (grid_tiles <= 0) return 0;
    bool direct = (p.ld_in & 7) == 0 && (p.ldf & 7) == 0 && (p.c & 63) == 0 && ((uintptr_t)p.f & 15) == 0 && (p.f_expert_elems & 7) == 0 &&
                  (uint64_t)64 * (uint64_t)p.ld_in * 2 < (1ull << 31) && (uint64_t)64 * (uint64_t)p.ldf * 2 < (1ull << 31);
    for (int seg = 0; seg < p.nseg; seg++) direct = direct && ((uintptr_t)p.in[seg] & 15) == 0;
    if (p.in_rows.on()) {
        if (p.nseg != 1 || p.in_rows.index_div <= 0 || p.in_rows.index_rows <= 0) return set_error(GGQ_ERR_SHAPE, "skinny_nt: a row index needs one segment and a positive divisor and row count");
        direct = direct && (uint64_t)p.in_rows.index_rows * (uint64_t)p.ld_in * 2 < (1ull << 32);
    }
    if (p.f_natural) {
        if (!skinny_nt_takes_natural_factor(p)) return set_error(GGQ_ERR_SHAPE, "skinny_nt: this shape needs the factor transposed");
        switch (r_pad / 16) {
            case 1: return launch_skinny_direct<1, true>(p, grid_tiles, s);
            case 2: return launch_skinny_direct<2, true>(p, grid_tiles, s);
            case 3: return launch_skinny_direct<3, true>(p, grid_tiles, s);
            case 4: return launch_skinny_direct<4, true>(p, grid_tiles, s);
            default: return set_error(GGQ_ERR_SHAPE, "LoRA rank must be between 1 and 64");
        }
    }
    if (direct) {
        switch (r_pad / 16) {
            case 1: return launch_skinny_direct<1, false>(p, grid_tiles, s);
            case 2: return launch_skinny_direct<2, false>(p, grid_tiles, s);
            case 3: return launch_skinny_direct<3, false>(p, grid_tiles, s);
            case 4: return launch_skinny_direct<4, false>(p, grid_tiles, s);
            default: return set_error(GGQ_ERR_SHAPE, "LoRA rank must be between 1 and 64");
        }
    }
    switch (r_pad / 16) {
        case 1: hipLaunchKernelGGL(skinny_nt_kernel<1>, dim3((4u * (unsigned)grid_tiles + 7u) & ~7u), dim3(256), 0, s, p); break;
        case 2: hipLaunchKernelGGL(skinny_nt_kernel<2>, dim3((4u * (unsigned)grid_tiles + 7u) & ~7u), dim3(256), 0, s, p); break;
        case 3: hipLaunchKernelGGL(skinny_nt_kernel<3>, dim3((4u * (unsigned)grid_tiles + 7u) & ~7u), dim3(256), 0, s, p); break;
        case 4: hipLaunchKernelGGL(skinny_nt_kernel<4>, dim3((4u * (unsigned)grid_tiles + 7u) & ~7u), dim3(256), 0, s, p); break;
        default: return set_error(GGQ_ERR_SHAPE, "LoRA rank must be between 1 and 64");
    }
    return check_launch("skinny_nt");
}

template <int CB>
static int launch_factor_grad(const FactorGradParams& p, int r_pad, hipStream_t s) {
    const int64_t grid = ((int64_t)p.units + 7) / 8 * 8;
    switch (r_pad / 16) {
        case 1: hipLaunchKernelGGL((factor_grad_kernel<1, CB>), dim3((unsigned)grid), dim3(256), 0, s, p); break;
        case 2: hipLaunchKernelGGL((factor_grad_kernel<2, CB>), dim3((unsigned)grid), dim3(256), 0, s, p); break;
        case 3: hipLaunchKernelGGL((factor_grad_kernel<3, CB>), dim3((unsigned)grid), dim3(256), 0, s, p); break;
        case 4: hipLaunchKernelGGL((factor_grad_kernel<4, CB>), dim3((unsigned)grid), dim3(256), 0, s, p); break;
        default: return set_error(GGQ_ERR_SHAPE, "LoRA rank must be between 1 and 64");
    }
    return check_launch("factor_grad");
}

int factor_grad_partial(FactorGradParams& p, int r_pad, int64_t experts, hipStream_t s) {
    const int64_t units = factor_grad_plan(p, r_pad, experts);
    if (units <= 0) return 0;
    if (units > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "factor_grad: grid too large");
    return p.c % 128 == 0 ? launch_factor_grad<2>(p, r_pad, s) : launch_factor_grad<1>(p, r_pad, s);
}

int factor_reduce(const FactorGradParams* const* ps, int count, int r_pad, hipStream_t s) {
    FactorReduceParams q{};
    int n = 0;
    int64_t most = 0;
    for (int i = 0; i < count; i++) {
        const FactorGradParams& p = *ps[i];
        if (p.row_splits <= 1) continue;  // its launch wrote the result
        q.partials[n] = p.partials, q.out[n] = p.out, q.ctot[n] = (int64_t)p.nseg * p.c, q.splits[n] = p.row_splits, q.out_j_major[n] = p.out_j_major;
        q.r = p.r, q.r_pad = r_pad, q.scale = p.scale;
        most = std::max(most, q.ctot[n] * r_pad);
        n++;
    }
    if (!n) return 0;
    hipLaunchKernelGGL(factor_reduce_kernel, dim3((unsigned)std::min<int64_t>((most + 255) / 256, 4096), n), dim3(256), 0, s, q);
    return check_launch("factor_reduce");
}

int factor_grad(const FactorGradParams& p_in, int r_pad, int64_t experts, hipStream_t s) {
    FactorGradParams p = p_in;
    if (int rc = factor_grad_partial(p, r_pad, experts, s)) return rc;
    const FactorGradParams* one = &p;
    return factor_reduce(&one, 1, r_pad, s);
}

}  // namespace ggq
