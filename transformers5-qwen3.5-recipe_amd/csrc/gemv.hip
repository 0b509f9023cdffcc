// Products of a few activation rows with packed weights: sampling (one row per sequence) and its expert layers.
//
// What bounds them is the packed bytes: every weight is used by 1 to 64 rows.  A tile of mmq_tile.h pads the rows to 256 and
// gives a 4096-column layer 32 workgroups; here a workgroup takes sixteen weight ROWS (a contiguous run of packed bytes,
// whatever the block format) at a time, moves them global -> LDS in whole 1 KB requests (a lane-per-row register load costs
// the vector cache an access per lane), and its waves decode them from LDS straight into 16x16x32 MFMA operands: lane
// (weight row lane % 16, quarter lane / 16) owns one 32-element run of a 128-element span and feeds its eight-element
// pieces to four MFMAs whose other operand holds the matching pieces of sixteen activation rows, in registers for the
// whole kernel.  The matrix pipe, idle otherwise, does the multiplication, so one row costs what sixteen do.
#include <algorithm>

#include "blocks.h"
#include "iq2xxs_grid.h"
#include "launch.h"
#include "mmq_host.h"

namespace ggq {

static __device__ const uint64_t d_iq2xxs_grid_gemv[256] = GGQ_IQ2XXS_GRID_INIT;

constexpr int kSpan = 128;                 // contraction elements of four runs
template <int QT>
constexpr int kTableBytes = QT == kIQ2_XXS ? Fmt<kIQ2_XXS>::kTableWords * 4 : 0;

template <int QT>
__device__ __forceinline__ void stage_tables(uint8_t* lds, int tid, int threads) {
    if constexpr (QT == kIQ2_XXS)
        for (int i = tid; i < Fmt<kIQ2_XXS>::kTableWords; i += threads) ((uint32_t*)lds)[i] = Fmt<kIQ2_XXS>::table_word(i, i < 1024 ? d_iq2xxs_grid_gemv[i >> 2] : 0ull);
}

__device__ __forceinline__ bf16x8_t as_operand(const uint4& v) { return __builtin_bit_cast(bf16x8_t, v); }
__device__ __forceinline__ f32x4_t mfma16(const bf16x8_t& a, const bf16x8_t& b, const f32x4_t& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Where byte `off` of packed rows lies in LDS.  Q4_K rows of 2048 and 4096 elements are an odd and an even number of 128-byte
// pieces, and the same byte of sixteen rows falls on an eighth of the banks and less: bank conflicts took half of the cycles
// of a launch.  32 bytes left free behind every 1024 put eight rows on eight different eighths.  (Every piece of a Q4_K block that is
// read at once is 16-byte aligned, so none straddles a gap; the other formats' rows spread over the banks as they are, or are read as words.)
template <int QT>
constexpr int kPieceGap = QT == kQ4_K ? 32 : 0;
template <int QT>
__host__ __device__ __forceinline__ int lds_at(int off) { return kPieceGap<QT> ? off + (off >> 10) * kPieceGap<QT> : off; }
__host__ __device__ __forceinline__ int row_block_bytes(int qt, int bytes) {  // LDS bytes of `bytes` of packed rows
    return (bytes + 1023) / 1024 * (1024 + (qt == kQ4_K ? kPieceGap<kQ4_K> : 0));
}

// A run of packed bytes global -> LDS, dealt to the workgroup's waves in 1 KB requests (kGap free bytes behind each); both ends
// 16-byte aligned except for the length, whose odd end (less than 16 bytes) a few lanes carry.  Returns the requests this wave made.
template <int kGap = 0>
__device__ __forceinline__ int request_bytes(const uint8_t* src, uint8_t* dst, int bytes, int wave, int waves, int lane) {
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)dst;
    const int whole = bytes & ~15;
    int made = 0;
    for (int c = wave; c * 1024 < whole; c += waves, made++)
        if (c * 1024 + lane * 16 < whole) load16_to_lds(__builtin_amdgcn_readfirstlane(lds + c * (1024 + kGap)), (uint32_t)lane * 16u, src + c * 1024);
    if (wave == 0 && lane * 2 < bytes - whole) *(uint16_t*)(dst + whole + (whole >> 10) * kGap + lane * 2) = *(const uint16_t*)(src + whole + lane * 2);
    return made;
}

// A run out of packed rows in LDS.  The blocks of most formats are only 2- or 4-byte aligned, and a wide LDS read that is not
// aligned to its width is taken apart by the hardware (reading Q6_K runs with 16-byte reads kept the LDS busy for three
// quarters of the kernel): those formats are read as aligned words, one more than the piece has, and shifted together.
template <int N>
__device__ __forceinline__ void lds_words(const uint8_t* lds, int off, uint32_t* out) {
    const uint32_t* p = (const uint32_t*)(lds + (off & ~3));
    uint32_t w[N + 1];
#pragma unroll
    for (int i = 0; i <= N; i++) w[i] = p[i];
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], off & 3);
}
__device__ __forceinline__ uint32_t lds_half(const uint8_t* lds, int off) { return *(const uint16_t*)(lds + off); }
__device__ __forceinline__ void lds_32_bytes(const uint8_t* lds, int off, uint4& a, uint4& b) {
    uint32_t w[8];
    lds_words<8>(lds, off, w);
    a = make_uint4(w[0], w[1], w[2], w[3]), b = make_uint4(w[4], w[5], w[6], w[7]);
}
// row: byte offset of the row in `lds` (even)
template <int QT>
__device__ __forceinline__ void load_run(typename Fmt<QT>::Raw& r, const uint8_t* lds, int row, int ksub) {
    if constexpr (QT == kQ5_K) {
        Fmt<QT>::load(r, lds + row, ksub);  // whole 16-byte pieces
    } else if constexpr (QT == kQ8_0) {
        const int blk = row + ksub * 34;
        r.d16 = lds_half(lds, blk);
        lds_32_bytes(lds, blk + 2, r.q0, r.q1);
    } else if constexpr (QT == kQ3_K) {
        const int blk = row + (ksub >> 3) * 110, u = ksub & 7, n = u >> 2, g = u >> 1, b = 2 * (u & 1);
        lds_32_bytes(lds, blk, r.h0, r.h1);
        lds_32_bytes(lds, blk + 32 + 32 * n, r.q0, r.q1);
        r.sl = lds_half(lds, blk + 96 + 4 * (g & 1) + b), r.sh = lds_half(lds, blk + 104 + b), r.d16 = lds_half(lds, blk + 108);
    } else {
        const int blk = row + (ksub >> 3) * 66;
        uint32_t w[2];
        r.d16 = lds_half(lds, blk);
        lds_words<2>(lds, blk + 2 + 8 * (ksub & 7), w);
        r.idx4 = w[0], r.aux = w[1];
    }
}

// The sixteen operand words of a lane for one span of a row: words 4 i .. 4 i + 3 go to MFMA i.
//
// Two ways to deal the span's 128 elements to the four lanes of a row.  A contraction may be summed in any order, so each
// format takes the cheaper one and the other operand follows (span_element):
//  * by run (Q8_0, Q3_K, Q5_K, IQ2_XXS): lane q owns run q, MFMA i its elements 8 i .. 8 i + 7;
//  * by position (Q2_K, Q4_K, Q6_K, whose runs share bytes): lane q owns elements 8 q .. 8 q + 7 of all four runs, MFMA i those
//    of run i: every byte is read and taken apart once (Q6_K by run: 64 bytes and 148 vector instructions per lane and span).
template <int QT>
constexpr bool kByPosition = QT == kQ2_K || QT == kQ4_K || QT == kQ6_K;
template <int QT>
__device__ __forceinline__ int span_element(int q, int i) { return kByPosition<QT> ? 32 * i + 8 * q : 32 * q + 8 * i; }

// Four small integers in the bytes of w (the bits of MASK) -> four bf16 of value scale * integer + offset.
template <uint32_t MASK = 0x00FF00FFu>
__device__ __forceinline__ void four_values(uint32_t w, float scale24, float offset, uint32_t* out) {
    // (opaque: taken apart by bytes instead, the two words would be three)
    const uint32_t e02 = opaque(w & MASK), e13 = opaque((w >> 8) & MASK);
    out[0] = pack_bf16(mix_lo(e02, scale24, offset), mix_lo(e13, scale24, offset));
    out[1] = pack_bf16(mix_hi(e02, scale24, offset), mix_hi(e13, scale24, offset));
}

template <int QT>
__device__ __forceinline__ void decode_span(const uint8_t* lds, int row, int span, int runs, int q, uint32_t* v, const uint2* tables) {
    if constexpr (QT == kQ4_K) {
        const int blk = row + (span >> 1) * 144, h = span & 1;
        const uint4 hdr = *(const uint4*)(lds + lds_at<QT>(blk));
        const int low = blk + 16 + 64 * h + 8 * q;
        const uint2 g0 = *(const uint2*)(lds + lds_at<QT>(low)), g1 = *(const uint2*)(lds + lds_at<QT>(low + 32));
        const float d = half_bits_to_f32(hdr.x & 0xFFFFu) * kMixScale, dmin = half_bits_to_f32(hdr.x >> 16);
        // (scale, min) of the four runs, one per byte
        const uint32_t sc = h ? (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u) : hdr.y & 0x3F3F3F3Fu;
        const uint32_t mn = h ? ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u) : hdr.z & 0x3F3F3F3Fu;
        const uint32_t so = opaque(sc), mo = opaque(mn);
        // (the high nibbles of runs 1 and 3 stay in place and are read as sixteen times their value)
        const float d16 = d * 0.0625f;
        const float dl[4] = {d * ubyte0(so), d16 * ubyte1(so), d * ubyte2(so), d16 * ubyte3(so)};
        const float nm[4] = {-(dmin * ubyte0(mo)), -(dmin * ubyte1(mo)), -(dmin * ubyte2(mo)), -(dmin * ubyte3(mo))};
        const uint32_t w[4] = {g0.x, g0.y, g1.x, g1.y};
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t b = w[2 * g + u];
                const uint32_t b8 = b >> 8, lo02 = b & 0x000F000Fu, hi02 = b & 0x00F000F0u, lo13 = b8 & 0x000F000Fu, hi13 = b8 & 0x00F000F0u;
                uint32_t* even = v + 8 * g + 2 * u;
                even[0] = pack_bf16(mix_lo(lo02, dl[2 * g], nm[2 * g]), mix_lo(lo13, dl[2 * g], nm[2 * g]));
                even[1] = pack_bf16(mix_hi(lo02, dl[2 * g], nm[2 * g]), mix_hi(lo13, dl[2 * g], nm[2 * g]));
                even[4] = pack_bf16(mix_lo(hi02, dl[2 * g + 1], nm[2 * g + 1]), mix_lo(hi13, dl[2 * g + 1], nm[2 * g + 1]));
                even[5] = pack_bf16(mix_hi(hi02, dl[2 * g + 1], nm[2 * g + 1]), mix_hi(hi13, dl[2 * g + 1], nm[2 * g + 1]));
            }
    } else if constexpr (QT == kQ6_K) {
        const int blk = row + (span >> 1) * 210, h = span & 1;
        uint32_t a[2], b[2], c[2];
        lds_words<2>(lds, blk + 64 * h + 8 * q, a);
        lds_words<2>(lds, blk + 64 * h + 32 + 8 * q, b);
        lds_words<2>(lds, blk + 128 + 32 * h + 8 * q, c);
        const float d = half_bits_to_f32(lds_half(lds, blk + 208));
        uint32_t sw[2];
        lds_words<2>(lds, blk + 192 + 8 * h, sw);  // the half's eight scales; run i takes scale 2 i + q / 2
        const int sh = (q >> 1) * 8;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float s = d * (float)(int)(int8_t)((sw[i >> 1] >> (16 * (i & 1) + sh)) & 0xFFu);
            const float s24 = s * kMixScale, off = -32.0f * s;
#pragma unroll
            for (int u = 0; u < 2; u++) {
                // low four bits of a byte from one word, the next two from the other (one v_bfi_b32); what is left above them
                // falls to the masks below
                const uint32_t nib = i == 0 ? a[u] : i == 1 ? b[u] : i == 2 ? a[u] >> 4 : b[u] >> 4;
                const uint32_t two = i == 0 ? c[u] << 4 : i == 1 ? c[u] << 2 : i == 2 ? c[u] : c[u] >> 2;
                four_values<0x003F003Fu>((nib & 0x0F0F0F0Fu) | (two & 0xF0F0F0F0u), s24, off, v + 4 * i + 2 * u);
            }
        }
    } else if constexpr (QT == kQ2_K) {
        const uint8_t* blk = lds + row + (span >> 1) * 84;  // (rows and blocks are multiples of four bytes)
        const int n = span & 1;
        const uint32_t* w = (const uint32_t*)(blk + 16 + 32 * n + 8 * q);
        const uint32_t w0 = w[0], w1 = w[1], dd = *(const uint32_t*)(blk + 80);
        const uint32_t* s8 = (const uint32_t*)(blk + 8 * n);  // the half's eight scale bytes; run i takes byte 2 i + q / 2
        const uint32_t sw[2] = {s8[0], s8[1]};
        const int sh = (q >> 1) * 8;
        const float d = half_bits_to_f32(dd & 0xFFFFu) * kMixScale, dmin = half_bits_to_f32(dd >> 16);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t sb = (sw[i >> 1] >> (16 * (i & 1) + sh)) & 0xFFu;
            const float dl = d * (float)(sb & 0xFu), nm = -(dmin * (float)(sb >> 4));
            four_values((w0 >> (2 * i)) & 0x03030303u, dl, nm, v + 4 * i);
            four_values((w1 >> (2 * i)) & 0x03030303u, dl, nm, v + 4 * i + 2);
        }
    } else {
        const int run = min(span * 4 + q, runs - 1);
        typename Fmt<QT>::Raw raw;
        load_run<QT>(raw, lds, row, run);
        Fmt<QT>::decode(raw, run, v, tables);
    }
}

// Eight consecutive factor elements p[0..valid) (zeros past it); vec: 16-byte aligned and whole.
__device__ __forceinline__ uint4 load_factor8(const bf16_t* p, int valid, bool vec) {
    if (vec && valid >= 8) return *(const uint4*)p;
    if (valid <= 0) return make_uint4(0, 0, 0, 0);
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 8; i++) e[i] = i < valid ? (uint32_t)p[i] : 0u;
    return make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
}

// ------------------------------------------------------------------------------------------------
// Dense: y [m, n] = x [m, k] . W [n, k]^T (+ scale (x A^T) B^T).
struct GemvParams {
    const bf16_t* x;
    int64_t ldx;
    int m, n, k;
    const uint8_t* w;               // at a 16-byte address: the matrix starts `head` bytes behind it
    int row_bytes, head;
    bf16_t* y;
    int64_t ldy;
    const bf16_t *lora_a, *lora_b;  // [r][k], [n][r]; null: none
    bf16_t* xa_out;                 // [m][r_pad]
    int r, r_pad;
    float lora_scale;
    int stage_bytes, buffers;       // LDS bytes of sixteen packed rows, one or two of them
};

// WAVES waves deal the spans of the contraction out (span s to wave s % WAVES, at most SP each); TB blocks of sixteen rows of x.
// LORA is a template parameter because a load the compiler tracks may stand nowhere in the block loop of a plain product: on
// whatever path, it makes every iteration wait for all requests, the block requested ahead among them.  (With LORA the row of B
// is such a load: there each request waits for the one before it, and the next block has landed before the current one is multiplied.)
template <int QT, int WAVES, int SP, int TB, bool LORA>  // TB <= WAVES
__global__ __launch_bounds__(64 * WAVES) void gemv_kernel(GemvParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t gemv_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    uint8_t* stage = gemv_lds + kTableBytes<QT>;
    f32x4_t* red = (f32x4_t*)(stage + p.buffers * p.stage_bytes);            // [WAVES][TB][64]
    bf16_t* xa = (bf16_t*)(red + WAVES * TB * 64);                           // [TB * 16][64]
    const int blocks = (p.n + 15) / 16, spans = (p.k + kSpan - 1) / kSpan;
    int block = blockIdx.x;
    auto request_block = [&](int b, int buf) __attribute__((always_inline)) {
        return request_bytes<kPieceGap<QT>>(p.w + (int64_t)b * 16 * p.row_bytes, stage + buf * p.stage_bytes, p.head + min(16, p.n - b * 16) * p.row_bytes, wave, WAVES, lane);
    };
    // (the barriers here order LDS traffic only: __syncthreads would also wait for the block requested ahead)
    // With a LoRA term x and the first sixteen factor rows go out ahead of the packed bytes: requests complete in order, and
    // x A^T is formed while the packed bytes are on their way.  (Where the factor rows of all spans leave the kernel its 128
    // registers, two workgroups per compute unit: else they come span by span.  At 4096 elements 165 registers, and 13.9 -> 16.6 us
    // for one row and 5120 columns of Q6_K.)
    constexpr bool kAhead = LORA && SP * TB <= 2;
    // (a factor is always there with LORA; asked at run time, the compiler keeps to the 128 registers)
    const bool lora = kAhead || (LORA && p.lora_a);
    if (!kAhead && block < blocks) request_block(block, 0);
    uint4 xf[SP][TB][4];
#pragma unroll
    for (int sp = 0; sp < SP; sp++)
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
            const bf16_t* src = p.x + min(tb * 16 + l16, p.m - 1) * p.ldx;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int e = (wave + WAVES * sp) * kSpan + span_element<QT>(q, i);
                xf[sp][tb][i] = e < p.k ? *(const uint4*)(src + e) : make_uint4(0, 0, 0, 0);  // (k is a multiple of 32: eight elements are whole or absent)
            }
        }
    uint4 a[kAhead ? SP : 1][4];
    auto load_a = [&](int r0, int sp, uint4* out) __attribute__((always_inline)) {
        const bf16_t* arow = p.lora_a + (int64_t)min(r0 + l16, p.r - 1) * p.k;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int e = (wave + WAVES * sp) * kSpan + span_element<QT>(q, i);
            out[i] = e < p.k && r0 + l16 < p.r ? *(const uint4*)(arow + e) : make_uint4(0, 0, 0, 0);
        }
    };
    if constexpr (kAhead) {
#pragma unroll
        for (int sp = 0; sp < SP; sp++) load_a(0, sp, a[sp]);
        if (block < blocks) request_block(block, 0);
    }
    stage_tables<QT>(gemv_lds, threadIdx.x, 64 * WAVES);
    if (lora) {  // x A^T over this wave's spans, added over the waves, kept as bf16 rows in LDS
        for (int r0 = 0; r0 < p.r_pad; r0 += 16) {
            f32x4_t acc[TB];
#pragma unroll
            for (int tb = 0; tb < TB; tb++) acc[tb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            if (kAhead && r0 > 0) {
#pragma unroll
                for (int sp = 0; sp < SP; sp++) load_a(r0, sp, a[sp]);
            }
#pragma unroll
            for (int sp = 0; sp < SP; sp++) {
                uint4* const as = a[kAhead ? sp : 0];
                if (!kAhead) load_a(r0, sp, as);
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int tb = 0; tb < TB; tb++) acc[tb] = mfma16(as_operand(as[i]), as_operand(xf[sp][tb][i]), acc[tb]);
            }
#pragma unroll
            for (int tb = 0; tb < TB; tb++) red[(wave * TB + tb) * 64 + lane] = acc[tb];
            lds_barrier();
            for (int tb = wave; tb < TB; tb += WAVES) {
                f32x4_t sum = red[tb * 64 + lane];
                for (int w = 1; w < WAVES; w++) sum += red[(w * TB + tb) * 64 + lane];
                const uint2 v = make_uint2(pack_bf16(sum[0], sum[1]), pack_bf16(sum[2], sum[3]));
                const int row = tb * 16 + l16;  // factor rows r0 + 4 q .. + 3 of x row `row`
                *(uint2*)(xa + row * 64 + r0 + 4 * q) = v;
                if (blockIdx.x == 0 && row < p.m) *(uint2*)(p.xa_out + (int64_t)row * p.r_pad + r0 + 4 * q) = v;
            }
            lds_barrier();
        }
    }
    const bool b_vec = (p.r & 7) == 0 && ((uintptr_t)p.lora_b & 15) == 0;
    const int own_row = p.head + l16 * p.row_bytes;
    for (int buf = 0; block < blocks; block += gridDim.x) {
        const int next = block + gridDim.x;
        if (p.buffers == 2 && next < blocks) wait_loads_at_most(request_block(next, buf ^ 1));
        else wait_loads_at_most(0);
        lds_barrier();
        // the factor rows of the block's LoRA term, for the waves that will add it, ahead of the work they would wait behind
        const bool adds = (wave + block) % WAVES < TB;
        const bf16_t* brow = p.lora_b + (int64_t)min(block * 16 + l16, p.n - 1) * p.r;
        uint4 b0 = make_uint4(0, 0, 0, 0);
        if (lora && adds) b0 = load_factor8(brow + 8 * q, p.r - 8 * q, b_vec);
        f32x4_t acc[TB];
#pragma unroll
        for (int tb = 0; tb < TB; tb++) acc[tb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        const int row = min(own_row, p.head + min(15, p.n - block * 16 - 1) * p.row_bytes);
#pragma unroll
        for (int sp = 0; sp < SP; sp++) {
            const int span = wave + WAVES * sp;
            if (span >= spans) break;  // uniform over the wave
            uint32_t v[16];
            decode_span<QT>(stage + buf * p.stage_bytes, row, span, p.k >> 5, q, v, (const uint2*)gemv_lds);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int tb = 0; tb < TB; tb++)
                    acc[tb] = mfma16(as_operand(make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3])), as_operand(xf[sp][tb][i]), acc[tb]);
        }
#pragma unroll
        for (int tb = 0; tb < TB; tb++) red[(wave * TB + tb) * 64 + lane] = acc[tb];
        lds_barrier();
        if (p.buffers == 1 && next < blocks) request_block(next, 0);
        // (a buffer is refilled, and the partial sums rewritten, only behind the next barrier)
        if (const int tb = (wave + block) % WAVES; adds) {
            f32x4_t sum = red[tb * 64 + lane];
            for (int w = 1; w < WAVES; w++) sum += red[(w * TB + tb) * 64 + lane];
            const int col = block * 16 + 4 * q, xrow = tb * 16 + l16;
            if (lora) {
                f32x4_t lo = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                for (int r0 = 0; r0 < p.r_pad; r0 += 32) {
                    const int j = r0 + 8 * q;
                    const uint4 b = r0 == 0 ? b0 : load_factor8(brow + j, p.r - j, b_vec);
                    const uint4 xv = j < p.r_pad ? *(const uint4*)(xa + xrow * 64 + j) : make_uint4(0, 0, 0, 0);
                    lo = mfma16(as_operand(b), as_operand(xv), lo);
                }
                sum += lo * p.lora_scale;
            }
            if (xrow < p.m) {
                bf16_t* dst = p.y + xrow * p.ldy + col;
                if (((p.n | p.ldy) & 3) == 0 && ((uintptr_t)p.y & 7) == 0) {
                    if (col < p.n) *(uint2*)dst = make_uint2(pack_bf16(sum[0], sum[1]), pack_bf16(sum[2], sum[3]));
                } else {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (col + v < p.n) dst[v] = to_bf16(sum[v]);
                }
            }
        }
        if (p.buffers == 2) buf ^= 1;
    }
}

// One row block of up to 2048 elements without a LoRA term: three workgroups per compute unit with one LDS buffer each, instead of
// two with two.  A block's way through its workgroup (requests, decoding, two barriers) is longer than the memory's, and three
// independent ones hide more of it than a request ahead does: 151936 x 2048 Q6_K, one row, 66.5 -> 58.0 us; Q8_0 109 -> 103.  (A
// fourth needs 64 registers and spills: 67 us.  Sixteen waves on one block: 88 us with two to five buffers.)  Six waves per SIMD need
// the kernel within 80 registers: Q3_K takes 88 and keeps two workgroups with two buffers, 67.3 -> 65.3 us.
static bool many_small_workgroups(int qt, bool lora, int64_t m, int64_t k) { return qt != kQ3_K && !lora && m <= 16 && k <= 2048; }
template <int QT, int WAVES, int SP, int TB, bool LORA>
static int launch_gemv(const GemvParams& p, hipStream_t s) {
    const int lds = kTableBytes<QT> + p.buffers * p.stage_bytes + WAVES * TB * 64 * 16 + TB * 16 * 64 * 2;
    static LdsLimit lim;
    if (int rc = raise_lds_limit(lim, (const void*)gemv_kernel<QT, WAVES, SP, TB, LORA>, 160 * 1024, "gemv")) return rc;
    const int per_cu = std::max(1, std::min(160 * 1024 / lds, (many_small_workgroups(QT, LORA, p.m, p.k) ? 24 : 16) / WAVES));
    hipLaunchKernelGGL((gemv_kernel<QT, WAVES, SP, TB, LORA>), dim3(std::min((p.n + 15) / 16, 256 * per_cu)), dim3(64 * WAVES), lds, s, p);
    return check_launch("gemv");
}
template <int QT, bool LORA>
static int launch_gemv_qt(const GemvParams& p, hipStream_t s) {
    const int tb = (p.m + 15) / 16;
    if (p.k <= 2048) {
        if (tb == 1) return launch_gemv<QT, 8, 2, 1, LORA>(p, s);
        if (tb == 2) return launch_gemv<QT, 8, 2, 2, LORA>(p, s);
        return launch_gemv<QT, 8, 2, 4, LORA>(p, s);
    }
    if (p.k <= 4096) return tb == 1 ? launch_gemv<QT, 8, 4, 1, LORA>(p, s) : launch_gemv<QT, 8, 4, 2, LORA>(p, s);
    return launch_gemv<QT, 16, 4, 1, LORA>(p, s);
}
template <int QT>
static int launch_gemv_qt(const GemvParams& p, hipStream_t s) {
    return p.lora_a ? launch_gemv_qt<QT, true>(p, s) : launch_gemv_qt<QT, false>(p, s);
}

// Rows up to which x fits the registers of the waves that share it: 64 of 2048 elements, 32 of 4096, 16 of 8192.
bool gemv_takes(int qt, int64_t m, int64_t n, int64_t k, const void* x, int64_t ldx) {
    if (m < 1 || n < 1 || k > 8192 || ((uintptr_t)x & 15) || ldx % 8) return false;
    if (m > (k <= 2048 ? 64 : k <= 4096 ? 32 : 16)) return false;
    return 16 * packed_row_bytes(qt, k) <= (k <= 4096 ? 72 : 136) * 1024;
}

// w: 16-byte aligned, or inside a buffer that starts at a 16-byte address (group g of a stack of matrices: its blocks of
// 34, 66, 84, 110 or 210 bytes start at any multiple of two).  The packed rows are moved as whole aligned pieces, so there the first
// piece begins with bytes of the matrix before.  (Sixteen rows are a multiple of 16 bytes: every block of them starts alike.)
int gemv(int qt, const void* x, int64_t ldx, const void* w, int64_t m, int64_t n, int64_t k, const void* lora_a, const void* lora_b, int r, float scale, void* xa_out,
         void* y, int64_t ldy, hipStream_t s) {
    GemvParams p{};
    p.x = (const bf16_t*)x, p.m = (int)m, p.n = (int)n, p.k = (int)k, p.row_bytes = (int)packed_row_bytes(qt, k), p.y = (bf16_t*)y;
    p.head = (int)((uintptr_t)w & 15), p.w = (const uint8_t*)w - p.head;
    p.ldx = ldx, p.ldy = ldy;
    if (lora_a) p.lora_a = (const bf16_t*)lora_a, p.lora_b = (const bf16_t*)lora_b, p.r = r, p.r_pad = (r + 15) / 16 * 16, p.lora_scale = scale, p.xa_out = (bf16_t*)xa_out;
    p.stage_bytes = row_block_bytes(qt, p.head + 16 * p.row_bytes);
    p.buffers = (p.n + 15) / 16 > 256 && p.stage_bytes <= 36 * 1024 && !many_small_workgroups(qt, lora_a != nullptr, m, k) ? 2 : 1;  // (one block per workgroup needs one buffer)
    TimedScope timed(qt, kModeNT, kEpiStore, kShapeFewRows, s);
    switch (qt) {
        case kQ8_0: return launch_gemv_qt<kQ8_0>(p, s);
        case kQ2_K: return launch_gemv_qt<kQ2_K>(p, s);
        case kQ3_K: return launch_gemv_qt<kQ3_K>(p, s);
        case kQ4_K: return launch_gemv_qt<kQ4_K>(p, s);
        case kQ5_K: return launch_gemv_qt<kQ5_K>(p, s);
        case kQ6_K: return launch_gemv_qt<kQ6_K>(p, s);
        case kIQ2_XXS: return launch_gemv_qt<kIQ2_XXS>(p, s);
    }
    return set_error(GGQ_ERR_QTYPE, "unsupported GGML type id %d", qt);
}

// ------------------------------------------------------------------------------------------------
// Grouped: the forward of expert-sorted rows (a projection, or a gate / up pair) while an expert has a few rows.  Such a launch
// ought to cost the packed bytes of the active experts; what bounds it is the decoding (about four vector instructions per
// weight and lane).  The tile kernels and the decoding-wave kernels pad an expert's rows to 32 at least and stage activations
// for 64 to 192.  Here a workgroup takes one row tile (up to sixteen rows of one expert, as operands in registers) and a part
// of the expert's weight rows, sixteen at a time, requested up to three blocks ahead.  Its waves form TEAMS teams of KW: a team
// deals the contraction of a sixteen-row block out to its waves (of a short contraction every wave takes a block of its own).
// x A^T is formed in the same launch.
// Router-less expert FFN with LoRA rank 16, 256 experts, top-8, before -> after:
//   Q6_K / Q8_0, 2048 / 512:       64 tokens 409 -> 260 us, 256 tokens 441 -> 278 us (tile kernel)
//   IQ2_XXS / Q2_K, 2048 / 2048:   64 tokens 565 -> 410 us, 192 tokens 651 -> 421 us (decoding-wave and tile kernel)
//   IQ2_XXS, 4096 / 1024:         128 tokens 534 -> 411 us
struct GroupedFewRowsParams {
    const bf16_t* x;
    int64_t ldx;
    RowIndex x_rows;
    const TileDesc* tiles;
    const int* num_tiles;
    int max_tiles, parts;
    const uint8_t* w[2];            // planes [experts][n][row_bytes]
    int64_t w_expert_bytes;
    int row_bytes, n, k, nseg;
    bf16_t* y[2];
    int64_t ldy;
    const bf16_t *lora_a, *lora_b;  // [experts][r][k], [experts][nseg * n][r]; null: none
    bf16_t* xa_out;                 // [rows][r_pad]
    int r, r_pad;
    float lora_scale;
    int lb_offset, stage_bytes, buffers;  // LDS bytes of sixteen packed rows, of those with their rows of B behind them; two to four buffers per team
};

template <int QT, int KW>
__global__ __launch_bounds__(64 * (KW < 4 ? 4 : KW)) __attribute__((amdgpu_waves_per_eu(4))) void grouped_few_rows_kernel(GroupedFewRowsParams p) {
    constexpr int WAVES = KW < 4 ? 4 : KW, TEAMS = WAVES / KW, SP = 4;
    extern __shared__ __attribute__((aligned(16))) uint8_t gfr_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4, kw = wave % KW, team = wave / KW;
    // the parts of a row tile follow one another on one XCD: they share its activation and factor rows in that L2
    const int slot = (int)(blockIdx.x >> 3), tile_id = (slot / p.parts) * 8 + (int)(blockIdx.x & 7), part = slot % p.parts;
    if (tile_id >= min(*p.num_tiles, p.max_tiles)) return;
    TileDesc tile = p.tiles[tile_id];
    tile.row_begin = __builtin_amdgcn_readfirstlane(tile.row_begin), tile.row_end = __builtin_amdgcn_readfirstlane(tile.row_end);
    tile.expert = __builtin_amdgcn_readfirstlane(tile.expert);
    const int rows = min(tile.row_end - tile.row_begin, kFewRowsTile);
    if (rows <= 0) return;
    const int seg_blocks = (p.n + 15) / 16, blocks = p.nseg * seg_blocks;
    const int b_begin = (int)((int64_t)blocks * part / p.parts), count = (int)((int64_t)blocks * (part + 1) / p.parts) - b_begin;
    const int spans = (p.k + kSpan - 1) / kSpan;
    uint8_t* stage = gfr_lds + kTableBytes<QT> + team * p.buffers * p.stage_bytes;
    f32x4_t* red_all = (f32x4_t*)(gfr_lds + kTableBytes<QT> + TEAMS * p.buffers * p.stage_bytes);  // [WAVES][64]
    f32x4_t* red = red_all + team * KW * 64;
    bf16_t* xa = (bf16_t*)(red_all + WAVES * 64);                                                  // [16][64]
    // A block's packed rows and its rows of the factor B, into one buffer.  (B comes with the untracked requests too: a load the
    // compiler tracks is waited for with vmcnt(0) where it is used, and that wait would cover every block requested ahead.)
    auto request_block = [&](int i, int buf) __attribute__((always_inline)) {
        const int b = b_begin + i, seg = b >= seg_blocks, row0 = (b - seg * seg_blocks) * 16, block_rows = min(16, p.n - row0);
        uint8_t* dst = stage + buf * p.stage_bytes;
        int made = request_bytes<kPieceGap<QT>>((seg ? p.w[1] : p.w[0]) + (int64_t)tile.expert * p.w_expert_bytes + (int64_t)row0 * p.row_bytes, dst,
                                                block_rows * p.row_bytes, kw, KW, lane);
        if (p.lora_a)
            made += request_bytes((const uint8_t*)(p.lora_b + ((int64_t)tile.expert * p.nseg * p.n + (int64_t)seg * p.n + row0) * p.r), dst + p.lb_offset,
                                  block_rows * p.r * 2, (kw + 1) % KW, KW, lane);
        return made;
    };
    // (the barriers here order LDS traffic only: __syncthreads would also wait for the blocks requested ahead)
    int ahead[2] = {0, 0};  // this wave's requests for the two blocks after the current one
    if (team < count) request_block(team, 0);
#pragma unroll
    for (int i = 1; i < 3; i++)
        if (i < p.buffers - 1 && team + i * TEAMS < count) ahead[i - 1] = request_block(team + i * TEAMS, i);
    stage_tables<QT>(gfr_lds, threadIdx.x, 64 * WAVES);

    uint4 xf[SP][4];
    {
        const bf16_t* src = p.x + (int64_t)p.x_rows.source(tile.row_begin + min(l16, rows - 1)) * p.ldx;
#pragma unroll
        for (int sp = 0; sp < SP; sp++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int e = (kw + KW * sp) * kSpan + span_element<QT>(q, i);
                xf[sp][i] = e < p.k ? *(const uint4*)(src + e) : make_uint4(0, 0, 0, 0);
            }
    }
    if (p.lora_a) {  // x A^T: a team takes sixteen factor rows at a time; kept as bf16 rows in LDS
        const bf16_t* a0 = p.lora_a + (int64_t)tile.expert * p.r * p.k;
        for (int base = 0; base < p.r_pad; base += 16 * TEAMS) {
            const int r0 = base + 16 * team;  // (past r_pad: zeros that nobody stores)
            f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            const bf16_t* arow = a0 + (int64_t)min(r0 + l16, p.r - 1) * p.k;
#pragma unroll
            for (int sp = 0; sp < SP; sp++) {
                uint4 a[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int e = (kw + KW * sp) * kSpan + span_element<QT>(q, i);
                    a[i] = e < p.k && r0 + l16 < p.r ? *(const uint4*)(arow + e) : make_uint4(0, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) acc = mfma16(as_operand(a[i]), as_operand(xf[sp][i]), acc);
            }
            red[kw * 64 + lane] = acc;
            lds_barrier();
            if (kw == 0 && r0 < p.r_pad) {
                f32x4_t sum = red[lane];
#pragma unroll
                for (int w = 1; w < KW; w++) sum += red[w * 64 + lane];
                const uint2 v = make_uint2(pack_bf16(sum[0], sum[1]), pack_bf16(sum[2], sum[3]));  // factor rows r0 + 4 q .. + 3 of tile row l16
                *(uint2*)(xa + l16 * 64 + r0 + 4 * q) = v;
                if (part == 0 && l16 < rows) *(uint2*)(p.xa_out + (int64_t)(tile.row_begin + l16) * p.r_pad + r0 + 4 * q) = v;
            }
            lds_barrier();
        }
    }
    const bool b_vec = (p.r & 7) == 0;
    const bool whole = ((p.n | p.ldy) & 3) == 0 && (((uintptr_t)p.y[0] | (uintptr_t)p.y[1]) & 7) == 0;
    int turn = 0, buf = 0;
    for (int i0 = 0; i0 < count; i0 += TEAMS) {  // uniform over the workgroup; a team's last block may not exist
        const int i = i0 + team, last = i + (p.buffers - 1) * TEAMS;
        const bool live = i < count;
        const int b = b_begin + i, seg = b >= seg_blocks, col0 = (b - seg * seg_blocks) * 16;
        wait_loads_at_most(ahead[0] + ahead[1]);
        lds_barrier();
        {  // every wave is done with the block before: its buffer takes the last block that fits ahead
            const int made = last < count ? request_block(last, buf == 0 ? p.buffers - 1 : buf - 1) : 0;
            if (p.buffers == 4) ahead[0] = ahead[1], ahead[1] = made;
            else if (p.buffers == 3) ahead[0] = made;
        }
        const uint8_t* block = stage + buf * p.stage_bytes;
        f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        if (live) {
            const int row = min(l16, p.n - col0 - 1) * p.row_bytes;
#pragma unroll
            for (int sp = 0; sp < SP; sp++) {
                const int span = kw + KW * sp;
                if (span >= spans) break;  // uniform over the wave
                uint32_t v[16];
                decode_span<QT>(block, row, span, p.k >> 5, q, v, (const uint2*)gfr_lds);
#pragma unroll
                for (int m = 0; m < 4; m++) acc = mfma16(as_operand(make_uint4(v[4 * m], v[4 * m + 1], v[4 * m + 2], v[4 * m + 3])), as_operand(xf[sp][m]), acc);
            }
        }
        red[kw * 64 + lane] = acc;
        lds_barrier();
        // (a buffer is refilled, and the partial sums rewritten, only behind the next barrier)
        if (live && kw == turn) {
            f32x4_t sum = red[lane];
#pragma unroll
            for (int w = 1; w < KW; w++) sum += red[w * 64 + lane];
            const int col = col0 + 4 * q;
            if (p.lora_a) {
                const bf16_t* brow = (const bf16_t*)(block + p.lb_offset) + min(l16, p.n - col0 - 1) * p.r;
                f32x4_t lo = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                for (int r0 = 0; r0 < p.r_pad; r0 += 32) {
                    const int j = r0 + 8 * q;
                    const uint4 xv = j < p.r_pad ? *(const uint4*)(xa + l16 * 64 + j) : make_uint4(0, 0, 0, 0);
                    lo = mfma16(as_operand(load_factor8(brow + j, p.r - j, b_vec)), as_operand(xv), lo);
                }
                sum += lo * p.lora_scale;
            }
            if (l16 < rows) {
                bf16_t* dst = (seg ? p.y[1] : p.y[0]) + (int64_t)(tile.row_begin + l16) * p.ldy + col;
                if (whole) {
                    if (col < p.n) *(uint2*)dst = make_uint2(pack_bf16(sum[0], sum[1]), pack_bf16(sum[2], sum[3]));
                } else {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (col + v < p.n) dst[v] = to_bf16(sum[v]);
                }
            }
        }
        turn = turn + 1 == KW ? 0 : turn + 1;  // the wave that adds the partial sums changes from block to block
        buf = buf + 1 == p.buffers ? 0 : buf + 1;
    }
}

template <int QT, int KW>
static int grouped_few_rows_lds(int stage_bytes, int buffers) {
    constexpr int kWaves = KW < 4 ? 4 : KW;
    return kTableBytes<QT> + kWaves / KW * buffers * stage_bytes + kWaves * 64 * 16 + 16 * 64 * 2;
}
static int few_rows_waves(int64_t k) { return k <= 512 ? 1 : k <= 1024 ? 2 : k <= 2048 ? 4 : 8; }  // waves that share a contraction
static int64_t few_rows_stage(int qt, int64_t k) { return row_block_bytes(qt, (int)(16 * packed_row_bytes(qt, k))); }

// Rows per expert, in the mean of a call, up to which these kernels are the faster ones.  Against the tile kernel (most
// formats) and the IQ2_XXS decoding waves the line is where experts with more than one row tile become common, each tile
// decoding the weights again: IQ2_XXS 4096 / 1024 at 8 rows 650 against 563 us, IQ2_XXS / Q2_K at 8 rows 554 against 654 us.
// The Q4_K decoding waves, whose waves share no decoded weight either, are as fast from half a row on (120 us both at 16 tokens
// of 2048 / 512, 212 against 203 us at 128).
static bool few_rows_per_expert(int qt, int64_t rows, int64_t groups) {
    if (qt == kQ4_K) return 2 * rows <= groups;
    return rows <= (qt == kIQ2_XXS ? 6 : kFewRowsPerGroup) * groups;
}
bool grouped_few_rows_takes(int qt, int64_t rows, int64_t groups, int64_t n, int64_t k, const void* x) {
    if (!few_rows_per_expert(qt, rows, groups) || k > 4096 || ((uintptr_t)x & 15) || n % 8) return false;  // (planes of B and of packed rows start at 16-byte addresses)
    const int waves = few_rows_waves(k), teams = waves < 4 ? 4 / waves : 1;
    return teams * 2 * (few_rows_stage(qt, k) + 2048) <= 140 * 1024;  // (two buffers, the partial sums, x A^T and tables: within 160 KB)
}

template <int QT, int KW>
static int launch_grouped_few_rows(GroupedFewRowsParams p, hipStream_t s) {
    constexpr int kThreadsWG = 64 * (KW < 4 ? 4 : KW);
    static LdsLimit lim;
    if (int rc = raise_lds_limit(lim, (const void*)grouped_few_rows_kernel<QT, KW>, 160 * 1024, "grouped_few_rows")) return rc;
    // as many buffers as leave room for sixteen waves on a compute unit, or else for two workgroups
    p.buffers = 4;
    while (p.buffers > 2 && grouped_few_rows_lds<QT, KW>(p.stage_bytes, p.buffers) > 160 * 1024 / (1024 / kThreadsWG)) p.buffers--;
    const int64_t grid = (int64_t)(p.max_tiles + 7) / 8 * 8 * p.parts;
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "grouped_few_rows: too many tiles for one launch");
    const int lds = grouped_few_rows_lds<QT, KW>(p.stage_bytes, p.buffers);
    hipLaunchKernelGGL((grouped_few_rows_kernel<QT, KW>), dim3((unsigned)grid), dim3(kThreadsWG), lds, s, p);
    return check_launch("grouped_few_rows");
}
template <int QT>
static int launch_grouped_few_rows_qt(const GroupedFewRowsParams& p, hipStream_t s) {
    switch (few_rows_waves(p.k)) {
        case 1: return launch_grouped_few_rows<QT, 1>(p, s);
        case 2: return launch_grouped_few_rows<QT, 2>(p, s);
        case 4: return launch_grouped_few_rows<QT, 4>(p, s);
    }
    return launch_grouped_few_rows<QT, 8>(p, s);
}

int grouped_few_rows(int qt, const GroupedFewRowsCall& c, hipStream_t s) {
    GroupedFewRowsParams p{};
    p.x = (const bf16_t*)c.x, p.ldx = c.k, p.x_rows = c.x_rows, p.tiles = c.tiles, p.num_tiles = c.num_tiles, p.max_tiles = c.max_tiles;
    p.row_bytes = (int)packed_row_bytes(qt, c.k), p.n = (int)c.n, p.k = (int)c.k, p.nseg = c.w2 ? 2 : 1, p.w_expert_bytes = c.n * p.row_bytes;
    p.w[0] = (const uint8_t*)c.w1, p.w[1] = (const uint8_t*)c.w2, p.y[0] = (bf16_t*)c.y1, p.y[1] = (bf16_t*)c.y2, p.ldy = c.n;
    if (c.lora_a)
        p.lora_a = (const bf16_t*)c.lora_a, p.lora_b = (const bf16_t*)c.lora_b, p.xa_out = (bf16_t*)c.xa_out, p.r = c.r, p.r_pad = (c.r + 15) / 16 * 16,
        p.lora_scale = c.lora_scale;
    p.lb_offset = (int)few_rows_stage(qt, c.k), p.stage_bytes = p.lb_offset + (p.lora_a ? 16 * p.r_pad * 2 : 0);
    const int64_t kSlots = few_rows_waves(c.k) <= 4 ? 1024 : 512;
    // a workgroup for every slot of the chip (sixteen waves per compute unit), while a part keeps four blocks per team
    const int64_t tiles = std::min<int64_t>(c.max_tiles, std::min(c.groups, c.rows)), blocks = p.nseg * ((c.n + 15) / 16), waves = few_rows_waves(c.k), teams = waves < 4 ? 4 / waves : 1;
    p.parts = (int)std::max<int64_t>(1, std::min((kSlots + tiles / 2) / std::max<int64_t>(1, tiles), blocks / (4 * teams)));
    TimedScope timed(qt, kModeNT, kEpiStore, kShapeFewRows, s);
    switch (qt) {
        case kQ8_0: return launch_grouped_few_rows_qt<kQ8_0>(p, s);
        case kQ2_K: return launch_grouped_few_rows_qt<kQ2_K>(p, s);
        case kQ3_K: return launch_grouped_few_rows_qt<kQ3_K>(p, s);
        case kQ4_K: return launch_grouped_few_rows_qt<kQ4_K>(p, s);
        case kQ5_K: return launch_grouped_few_rows_qt<kQ5_K>(p, s);
        case kQ6_K: return launch_grouped_few_rows_qt<kQ6_K>(p, s);
        case kIQ2_XXS: return launch_grouped_few_rows_qt<kIQ2_XXS>(p, s);
    }
    return set_error(GGQ_ERR_QTYPE, "unsupported GGML type id %d", qt);
}

// ------------------------------------------------------------------------------------------------
// Router logits of up to eight tokens: y [m, n] = x [m, k] . w [n, k]^T, all bf16.  A workgroup takes sixteen weight rows, its
// eight waves deal the contraction out in spans of 128.  (A library product of this size costs 19 us of host time per call.)
__global__ __launch_bounds__(512) void few_rows_bf16_kernel(const bf16_t* x, const bf16_t* w, int m, int n, int k, bf16_t* y) {
    constexpr int WAVES = 8;
    __shared__ f32x4_t red[WAVES][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4, n0 = blockIdx.x * 16;
    const bf16_t* wr = w + (int64_t)min(n0 + l16, n - 1) * k;
    const bf16_t* xr = x + (int64_t)min(l16, m - 1) * k;
    f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int steps = (k + kSpan - 1) / kSpan;
    for (int s = wave; s < steps; s += WAVES) {
        uint4 a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int e = s * kSpan + 32 * i + 8 * q;
            a[i] = e < k ? *(const uint4*)(wr + e) : make_uint4(0, 0, 0, 0);
            b[i] = e < k ? *(const uint4*)(xr + e) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) acc = mfma16(as_operand(a[i]), as_operand(b[i]), acc);
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave > 0) return;
    for (int i = 1; i < WAVES; i++) acc += red[i][lane];
    if (l16 < m) {
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (n0 + 4 * q + v < n) y[(int64_t)l16 * n + n0 + 4 * q + v] = to_bf16(acc[v]);
    }
}

int router_logits(const void* x, const void* w, int64_t m, int64_t n, int64_t k, void* y, hipStream_t s) {
    if (m < 1 || m > kRouterLogitsMaxTokens || n < 1 || k < 1 || k % 8 || n >= (1 << 20) || k >= (1 << 20)) return set_error(GGQ_ERR_SHAPE, "router_logits: takes 1 to %d tokens of a multiple of 8 elements", kRouterLogitsMaxTokens);
    if (((uintptr_t)x | (uintptr_t)w) & 15) return set_error(GGQ_ERR_ALIGN, "router_logits: operands must be 16-byte aligned");
    hipLaunchKernelGGL(few_rows_bf16_kernel, dim3((unsigned)((n + 15) / 16)), dim3(512), 0, s, (const bf16_t*)x, (const bf16_t*)w, (int)m, (int)n, (int)k, (bf16_t*)y);
    return check_launch("router_logits");
}

// ------------------------------------------------------------------------------------------------
// Expert FFN of a few routes, without a routing plan: with a handful of routes hardly two share an expert, so every route
// reads its own expert's weights and the four launches of plan and tables, the gather by expert and the combine's pass fall
// away.  Two launches:
//   act[route] = silu(gate) * up         one workgroup per (route, eight or sixteen gate rows and the up rows of the same columns)
//   out[token] = sum w[route] * down     one workgroup per (token, sixteen output columns), one wave per route
// The LoRA products x A^T are formed by every workgroup for itself (64 KB of factor out of the L2 at rank 16 and 2048
// columns): cheaper than a launch.  One token, 8 of 256 Q4_K experts, 2048 / 512: 7.5 and 9.2 us; with the factor rows read
// as MFMA operands and eight gate rows per workgroup 10.4 and 11.3.
struct FewRoutesParams {
    const bf16_t* x;       // [tokens, hidden]
    const void* ids;
    int ids64;
    const void* weights;   // [tokens, top_k]
    int weights_bf16;
    int tokens, top_k, experts, hidden, inter;
    const uint8_t *gate, *up, *down;
    int row_bytes_in, row_bytes_down;
    const bf16_t *a1, *b1, *a2, *b2;
    int r1, r2;
    float scale, limit;
    int x_in_lds;          // down: room for 512 elements of x per wave
    bf16_t* act;           // [routes, inter]
    bf16_t* out;           // [tokens, hidden]
};

__device__ __forceinline__ int route_expert(const FewRoutesParams& p, int route) {
    const int64_t e = p.ids64 ? ((const int64_t*)p.ids)[route] : (int64_t)((const int32_t*)p.ids)[route];
    return (int)(e < 0 ? 0 : e >= p.experts ? p.experts - 1 : e);  // (the routing plan clamps in the same way)
}

// sum over j of b[j] * xa[j] for the sixteen rows of a block: lane (row lane % 16, quarter) takes every fourth group of eight
// ranks, the first of them loaded by the caller ahead of the work it would wait behind; every lane of a row returns the sum.
__device__ __forceinline__ float lora_row_dot(const uint4& first, const bf16_t* brow, const bf16_t* xa, int r, bool vec, int q) {
    float s = 0.f;
    for (int j = 8 * q; j < r; j += 32) {
        const uint4 b = j < 32 ? first : load_factor8(brow + j, r - j, vec), x = *(const uint4*)(xa + j);
        const uint32_t bw[4] = {b.x, b.y, b.z, b.w}, xw[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; i++) s = fmaf(bf16_lo(bw[i]), bf16_lo(xw[i]), s), s = fmaf(bf16_hi(bw[i]), bf16_hi(xw[i]), s);
    }
    s += __shfl_xor(s, 16, 64);
    return s + __shfl_xor(s, 32, 64);
}

// x . row for a row of k bf16 values, eight of every 512 per lane (x as loaded by load_row_pieces); the sum over the lanes is the caller's.
template <int PIECES>
__device__ __forceinline__ void load_row_pieces(const bf16_t* row, int k, int lane, uint4 (&v)[PIECES]) {
#pragma unroll
    for (int t = 0; t < PIECES; t++) {
        const int e = 512 * t + 8 * lane;
        if constexpr (PIECES == 1) {
            // (the down kernel's) 32-bit offsets from a row that all lanes share, and no branch: past the end a lane reads the last piece and drops
            // it.  One token, 8 of 256 Q4_K experts, 2048 / 512: 9.5 -> 9.2 us.
            const uint4 p = *(const uint4*)((const uint8_t*)row + 2u * (uint32_t)min(e, k - 8));
            v[t] = make_uint4(e < k ? p.x : 0u, e < k ? p.y : 0u, e < k ? p.z : 0u, e < k ? p.w : 0u);
        } else {  // (gate / up: without the branch 12 registers more and nothing gained, one token 7.5 and 7.5 us, four tokens 18.3 and 18.6)
            v[t] = e < k ? *(const uint4*)(row + e) : make_uint4(0, 0, 0, 0);
        }
    }
}
__device__ __forceinline__ float dot8(const uint4& a, const uint4& b, float s) {
    const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; i++) s = fmaf(bf16_lo(aw[i]), bf16_lo(bw[i]), s), s = fmaf(bf16_hi(aw[i]), bf16_hi(bw[i]), s);
    return s;
}
__device__ __forceinline__ float wave_sum(float s) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) s += __shfl_xor(s, off, 64);
    return s;
}

// Eight gate rows and eight up rows per set; a workgroup takes SETS sets of one route.  What bounds it is latency and the
// vector cache's requests: every workgroup forms x A^T for itself, and as MFMA operands (16 rows x 64 bytes a request) the 64 KB
// of A cost two workgroups of a compute unit 2.3 us.  So each wave takes whole rows of A (1 KB a request, half the time), x
// comes to LDS once, and two sets share one x A^T where that leaves enough workgroups.  The requests of the packed rows are ahead of A's,
// not beside them: x is unpacked in front of the loop over the ranks, and the wait for x takes the packed rows along.
__host__ __device__ __forceinline__ int gate_up_half_lds(int qt, int row_bytes, int sets) {
    const int bytes = 8 * sets * row_bytes;
    return qt == kQ4_K ? (bytes + (bytes >> 10) * kPieceGap<kQ4_K> + 127) & ~127 : (bytes + 15) & ~15;
}
template <int QT, int SP, int SETS>
__global__ __launch_bounds__(512) void few_routes_gate_up_kernel(FewRoutesParams p) {
    constexpr int WAVES = 8, PIECES = SP * 2;  // 512-element pieces of x: k <= 1024 SP
    extern __shared__ __attribute__((aligned(16))) uint8_t gu_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int half_bytes = 8 * SETS * p.row_bytes_in, half_lds = gate_up_half_lds(QT, p.row_bytes_in, SETS);
    uint8_t* stage = gu_lds + kTableBytes<QT>;
    bf16_t* xs = (bf16_t*)(stage + 2 * half_lds);     // [512 PIECES]
    float* red = (float*)(xs + 512 * PIECES);         // [SETS][WAVES][16]
    bf16_t* xa = (bf16_t*)(red + SETS * WAVES * 16);  // [64]
    const int route = blockIdx.y, i0 = blockIdx.x * 8 * SETS, k = p.hidden;
    const bf16_t* x = p.x + (int64_t)(route / p.top_k) * k;
    uint4 xr[PIECES];
    load_row_pieces(x, k, lane, xr);
    const int expert = route_expert(p, route);
    const int64_t row0 = (int64_t)expert * p.inter + i0;
    request_bytes<kPieceGap<QT>>(p.gate + row0 * p.row_bytes_in, stage, half_bytes, wave, WAVES, lane);
    request_bytes<kPieceGap<QT>>(p.up + row0 * p.row_bytes_in, stage + half_lds, half_bytes, (wave + 4) & 7, WAVES, lane);
    stage_tables<QT>(gu_lds, threadIdx.x, 512);
    const int r_pad = (p.r1 + 15) & ~15;
    const bool b_vec = (p.r1 & 7) == 0;
    // the wave that finishes set `wave`: its row of B ahead of the work it would wait behind
    const int own_row = (l16 < 8 ? i0 + l16 : p.inter + i0 + l16 - 8) + 8 * wave;
    const bf16_t* brow = p.b1 + ((int64_t)expert * 2 * p.inter + own_row) * p.r1;
    uint4 b0 = make_uint4(0, 0, 0, 0);
    if (p.a1 && wave < SETS) b0 = load_factor8(brow + 8 * q, p.r1 - 8 * q, b_vec);
    if (p.a1) {
        const bf16_t* a = p.a1 + (int64_t)expert * p.r1 * k;
        for (int j0 = wave; j0 < r_pad; j0 += 2 * WAVES) {  // ranks j0 and j0 + 8 together
            // Opaque: unpacked once ahead of the loop, x would be twice the registers (183, of more than 2048 elements), and a compute unit
            // would have one workgroup.  One token, 8 Q4_K experts, 4096 / 1536, with router and down: 68.8 -> 56.6 us, 3072 / 1024: 41.5 -> 38.0.
#pragma unroll
            for (int t = 0; SP > 2 && t < PIECES; t++) xr[t] = make_uint4(opaque(xr[t].x), opaque(xr[t].y), opaque(xr[t].z), opaque(xr[t].w));
            uint4 a0[PIECES], a8[PIECES];
            load_row_pieces(a + (int64_t)min(j0, p.r1 - 1) * k, k, lane, a0);
            load_row_pieces(a + (int64_t)min(j0 + WAVES, p.r1 - 1) * k, k, lane, a8);
            float s0 = 0.f, s8 = 0.f;
#pragma unroll
            for (int t = 0; t < PIECES; t++) s0 = dot8(a0[t], xr[t], s0), s8 = dot8(a8[t], xr[t], s8);
            s0 = wave_sum(s0), s8 = wave_sum(s8);
            if (lane == 0) xa[j0] = j0 < p.r1 ? to_bf16(s0) : (bf16_t)0, xa[j0 + WAVES] = j0 + WAVES < p.r1 ? to_bf16(s8) : (bf16_t)0;
        }
    }
#pragma unroll
    for (int t = 0; t < PIECES; t++)
        if (wave == t % WAVES) *(uint4*)(xs + 512 * t + 8 * lane) = xr[t];
    wait_loads_at_most(0);
    __syncthreads();
    const uint8_t* half = stage + (l16 < 8 ? 0 : half_lds);  // rows 0..7 gate, 8..15 up
    const int spans = (k + kSpan - 1) / kSpan;
    f32x4_t acc[SETS];
#pragma unroll
    for (int b = 0; b < SETS; b++) acc[b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sp = 0; sp < SP; sp++) {
        const int span = wave + WAVES * sp;
        if (span >= spans) break;
        uint4 xf[4];
#pragma unroll
        for (int i = 0; i < 4; i++) xf[i] = *(const uint4*)(xs + span * kSpan + span_element<QT>(q, i));  // (zeros past k)
#pragma unroll
        for (int b = 0; b < SETS; b++) {
            uint32_t v[16];
            decode_span<QT>(half, (8 * b + (l16 & 7)) * p.row_bytes_in, span, k >> 5, q, v, (const uint2*)gu_lds);
#pragma unroll
            for (int i = 0; i < 4; i++) acc[b] = mfma16(as_operand(make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3])), as_operand(xf[i]), acc[b]);
        }
    }
#pragma unroll
    for (int b = 0; b < SETS; b++)
        if (l16 == 0) *(f32x4_t*)(red + (b * WAVES + wave) * 16 + 4 * q) = acc[b];
    __syncthreads();
    if (wave >= SETS) return;
    float y = 0.f;  // of row l16 of set `wave`, in all four quarters
#pragma unroll
    for (int w = 0; w < WAVES; w++) y += red[(wave * WAVES + w) * 16 + l16];
    if (p.a1) y = fmaf(p.scale, lora_row_dot(b0, brow, xa, p.r1, b_vec, q), y);
    y = bf16_to_f32(to_bf16(y));
    const float up = __shfl(y, (lane & 7) + 8, 64), gate = __shfl(y, lane & 7, 64);
    if (lane < 8) {
        const float hi = p.limit > 0.0f ? p.limit : INFINITY;
        const float g = fminf(gate, hi), u = fminf(fmaxf(up, -hi), hi);
        p.act[(int64_t)route * p.inter + i0 + 8 * wave + lane] = to_bf16(g / (1.0f + __expf(-g)) * u);
    }
}

// What bounds it is round trips one after another: the expert's id, the route's weight, the packed rows (the compiler waits for every
// request of request_bytes before the next, for Q4_K rows of 512 elements five), x, and the rows of A in eights.
template <int QT>
__global__ __launch_bounds__(512) void few_routes_down_kernel(FewRoutesParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t down_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int stage_bytes = row_block_bytes(QT, 16 * p.row_bytes_down);
    uint8_t* mine = down_lds + kTableBytes<QT> + wave * stage_bytes;
    float* red = (float*)(down_lds + kTableBytes<QT> + 8 * stage_bytes);  // [16 routes][16]
    bf16_t* xa = (bf16_t*)(red + 256) + wave * 64;
    bf16_t* xs = (bf16_t*)(red + 256) + 8 * 64 + wave * 512;  // this wave's 512 elements of x (where the LDS has room for them)
    const int token = blockIdx.y, h0 = blockIdx.x * 16, k = p.inter, spans = (k + kSpan - 1) / kSpan;
    const int rows = min(16, p.hidden - h0);
    stage_tables<QT>(down_lds, threadIdx.x, 512);
    if (kTableBytes<QT>) __syncthreads();
    for (int rank = wave; rank < p.top_k; rank += 8) {
        const int route = token * p.top_k + rank, expert = route_expert(p, route);
        // (ahead of the work: behind the last barrier its latency would be the workgroup's)
        const float weight = p.weights_bf16 ? bf16_to_f32(((const bf16_t*)p.weights)[route]) : ((const float*)p.weights)[route];
        // this wave's own sixteen rows: no other wave touches them, so no barrier stands between their requests and their use
        request_bytes<kPieceGap<QT>>(p.down + ((int64_t)expert * p.hidden + h0) * p.row_bytes_down, mine, rows * p.row_bytes_down, 0, 1, lane);
        const bf16_t* x = p.act + (int64_t)route * k;
        const bf16_t* a = p.a2 ? p.a2 + (int64_t)expert * p.r2 * k : nullptr;
        const bool b_vec = (p.r2 & 7) == 0;
        const bf16_t* brow = p.b2 + ((int64_t)expert * p.hidden + min(h0 + l16, p.hidden - 1)) * p.r2;
        uint4 b0 = make_uint4(0, 0, 0, 0);
        if (a) b0 = load_factor8(brow + 8 * q, p.r2 - 8 * q, b_vec);
        f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        float part[4] = {0.f, 0.f, 0.f, 0.f};  // x A^T of rank 16 j + lane / 4, of a sixteenth of the elements
        const int row = min(l16, rows - 1) * p.row_bytes_down;
        for (int s0 = 0; s0 < spans; s0 += 4) {  // 512 elements of x at a time
            uint4 xr[1];
            load_row_pieces(x + s0 * kSpan, k - s0 * kSpan, lane, xr);
            if (a) {
                // Sixteen ranks at a time, whole rows of A (1 KB a request: as MFMA operands, 16 rows x 64 bytes, a request cost
                // the vector cache twice that): each lane has eight terms of every rank, and four exchanges leave each with one rank.
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (16 * j >= p.r2) break;
                    float d[16];
#pragma unroll
                    for (int h = 0; h < 16; h++) {
                        uint4 av[1];
                        load_row_pieces(a + (int64_t)min(16 * j + h, p.r2 - 1) * k + s0 * kSpan, k - s0 * kSpan, lane, av);
                        d[h] = dot8(av[0], xr[0], 0.f);
                    }
#pragma unroll
                    for (int n = 8, bit = 32; n >= 1; n >>= 1, bit >>= 1)
#pragma unroll
                        for (int h = 0; h < n; h++) {
                            const float give = (lane & bit) ? d[h] : d[h + n], keep = (lane & bit) ? d[h + n] : d[h];
                            d[h] = keep + __shfl_xor(give, bit, 64);
                        }
                    part[j] += d[0];  // of rank 16 j + lane / 4, summed over all lanes but the low two bits
                }
            }
            if (p.x_in_lds) *(uint4*)(xs + 8 * lane) = xr[0];
            uint4 xf[4][4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int e = u * kSpan + span_element<QT>(q, i);
                    if (p.x_in_lds) xf[u][i] = *(const uint4*)(xs + e);  // (LDS serves a wave in order)
                    else xf[u][i] = s0 * kSpan + e < k ? *(const uint4*)(x + s0 * kSpan + e) : make_uint4(0, 0, 0, 0);
                }
            }
            if (s0 == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (s0 + u >= spans) break;  // uniform
                uint32_t v[16];
                decode_span<QT>(mine, row, s0 + u, k >> 5, q, v, (const uint2*)down_lds);
#pragma unroll
                for (int i = 0; i < 4; i++) acc = mfma16(as_operand(make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3])), as_operand(xf[u][i]), acc);
            }
        }
        if (a) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (16 * j >= p.r2) break;
                float t = part[j] + __shfl_xor(part[j], 1, 64);
                t += __shfl_xor(t, 2, 64);
                const int rank_a = 16 * j + (lane >> 2);
                if ((lane & 3) == 0) xa[rank_a] = rank_a < p.r2 ? to_bf16(t) : (bf16_t)0;
            }
        }
        if (l16 == 0) *(f32x4_t*)(red + rank * 16 + 4 * q) = acc;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        float y = red[rank * 16 + l16];
        if (p.a2) y = fmaf(p.scale, lora_row_dot(b0, brow, xa, p.r2, b_vec, q), y);
        // (weights and rows act at bf16 precision: their product is exact)
        if (q == 0) red[rank * 16 + l16] = bf16_to_f32(to_bf16(y)) * bf16_to_f32(to_bf16(weight));
    }
    __syncthreads();
    if ((int)threadIdx.x < rows) {  // the combine: routes in rank order
        float sum = 0.f;
        for (int rank = 0; rank < p.top_k; rank++) sum += red[rank * 16 + threadIdx.x];
        p.out[(int64_t)token * p.hidden + h0 + threadIdx.x] = to_bf16(sum);
    }
}

static int gate_up_lds(int qt, int row_bytes, int64_t hidden, int sets) {
    return (qt == kIQ2_XXS ? kTableBytes<kIQ2_XXS> : 0) + 2 * gate_up_half_lds(qt, row_bytes, sets) + (hidden <= 2048 ? 4096 : 8192) + sets * 8 * 16 * 4 + 128;
}
static int down_lds_bytes(int qt, int row_bytes) { return (qt == kIQ2_XXS ? kTableBytes<kIQ2_XXS> : 0) + 8 * row_block_bytes(qt, 16 * row_bytes) + 256 * 4 + 8 * 128; }

template <int QT, int SP, int SETS>
static int launch_gate_up_sets(const FewRoutesParams& p, hipStream_t s) {
    static LdsLimit lim;
    if (int rc = raise_lds_limit(lim, (const void*)few_routes_gate_up_kernel<QT, SP, SETS>, 160 * 1024, "few_routes_gate_up")) return rc;
    hipLaunchKernelGGL((few_routes_gate_up_kernel<QT, SP, SETS>), dim3(p.inter / (8 * SETS), p.tokens * p.top_k), dim3(512), gate_up_lds(QT, p.row_bytes_in, p.hidden, SETS), s, p);
    return check_launch("few_routes_gate_up");
}
template <int QT>
static int launch_gate_up(const FewRoutesParams& p, hipStream_t s) {
    // two sets where every compute unit still has a workgroup, and two workgroups of a unit fit its LDS
    const bool two = p.inter % 16 == 0 && (int64_t)p.tokens * p.top_k * p.inter / 16 >= 256 && gate_up_lds(QT, p.row_bytes_in, p.hidden, 2) <= 80 * 1024;
    if (p.hidden <= 2048) return two ? launch_gate_up_sets<QT, 2, 2>(p, s) : launch_gate_up_sets<QT, 2, 1>(p, s);
    return two ? launch_gate_up_sets<QT, 4, 2>(p, s) : launch_gate_up_sets<QT, 4, 1>(p, s);
}
template <int QT>
static int launch_down(const FewRoutesParams& p, hipStream_t s) {
    static LdsLimit lim;
    if (int rc = raise_lds_limit(lim, (const void*)few_routes_down_kernel<QT>, 160 * 1024, "few_routes_down")) return rc;
    FewRoutesParams q = p;
    const int lds = down_lds_bytes(QT, p.row_bytes_down);
    q.x_in_lds = lds + 8 * 1024 <= 160 * 1024;
    hipLaunchKernelGGL(few_routes_down_kernel<QT>, dim3((p.hidden + 15) / 16, p.tokens), dim3(512), lds + (q.x_in_lds ? 8 * 1024 : 0), s, q);
    return check_launch("few_routes_down");
}

// Up to this many routes every route reads its own expert's weights.  Beyond, the routing plan and the grouped kernels are
// faster: 2048 / 512, 256 experts, 32 / 64 routes: Q4_K 54 / 97 against 54 / 70 us, Q6_K with Q8_0 58 / 111 against 62 / 92 us; the
// decoder's tables, staged by every workgroup, set the line lower: IQ2_XXS 8 / 16 / 64 routes of 4096 / 1024: 52 / 95 / 351
// against 54 / 69 / 135 us.
static int64_t few_routes_limit(int qt_in, int qt_down) { return qt_in == kIQ2_XXS || qt_down == kIQ2_XXS ? 4 : 32; }

bool few_routes_takes(int qt_in, int qt_down, int64_t tokens, int top_k, int64_t hidden, int64_t inter) {
    return tokens > 0 && top_k > 0 && top_k <= 16 && tokens * top_k <= few_routes_limit(qt_in, qt_down) && hidden <= 4096 && inter % 8 == 0 && hidden % 8 == 0 &&
           gate_up_lds(qt_in, (int)packed_row_bytes(qt_in, hidden), hidden, 1) <= 88 * 1024 && down_lds_bytes(qt_down, (int)packed_row_bytes(qt_down, inter)) <= 160 * 1024;
}

int few_routes_forward(const void* x, const void* ids, int ids64, const void* weights, int weights_bf16, int64_t tokens, int top_k, int64_t experts, int64_t hidden,
                       int64_t inter, int qt_in, int qt_down, const void* gate, const void* up, const void* down, const void* a1, const void* b1, int r1,
                       const void* a2, const void* b2, int r2, float scale, float limit, void* act, void* out, hipStream_t s) {
    FewRoutesParams p{};
    p.x = (const bf16_t*)x, p.ids = ids, p.ids64 = ids64, p.weights = weights, p.weights_bf16 = weights_bf16;
    p.tokens = (int)tokens, p.top_k = top_k, p.experts = (int)experts, p.hidden = (int)hidden, p.inter = (int)inter;
    p.gate = (const uint8_t*)gate, p.up = (const uint8_t*)up, p.down = (const uint8_t*)down;
    p.row_bytes_in = (int)packed_row_bytes(qt_in, hidden), p.row_bytes_down = (int)packed_row_bytes(qt_down, inter);
    p.a1 = (const bf16_t*)a1, p.b1 = (const bf16_t*)b1, p.a2 = (const bf16_t*)a2, p.b2 = (const bf16_t*)b2, p.r1 = r1, p.r2 = r2;
    p.scale = scale, p.limit = limit, p.act = (bf16_t*)act, p.out = (bf16_t*)out;
#define GGQ_FEW(F, QT) \
    case QT: rc = F<QT>(p, s); break
    int rc = GGQ_ERR_QTYPE;
    switch (qt_in) {
        GGQ_FEW(launch_gate_up, kQ8_0); GGQ_FEW(launch_gate_up, kQ2_K); GGQ_FEW(launch_gate_up, kQ3_K); GGQ_FEW(launch_gate_up, kQ4_K);
        GGQ_FEW(launch_gate_up, kQ5_K); GGQ_FEW(launch_gate_up, kQ6_K); GGQ_FEW(launch_gate_up, kIQ2_XXS);
    }
    if (rc) return rc;
    rc = GGQ_ERR_QTYPE;
    switch (qt_down) {
        GGQ_FEW(launch_down, kQ8_0); GGQ_FEW(launch_down, kQ2_K); GGQ_FEW(launch_down, kQ3_K); GGQ_FEW(launch_down, kQ4_K);
        GGQ_FEW(launch_down, kQ5_K); GGQ_FEW(launch_down, kQ6_K); GGQ_FEW(launch_down, kIQ2_XXS);
    }
#undef GGQ_FEW
    return rc;
}

}  // namespace ggq
