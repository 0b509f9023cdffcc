// Chunked cross-entropy through a packed lm_head without ever holding [rows, vocab] logits.
//
// Per block of up to kGradRows rows the vocabulary is swept once, in blocks of columns, with a running (max, sum exp) per row
// as in a streaming softmax: the dense launch over the block's decoded weights writes the block's logits into a slab; a row
// kernel updates the running statistics and rewrites the slab as exp(logit - running max); the grad-input launch adds
// slab . W_block to an fp32 accumulator that it first rescales by exp(old max - new max).  At the end
// dH = (accumulator / sum - W[label]) * row_scale.  Two vocabulary-sized matmuls.
#include <algorithm>

#include "common.h"
#include "launch.h"
#include "mmq_host.h"

namespace ggq {

// The sweep takes up to this many rows at a time, whatever the caller's chunk (which stands for the reference's
// [chunk, vocab] logits): 4096 rows fill the chip with tiles of the [rows, hidden] grad-input output.
constexpr int64_t kGradRows = 4096;
// The slab holds kSlabElems logits (64 MB): 8192 columns of 4096 rows, and more columns of fewer rows, so that a short
// sequence does not pay the launches of a step, and the grad-input launch its accumulator's traffic, nineteen times over a
// 152k vocabulary.  Up to 32768 columns: a row kernel's workgroup holds a row's block in registers.
constexpr int64_t kSlabElems = 4096 * 8192;
constexpr int kMaxVocabBlock = 32768;
static int vocab_block(int64_t rows, int64_t vocab) {
    int block = 8192;
    while (block < kMaxVocabBlock && 2 * block * std::min(rows, kGradRows) <= kSlabElems) block *= 2;
    return (int)std::min<int64_t>(block, (vocab + 63) / 64 * 64);
}

// row_scale[m] = 0 for ignored rows, else 1/n_valid (mean) or 1 (sum); n_valid = 0 gives all zeros.  A label outside
// [0, vocab) that is not ignore_index is treated as ignored (no loss, no gradient) and counted in status[1].
__device__ __forceinline__ bool label_counts(int64_t label, int64_t vocab, int64_t ignore_index) {
    return label != ignore_index && label >= 0 && label < vocab;
}
__global__ __launch_bounds__(1024) void ce_row_scale_kernel(const int64_t* labels, int64_t rows, int64_t vocab, int64_t ignore_index,
                                                             int mean, float* row_scale, int* status, float* run_max, float* run_sum, float* target) {
    __shared__ int partial[1024], partial_bad[1024];
    int c = 0, bad = 0;
    for (int64_t i = threadIdx.x; i < rows; i += 1024) {
        const int64_t l = labels[i];
        c += label_counts(l, vocab, ignore_index);
        bad += l != ignore_index && (l < 0 || l >= vocab);
    }
    partial[threadIdx.x] = c, partial_bad[threadIdx.x] = bad;
    __syncthreads();
    for (int off = 512; off >= 1; off >>= 1) {
        if ((int)threadIdx.x < off) partial[threadIdx.x] += partial[threadIdx.x + off], partial_bad[threadIdx.x] += partial_bad[threadIdx.x + off];
        __syncthreads();
    }
    const int n = partial[0];
    const float scale = n == 0 ? 0.f : (mean ? 1.0f / (float)n : 1.0f);
    for (int64_t i = threadIdx.x; i < rows; i += 1024) {
        row_scale[i] = label_counts(labels[i], vocab, ignore_index) ? scale : 0.f;
        run_max[i] = -INFINITY, run_sum[i] = 0.f, target[i] = 0.f;
    }
    if (threadIdx.x == 0 && status) status[0] = n, status[1] = partial_bad[0];
}

// One workgroup per row.  The row's block of logits is read once and kept in registers (four 16-byte pieces per lane);
// it becomes p = exp(logit - running max) in place (bf16), alpha = exp(old max - new max) rescales what was accumulated so
// far.  HBM-bound: 27.7 us per 4096 x 8192 block when the block was read twice.
constexpr int kStreamPieces = 4;
template <int kStreamThreads>
__global__ __launch_bounds__(kStreamThreads) void ce_stream_block_kernel(bf16_t* slab, int64_t ld, int nb, int64_t v0, const int64_t* labels, float* run_max,
                                                                         float* run_sum, float* target, float* alpha, int64_t* run_arg) {
    constexpr int kWaves = kStreamThreads / 64;
    __shared__ float red[2][kWaves];
    __shared__ int red_i[kWaves];
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint4* p = (uint4*)(slab + row * ld);
    const int chunks = (nb + 63) / 64 * 8;  // the contraction of the grad-input launch runs to the next multiple of 64
    const int64_t label = labels[row];
    const float m_old = run_max[row];
    uint4 v[kStreamPieces];
    float bm = -INFINITY;
#pragma unroll
    for (int i = 0; i < kStreamPieces; i++) {
        const int c8 = i * kStreamThreads + threadIdx.x;
        if (c8 >= chunks) continue;
        v[i] = p[c8];
        const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x = (e & 1) ? bf16_hi(w[e >> 1]) : bf16_lo(w[e >> 1]);
            const int col = c8 * 8 + e;
            if (col < nb) bm = fmaxf(bm, x);
            if (v0 + col == label && col < nb) target[row] = x;  // (an ignore_index inside the range is masked by its zero row scale)
        }
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) bm = fmaxf(bm, __shfl_xor(bm, off, 64));
    if (lane == 0) red[0][wave] = bm;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; w++) bm = fmaxf(bm, red[0][w]);
    const float m_new = fmaxf(m_old, bm);
    float sum = 0.f;
    int first = 0x7FFFFFFF;  // first column of the block that holds the block's maximum
#pragma unroll
    for (int i = 0; i < kStreamPieces; i++) {
        const int c8 = i * kStreamThreads + threadIdx.x;
        if (c8 >= chunks) continue;
        const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float g[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float logit = h ? bf16_hi(w[e]) : bf16_lo(w[e]);
                const int col = c8 * 8 + 2 * e + h;
                if (col < nb && logit == bm) first = min(first, col);
                g[h] = col < nb ? __expf(logit - m_new) : 0.0f;
            }
            o[e] = pack_bf16(g[0], g[1]);
            // the sum runs over the rounded values the accumulator receives, so that numerator and denominator agree
            sum += bf16_lo(o[e]) + bf16_hi(o[e]);
        }
        p[c8] = make_uint4(o[0], o[1], o[2], o[3]);
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        sum += __shfl_xor(sum, off, 64);
        first = min(first, __shfl_xor(first, off, 64));
    }
    if (lane == 0) red[1][wave] = sum, red_i[wave] = first;
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
        for (int w = 0; w < kWaves; w++) total += red[1][w], first = min(first, red_i[w]);
        // a later block takes the argmax over only with a strictly larger maximum: equal maxima keep the first column
        if (run_arg && bm > m_old) run_arg[row] = v0 + first;
        const float a = m_old == -INFINITY ? 0.f : __expf(m_old - m_new);
        alpha[row] = a;
        run_sum[row] = run_sum[row] * a + total;
        run_max[row] = m_new;
    }
}

__global__ void fill_f32_kernel(float* p, int64_t n, float v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

static unsigned grid1d(int64_t n) {
    int64_t g = (n + 255) / 256;
    return (unsigned)(g < 1 ? 1 : (g > 16384 ? 16384 : g));
}

static void launch_stream_block(int rows, bf16_t* slab, int64_t ld, int nb, int64_t v0, const int64_t* labels, float* run_max, float* run_sum, float* target, float* alpha,
                                int64_t* run_arg, hipStream_t s) {
    static_assert(1024 * kStreamPieces * 8 >= kMaxVocabBlock, "a block fits the registers of one workgroup");
    if (nb <= 256 * kStreamPieces * 8)
        hipLaunchKernelGGL(ce_stream_block_kernel<256>, dim3((unsigned)rows), dim3(256), 0, s, slab, ld, nb, v0, labels, run_max, run_sum, target, alpha, run_arg);
    else if (nb <= 512 * kStreamPieces * 8)
        hipLaunchKernelGGL(ce_stream_block_kernel<512>, dim3((unsigned)rows), dim3(512), 0, s, slab, ld, nb, v0, labels, run_max, run_sum, target, alpha, run_arg);
    else
        hipLaunchKernelGGL(ce_stream_block_kernel<1024>, dim3((unsigned)rows), dim3(1024), 0, s, slab, ld, nb, v0, labels, run_max, run_sum, target, alpha, run_arg);
}

// Packed rows of the labels (row 0 for ignored or out-of-range labels: their gradient is zero or undefined anyway).
__global__ __launch_bounds__(256) void gather_label_rows_kernel(const uint8_t* packed, int64_t row_bytes, const int64_t* labels, int64_t vocab, uint8_t* out) {
    const int64_t row = blockIdx.x;
    const int64_t label = labels[row];
    const uint16_t* src = (const uint16_t*)(packed + (label >= 0 && label < vocab ? label : 0) * row_bytes);
    uint16_t* dst = (uint16_t*)(out + row * row_bytes);
    for (int64_t i = threadIdx.x; i < row_bytes / 2; i += 256) dst[i] = src[i];
}

// lse, loss and dH = ((acc / sum) - W[label]) * row_scale, rounded to bf16.  One workgroup per row.
__global__ __launch_bounds__(256) void ce_stream_finish_kernel(const float* acc, const bf16_t* w_label, int64_t hidden, const int64_t* labels, int64_t vocab,
                                                               const float* run_max, const float* run_sum, const float* target, const float* row_scale,
                                                               float* lse_out, float* loss_out, bf16_t* grad_hidden, int64_t ignore_index,
                                                               const int64_t* run_arg, int64_t* predicted, float* correct) {
    const int64_t row = blockIdx.x;
    const float rs = row_scale[row], inv = 1.0f / run_sum[row];
    const int64_t label = labels[row];
    const bool has_target = label_counts(label, vocab, ignore_index);
    if (threadIdx.x == 0) {
        const float lse = run_max[row] + __logf(run_sum[row]);
        lse_out[row] = lse;
        loss_out[row] = rs != 0.f ? (lse - (has_target ? target[row] : 0.f)) * rs : 0.f;
        if (run_arg) {
            const int64_t arg = run_arg[row];
            if (correct) correct[row] = has_target && arg == label ? 1.0f : 0.0f;
            if (predicted) predicted[row] = has_target ? arg : -1;  // (may be the running storage itself: read first)
        }
    }
    for (int64_t c = threadIdx.x; c < hidden; c += 256) {
        const float wl = has_target ? bf16_to_f32(w_label[row * hidden + c]) : 0.f;
        grad_hidden[row * hidden + c] = to_bf16((acc[row * hidden + c] * inv - wl) * rs);
    }
}

static int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// The logits and grad-input launches of a block run over decoded panels where the rows are enough to pay for decoding
// (dense_takes), on the packed-weight tile kernel otherwise.
int64_t lmhead_ce_workspace_bytes(int64_t rows, int64_t vocab, int64_t hidden, int64_t chunk) {
    (void)chunk;
    const int64_t gr = std::min(rows, kGradRows), nb = vocab_block(rows, vocab);
    const int64_t last = rows % kGradRows ? rows % kGradRows : gr;  // (fewer rows may want more splits)
    return align256(rows * 4) * 6 + align256(rows * 8) + align256(gr * nb * 2) + align256(gr * hidden * 4) + align256(gr * hidden * 2) * 2 + 1024 +
           std::max(dense_workspace_bytes(gr, nb, hidden), dense_workspace_bytes(last, nb, hidden));
}

int lmhead_ce(int qt, const void* hidden, const void* packed, const int64_t* labels, int64_t rows, int64_t vocab,
              int64_t hidden_dim, int64_t chunk, int64_t ignore_index, int reduction_mean, float* loss_1d,
              void* grad_hidden, float* lse_out, int* n_valid_out, int64_t* predicted, float* correct, void* ws, int64_t ws_bytes, hipStream_t s) {
    if (rows < 0 || vocab <= 0 || hidden_dim <= 0 || chunk <= 0) return set_error(GGQ_ERR_SHAPE, "lmhead_ce: bad shape");
    if (rows >= (1 << 30) || vocab >= (1 << 30)) return set_error(GGQ_ERR_SHAPE, "lmhead_ce: shape too large");
    if (!hidden || !packed || !labels || !loss_1d || !grad_hidden || !ws) return set_error(GGQ_ERR_NULL, "lmhead_ce: null pointer");
    if (ws_bytes < lmhead_ce_workspace_bytes(rows, vocab, hidden_dim, chunk)) return set_error(GGQ_ERR_WORKSPACE, "lmhead_ce: workspace too small");
    if (((uintptr_t)hidden | (uintptr_t)packed | (uintptr_t)grad_hidden | (uintptr_t)ws) & 15) return set_error(GGQ_ERR_ALIGN, "lmhead_ce: pointers must be 16-byte aligned");
    if (rows == 0) return GGQ_OK;
    const int64_t gr_max = std::min(rows, kGradRows);
    const int block = vocab_block(rows, vocab);
    char* w = (char*)ws;
    float* row_scale = (float*)w; w += align256(rows * 4);
    float* lse = lse_out ? lse_out : (float*)w; w += align256(rows * 4);
    float* target = (float*)w; w += align256(rows * 4);
    float* run_max = (float*)w; w += align256(rows * 4);
    float* run_sum = (float*)w; w += align256(rows * 4);
    float* alpha = (float*)w; w += align256(rows * 4);
    int64_t* run_arg = (predicted || correct) ? (int64_t*)w : nullptr; w += align256(rows * 8);  // running argmax column per row
    bf16_t* slab = (bf16_t*)w; w += align256(gr_max * block * 2);
    float* dh32 = (float*)w; w += align256(gr_max * hidden_dim * 4);
    uint8_t* label_rows = (uint8_t*)w; w += align256(gr_max * hidden_dim * 2);  // packed rows are smaller than bf16 rows
    bf16_t* w_label = (bf16_t*)w; w += align256(gr_max * hidden_dim * 2);
    void* panels = w;
    const int64_t panel_bytes = (char*)ws + ws_bytes - w;

    const int64_t row_bytes = packed_row_bytes(qt, hidden_dim);
    if (row_bytes <= 0 || row_bytes > hidden_dim * 2 || (row_bytes & 1)) return set_error(GGQ_ERR_QTYPE, "lmhead_ce: unsupported packed row size");
    hipLaunchKernelGGL(ce_row_scale_kernel, dim3(1), dim3(1024), 0, s, labels, rows, vocab, ignore_index, reduction_mean, row_scale, n_valid_out, run_max, run_sum, target);
    for (int64_t r0 = 0; r0 < rows; r0 += gr_max) {
        const int rc = (int)std::min(rows - r0, gr_max);
        const bf16_t* hid = (const bf16_t*)hidden + r0 * hidden_dim;
        for (int64_t v0 = 0; v0 < vocab; v0 += block) {
            const int nb = (int)std::min<int64_t>(vocab - v0, block);
            const uint8_t* wb = (const uint8_t*)packed + v0 * row_bytes;
            // (1) the block's logits
            DenseCall q{};
            q.qt = qt, q.mode = kModeNT, q.m = rc, q.n = nb, q.k = hidden_dim, q.a = hid, q.lda = hidden_dim, q.w = wb, q.c = slab, q.ldc = block;
            const bool panel_path = dense_takes(kModeNT, rc, nb, hidden_dim, hid, hidden_dim) && dense_takes(kModeNN, rc, nb, hidden_dim, slab, block, true);
            if (panel_path) {
                if (int rcode = dense_mmq(q, panels, panel_bytes, s)) return rcode;
            } else {
                MmqParams g;
                if (int rcode = init_params(g, qt, kModeNT, rc, nb, (int)hidden_dim, 1)) return rcode;
                g.a[0] = hid, g.lda = hidden_dim, g.w[0] = wb, g.c[0] = slab, g.ldc = block;
                if (int rcode = launch_mmq(qt, kModeNT, kEpiStore, g, s)) return rcode;
            }
            // (2) running statistics; the slab becomes exp(logit - running max)
            launch_stream_block(rc, slab, block, nb, v0, labels + r0, run_max + r0, run_sum + r0, target + r0, alpha + r0, run_arg ? run_arg + r0 : nullptr, s);
            // (3) acc = acc * alpha + p . W_block; the first block starts the accumulator
            if (panel_path) {
                q.mode = kModeNN, q.a = slab, q.lda = block, q.a_zero_padded = true, q.c = dh32, q.ldc = hidden_dim;
                q.panel_ready = dense_panel_whole(nb, hidden_dim), q.fp32 = true, q.accumulate = v0 > 0, q.row_scale = alpha + r0;
                if (int rcode = dense_mmq(q, panels, panel_bytes, s)) return rcode;
            } else {
                if (v0 == 0) hipLaunchKernelGGL(fill_f32_kernel, dim3(grid1d((int64_t)rc * hidden_dim)), dim3(256), 0, s, dh32, (int64_t)rc * hidden_dim, 0.f);
                MmqParams b;
                if (int rcode = init_params(b, qt, kModeNN, rc, nb, (int)hidden_dim, 1)) return rcode;
                b.a[0] = slab, b.lda = block, b.a_zero_padded = 1, b.w[0] = wb, b.c[0] = dh32, b.ldc = hidden_dim, b.row_scale = alpha + r0;
                if (int rcode = launch_mmq(qt, kModeNN, kEpiAccumF32, b, s)) return rcode;
            }
        }
        hipLaunchKernelGGL(gather_label_rows_kernel, dim3((unsigned)rc), dim3(256), 0, s, (const uint8_t*)packed, row_bytes, labels + r0, vocab, label_rows);
        if (int rcode = dequantize(qt, label_rows, rc, hidden_dim, w_label, 0, s)) return rcode;
        hipLaunchKernelGGL(ce_stream_finish_kernel, dim3((unsigned)rc), dim3(256), 0, s, dh32, w_label, hidden_dim, labels + r0, vocab, run_max + r0, run_sum + r0,
                           target + r0, row_scale + r0, lse + r0, loss_1d + r0, (bf16_t*)grad_hidden + r0 * hidden_dim, ignore_index,
                           run_arg ? run_arg + r0 : nullptr, predicted ? predicted + r0 : nullptr, correct ? correct + r0 : nullptr);
    }
    return check_launch("lmhead_ce");
}

}  // namespace ggq
