// Host launchers for the packed-weight tile kernel, the expert row-tile table and the error state.
#include "mmq_tile.h"
#include "mmq_direct8.h"
#include "mmq_direct8_nn.h"
#include "mmq_small_nn.h"
#include "mmq_small_iq2.h"
#include "mmq_small_nn_iq2.h"
#include "launch.h"

#include <stdarg.h>
#include <stdio.h>
#include "row_tiles.h"

namespace ggq {

// ------------------------------------------------------------------------------------------------
static thread_local char g_last_error[512] = "";

int set_error(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
    va_end(ap);
    return code;
}
const char* last_error() { return g_last_error; }

int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(GGQ_ERR_RUNTIME, "%s: %s", what, hipGetErrorString(e));
    return GGQ_OK;
}

// ------------------------------------------------------------------------------------------------
// Row-tile tables.  One workgroup per table.
__global__ __launch_bounds__(256) void build_row_tiles_kernel(const int64_t* expert_ids, const int32_t* end_offsets, int groups, RowTileTables tb, int* expert_ranges,
                                                              int num_experts) {
    build_row_tiles_body(expert_ids, end_offsets, groups, tb, expert_ranges, num_experts, blockIdx.x, threadIdx.x);
}

int build_row_tile_tables(const int64_t* expert_ids, const int32_t* end_offsets, int groups, const RowTileTables& tb,
                          int* expert_ranges, int num_experts, hipStream_t s) {
    if (tb.count <= 0) return GGQ_OK;
    hipLaunchKernelGGL(build_row_tiles_kernel, dim3(tb.count), dim3(256), 0, s, expert_ids, end_offsets, groups, tb,
                       expert_ranges, num_experts);
    return check_launch("build_row_tiles");
}

int build_row_tiles(const int64_t* expert_ids, const int32_t* end_offsets, int groups, int bm, TileDesc* tiles,
                    int* num_tiles, int* expert_ranges, int num_experts, hipStream_t s, int min_rows, int max_rows) {
    RowTileTables tb{};
    tb.add(bm, min_rows, max_rows, tiles, num_tiles);
    return build_row_tile_tables(expert_ids, end_offsets, groups, tb, expert_ranges, num_experts, s);
}

// ------------------------------------------------------------------------------------------------
// Optional per-launch timing of the tile kernel with HIP events on the launch stream (off by default).
struct TimedLaunch {
    hipEvent_t start, stop;
    int qt, mode, epi, shape;
};
static TimedLaunch g_timed[kMaxTimedLaunches];
static int g_timed_count = 0;
static bool g_timing = false;

int profile_begin() {
    g_timed_count = 0;
    g_timing = true;
    return GGQ_OK;
}

int profile_end(float* ms, int* qt, int* mode, int* epi, int* shape, int capacity) {
    g_timing = false;
    int n = 0;
    for (int i = 0; i < g_timed_count; i++) {
        float t = 0.f;
        if (hipEventSynchronize(g_timed[i].stop) != hipSuccess || hipEventElapsedTime(&t, g_timed[i].start, g_timed[i].stop) != hipSuccess)
            return set_error(GGQ_ERR_RUNTIME, "profile_end: event query failed");
        if (n < capacity) {
            ms[n] = t, qt[n] = g_timed[i].qt, mode[n] = g_timed[i].mode, epi[n] = g_timed[i].epi;
            if (shape) shape[n] = g_timed[i].shape;
            n++;
        }
        (void)hipEventDestroy(g_timed[i].start);
        (void)hipEventDestroy(g_timed[i].stop);
    }
    g_timed_count = 0;
    return n;
}

TimedScope::TimedScope(int qt, int mode, int epi, int shape, hipStream_t s) : stream_(s) {
    if (!g_timing || g_timed_count >= kMaxTimedLaunches) return;
    TimedLaunch* t = &g_timed[g_timed_count];
    if (hipEventCreate(&t->start) != hipSuccess || hipEventCreate(&t->stop) != hipSuccess) return;
    t->qt = qt, t->mode = mode, t->epi = epi, t->shape = shape;
    slot_ = g_timed_count++;
    (void)hipEventRecord(t->start, s);
}
TimedScope::~TimedScope() {
    if (slot_ >= 0) (void)hipEventRecord(g_timed[slot_].stop, stream_);
}

template <int QT, int MODE, int EPI, int SH>
static int launch_one(const MmqParams& p, hipStream_t s) {
    const int col_tiles = (MODE == kModeNT ? p.nseg : 1) * p.col_tiles_per_seg;
    const int64_t total = (int64_t)p.max_row_tiles * col_tiles;
    if (total <= 0) return GGQ_OK;
    const int64_t grid = (total + 7) / 8 * 8;  // the XCD remap inside the kernel needs a multiple of 8
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "mmq: too many tiles for one launch");
    TimedLaunch* t = nullptr;
    if (g_timing && g_timed_count < kMaxTimedLaunches) {
        t = &g_timed[g_timed_count];
        if (hipEventCreate(&t->start) != hipSuccess || hipEventCreate(&t->stop) != hipSuccess) return set_error(GGQ_ERR_RUNTIME, "mmq: event creation failed");
        t->qt = QT, t->mode = MODE, t->epi = EPI, t->shape = SH;
        g_timed_count++;
        (void)hipEventRecord(t->start, s);
    }
    constexpr int kSmemBytes = Tile<SH>::kTileLdsBytes + (QT == kIQ2_XXS ? Fmt<kIQ2_XXS>::kTableWords * 4 : 0) +
                               (EPI != kEpiStore ? Tile<SH>::kTM * 16 : 0);
    static LdsLimit lds_limit;  // per instantiation
    if (int rc = raise_lds_limit(lds_limit, (const void*)mmq_tile_kernel<QT, MODE, EPI, SH>, kSmemBytes, "mmq")) return rc;
    hipLaunchKernelGGL((mmq_tile_kernel<QT, MODE, EPI, SH>), dim3((unsigned)grid), dim3(kThreads), kSmemBytes, s, p);
    if (t) (void)hipEventRecord(t->stop, s);
    return check_launch("mmq_tile_kernel");
}

// Q4_K, store epilogue, direct shape: forward or grad-input.
template <int MODE>
static int launch_direct(const MmqParams& p, hipStream_t s) {
    const int col_tiles = (MODE == kModeNT ? p.nseg : 1) * p.col_tiles_per_seg;
    if (p.col_tiles_per_wg < 1) return set_error(GGQ_ERR_SHAPE, "mmq: column tiles per workgroup must be at least 1");
    const bool few_rows = MODE == kModeNN && p.few_rows;  // 512 columns per workgroup
    if (few_rows && ((p.k & 511) || p.r_pad > 32)) return set_error(GGQ_ERR_SHAPE, "mmq: the grad-input kernel for few rows needs whole pairs of blocks and ranks up to 32");
    // row tiles are dealt round-robin over the eight XCDs; each XCD walks its row tiles' column-tile runs
    const int per_wg = few_rows ? 2 : p.col_tiles_per_wg;
    const int64_t total = (int64_t)((p.max_row_tiles + 7) / 8) * ((col_tiles + per_wg - 1) / per_wg);
    if (total <= 0) return GGQ_OK;
    const int64_t grid = total * 8;
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "mmq: too many tiles for one launch");
    if (MODE == kModeNN && ((p.n & 63) || ((p.nseg * p.steps_per_seg) & 1) || p.nseg * p.steps_per_seg < 4))
        return set_error(GGQ_ERR_SHAPE, "mmq: the direct grad-input kernel needs an even number, four or more, of whole 64-row steps");
    TimedLaunch* t = nullptr;
    if (g_timing && g_timed_count < kMaxTimedLaunches) {
        t = &g_timed[g_timed_count];
        if (hipEventCreate(&t->start) != hipSuccess || hipEventCreate(&t->stop) != hipSuccess) return set_error(GGQ_ERR_RUNTIME, "mmq: event creation failed");
        t->qt = kQ4_K, t->mode = MODE, t->epi = kEpiStore, t->shape = few_rows ? kShapeSmall : kShapeDirect;
        g_timed_count++;
        (void)hipEventRecord(t->start, s);
    }
    if (few_rows) {  // (its 43 KB need no raised limit)
        hipLaunchKernelGGL(mmq_small_nn_q4k_kernel, dim3((unsigned)grid), dim3(SmallNN::kThreadsWG), SmallNN::kLdsBytes, s, p);
        if (t) (void)hipEventRecord(t->stop, s);
        return check_launch("mmq_small_nn_q4k_kernel");
    }
    constexpr int kSmemBytes = MODE == kModeNT ? Direct8::kLdsBytes : Direct8NN::kLdsBytes;
    const void* fn = MODE == kModeNT ? (const void*)mmq_direct8_q4k_kernel : (const void*)mmq_direct8_nn_q4k_kernel;
    static LdsLimit lds_limit;  // per instantiation
    if (int rc = raise_lds_limit(lds_limit, fn, kSmemBytes, "mmq")) return rc;
    if (MODE == kModeNT) hipLaunchKernelGGL(mmq_direct8_q4k_kernel, dim3((unsigned)grid), dim3(Direct8::kThreadsWG), kSmemBytes, s, p);
    else hipLaunchKernelGGL(mmq_direct8_nn_q4k_kernel, dim3((unsigned)grid), dim3(Direct8NN::kThreadsWG), kSmemBytes, s, p);
    if (t) (void)hipEventRecord(t->stop, s);
    return check_launch(MODE == kModeNT ? "mmq_direct8_q4k_kernel" : "mmq_direct8_nn_q4k_kernel");
}

template <int QT, int MODE>
static int launch_mixed_mode(const MmqParams& p, hipStream_t s) {
    const int segs = MODE == kModeNT ? p.nseg : 1;
    // per XCD: ceil(wide units / 8) * wide column tiles + ceil(tall units / 8) * tall column tiles slots
    const int64_t slots = (int64_t)((p.max_row_tiles + 7) / 8) * segs * p.col_tiles_per_seg +
                          (int64_t)((p.max_row_tiles2 + 7) / 8) * segs * p.col_tiles_per_seg2;
    if (slots <= 0) return GGQ_OK;
    const int64_t grid = slots * 8;
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "mmq: too many tiles for one launch");
    TimedLaunch* t = nullptr;
    if (g_timing && g_timed_count < kMaxTimedLaunches) {
        t = &g_timed[g_timed_count];
        if (hipEventCreate(&t->start) != hipSuccess || hipEventCreate(&t->stop) != hipSuccess) return set_error(GGQ_ERR_RUNTIME, "mmq: event creation failed");
        t->qt = QT, t->mode = MODE, t->epi = kEpiStore, t->shape = kShapeMixed;
        g_timed_count++;
        (void)hipEventRecord(t->start, s);
    }
    constexpr int kSmemBytes = (Tile<kShapeWide>::kTileLdsBytes > Tile<kShapeTall>::kTileLdsBytes ? Tile<kShapeWide>::kTileLdsBytes : Tile<kShapeTall>::kTileLdsBytes) +
                               (QT == kIQ2_XXS ? Fmt<kIQ2_XXS>::kTableWords * 4 : 0);
    static LdsLimit lds_limit;  // per instantiation
    if (int rc = raise_lds_limit(lds_limit, (const void*)mmq_mixed_kernel<QT, MODE, kEpiStore>, kSmemBytes, "mmq")) return rc;
    hipLaunchKernelGGL((mmq_mixed_kernel<QT, MODE, kEpiStore>), dim3((unsigned)grid), dim3(kThreads), kSmemBytes, s, p);
    if (t) (void)hipEventRecord(t->stop, s);
    return check_launch("mmq_mixed_kernel");
}

// IQ2_XXS, forward, store epilogue: tiles of up to kSmallBM rows (p.tiles) on the decoding-wave kernel.
int launch_mmq_small(const MmqParams& p, hipStream_t s) {
    const int col_tiles = p.nseg * p.col_tiles_per_seg;
    if (p.col_tiles_per_wg < 1) return set_error(GGQ_ERR_SHAPE, "mmq: column tiles per workgroup must be at least 1");
    if (p.steps_per_seg & 3) return set_error(GGQ_ERR_SHAPE, "mmq: the small-group kernel needs a contraction of whole 256-wide blocks");
    // row tiles are dealt round-robin over the eight XCDs; each XCD walks its row tiles' column-tile runs
    const int64_t total = (int64_t)((p.max_row_tiles + 7) / 8) * ((col_tiles + p.col_tiles_per_wg - 1) / p.col_tiles_per_wg);
    if (total <= 0) return GGQ_OK;
    const int64_t grid = total * 8;
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "mmq: too many tiles for one launch");
    TimedLaunch* t = nullptr;
    if (g_timing && g_timed_count < kMaxTimedLaunches) {
        t = &g_timed[g_timed_count];
        if (hipEventCreate(&t->start) != hipSuccess || hipEventCreate(&t->stop) != hipSuccess) return set_error(GGQ_ERR_RUNTIME, "mmq: event creation failed");
        t->qt = kIQ2_XXS, t->mode = kModeNT, t->epi = kEpiStore, t->shape = kShapeSmall;
        g_timed_count++;
        (void)hipEventRecord(t->start, s);
    }
    static LdsLimit lds_limit;
    if (int rc = raise_lds_limit(lds_limit, (const void*)mmq_small_iq2xxs_kernel, SmallIq2::kLdsBytes, "mmq")) return rc;
    hipLaunchKernelGGL(mmq_small_iq2xxs_kernel, dim3((unsigned)grid), dim3(SmallIq2::kThreadsWG), SmallIq2::kLdsBytes, s, p);
    if (t) (void)hipEventRecord(t->stop, s);
    return check_launch("mmq_small_iq2xxs_kernel");
}

// IQ2_XXS, grad-input, store epilogue: entries of up to kSmallNNIq2Rows rows (p.tiles).
int launch_mmq_small_nn(const MmqParams& p, hipStream_t s) {
    if ((p.k & 511) || (p.n & 127)) return set_error(GGQ_ERR_SHAPE, "mmq: the small-group grad-input kernel needs whole pairs of blocks and a contraction of whole groups of 128 rows");
    // row tiles are dealt round-robin over the eight XCDs; the column tiles of a row tile follow one another
    const int64_t grid = (int64_t)((p.max_row_tiles + 7) / 8) * (p.k / SmallNNIq2::kCols) * 8;
    if (grid <= 0) return GGQ_OK;
    if (grid > 0x7FFFFFF0) return set_error(GGQ_ERR_SHAPE, "mmq: too many tiles for one launch");
    TimedScope timed(kIQ2_XXS, kModeNN, kEpiStore, kShapeSmall, s);
    static LdsLimit lds_limit;
    if (int rc = raise_lds_limit(lds_limit, (const void*)mmq_small_nn_iq2xxs_kernel, SmallNNIq2::kLdsBytes, "mmq")) return rc;
    hipLaunchKernelGGL(mmq_small_nn_iq2xxs_kernel, dim3((unsigned)grid), dim3(SmallNNIq2::kThreadsWG), SmallNNIq2::kLdsBytes, s, p);
    return check_launch("mmq_small_nn_iq2xxs_kernel");
}

int launch_mmq_mixed(int qt, int mode, const MmqParams& p, hipStream_t s) {
#define GGQ_MIXED(QT) return mode == kModeNT ? launch_mixed_mode<QT, kModeNT>(p, s) : launch_mixed_mode<QT, kModeNN>(p, s)
    switch (qt) {
        case kQ8_0: GGQ_MIXED(kQ8_0);
        case kQ2_K: GGQ_MIXED(kQ2_K);
        case kQ3_K: GGQ_MIXED(kQ3_K);
        case kQ4_K: GGQ_MIXED(kQ4_K);
        case kQ5_K: GGQ_MIXED(kQ5_K);
        case kQ6_K: GGQ_MIXED(kQ6_K);
        case kIQ2_XXS: GGQ_MIXED(kIQ2_XXS);
    }
#undef GGQ_MIXED
    return set_error(GGQ_ERR_QTYPE, "unsupported GGML type id %d", qt);
}

template <int QT>
static int launch_qt(int mode, int epi, const MmqParams& p, hipStream_t s) {
    if (mode == kModeNT) {
        switch (epi) {
            case kEpiStore:
                if (QT == kQ4_K && p.shape == kShapeDirect) return launch_direct<kModeNT>(p, s);
                if (p.shape == kShapeWide) return launch_one<QT, kModeNT, kEpiStore, 1>(p, s);
                return launch_one<QT, kModeNT, kEpiStore, 0>(p, s);
        }
    } else {
        switch (epi) {
            case kEpiStore:
                if (QT == kQ4_K && p.shape == kShapeDirect) return launch_direct<kModeNN>(p, s);
                if (p.shape == kShapeWide) return launch_one<QT, kModeNN, kEpiStore, 1>(p, s);
                return launch_one<QT, kModeNN, kEpiStore, 0>(p, s);
            case kEpiAccumF32: return launch_one<QT, kModeNN, kEpiAccumF32, 0>(p, s);
        }
    }
    return set_error(GGQ_ERR_SHAPE, "mmq: unsupported mode/epilogue combination");
}

int launch_mmq(int qt, int mode, int epi, const MmqParams& p, hipStream_t s) {
    switch (qt) {
        case kQ8_0: return launch_qt<kQ8_0>(mode, epi, p, s);
        case kQ2_K: return launch_qt<kQ2_K>(mode, epi, p, s);
        case kQ3_K: return launch_qt<kQ3_K>(mode, epi, p, s);
        case kQ4_K: return launch_qt<kQ4_K>(mode, epi, p, s);
        case kQ5_K: return launch_qt<kQ5_K>(mode, epi, p, s);
        case kQ6_K: return launch_qt<kQ6_K>(mode, epi, p, s);
        case kIQ2_XXS: return launch_qt<kIQ2_XXS>(mode, epi, p, s);
    }
    return set_error(GGQ_ERR_QTYPE, "unsupported GGML type id %d (supported: 8 Q8_0, 10 Q2_K, 11 Q3_K, 12 Q4_K, 13 Q5_K, 14 Q6_K, 16 IQ2_XXS)", qt);
}

// Fills the shape-derived fields of a parameter block.  n, k describe one weight segment [n, k].
int init_params(MmqParams& p, int qt, int mode, int m, int n, int k, int nseg, int shape) {
    if (m < 0 || n <= 0 || k <= 0) return set_error(GGQ_ERR_SHAPE, "mmq: bad shape m=%d n=%d k=%d", m, n, k);
    if (packed_row_bytes(qt, k) < 0) return set_error(GGQ_ERR_QTYPE, "unsupported GGML type id %d", qt);
    if (!block_multiple(qt, k)) return set_error(GGQ_ERR_SHAPE, "mmq: K=%d is not a multiple of the block size of type %d", k, qt);
    if (k % 64) return set_error(GGQ_ERR_SHAPE, "mmq: K=%d must be a multiple of 64", k);
    p = MmqParams{};
    p.m = m, p.n = n, p.k = k, p.nseg = nseg;
    p.w_row_bytes = packed_row_bytes(qt, k);
    p.w_expert_bytes = p.w_row_bytes * n;
    if (shape == kShapeDirect && qt != kQ4_K) shape = kShapeTall;  // the decoding-wave kernels exist for Q4_K only
    const int bm = shape == kShapeDirect ? kDirectBM : shape == kShapeTall ? kBM : kWideBM;
    const int bn = shape == kShapeDirect ? kDirectBN : shape == kShapeWide ? kWideBN : kBN;
    p.shape = shape;
    if (mode == kModeNT) {
        p.col_tiles_per_seg = (n + bn - 1) / bn;
        p.steps_per_seg = k / kBK;
    } else {
        p.col_tiles_per_seg = (k + bn - 1) / bn;
        p.steps_per_seg = (n + kBK - 1) / kBK;
    }
    p.max_row_tiles = (m + bm - 1) / bm;
    p.col_tiles_per_wg = 1;
    return GGQ_OK;
}


}  // namespace ggq
