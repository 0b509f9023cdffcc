// Row-tile tables of an expert-sorted layout, as a device function that several launches share.
#pragma once
#include "common.h"
#include "mmq_host.h"

namespace ggq {

// Inclusive prefix sum over the 256 threads of the workgroup: a shuffle scan inside each wave, then the wave totals
// through LDS (one barrier; `totals` must not be reused before the next barrier of the caller).
__device__ __forceinline__ int block_scan_inclusive(int v, int tid, int* totals) {
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(v, off, 64);
        if (lane >= off) v += u;
    }
    if (lane == 63) totals[wave] = v;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int w = 0; w < 3; w++) before += w < wave ? totals[w] : 0;
    return v + before;
}

// Table t, by 256 threads (tid 0..255, whole waves); groups are walked 256 at a time with a prefix sum, so
// a table is in group order and identical from run to run.  Table t keeps the groups with
// min_rows[t] < rows <= max_rows[t] and cuts them into tiles of bm[t] rows.
__device__ __forceinline__ void build_row_tiles_body(const int64_t* expert_ids, const int32_t* end_offsets, int groups, const RowTileTables& tb, int* expert_ranges,
                                                     int num_experts, int t, int tid) {
    __shared__ int totals[2][4];
    const int bm = tb.bm[t], min_rows = tb.min_rows[t], max_rows = tb.max_rows[t];
    TileDesc* tiles = tb.tiles[t];
    if (expert_ranges && t == 0) {
        for (int e = tid; e < num_experts; e += 256) expert_ranges[2 * e] = expert_ranges[2 * e + 1] = 0;
        __syncthreads();  // (the ranges of the listed groups are written below, by other threads)
    }
    int base = 0;  // tiles of the groups walked so far (the same value in every thread)
    int flip = 0;
    for (int g0 = 0; g0 < groups; g0 += 256) {
        const int g = g0 + tid;
        int r0 = 0, r1 = 0, count = 0, expert = 0;
        if (g < groups) {
            expert = expert_ids ? (int)expert_ids[g] : g;
            r0 = g == 0 ? 0 : end_offsets[g - 1];
            r1 = end_offsets[g];
            count = (r1 - r0 > min_rows && r1 - r0 <= max_rows) ? (r1 - r0 + bm - 1) / bm : 0;
            if (expert_ranges && t == 0) {
                const int64_t e = expert_ids ? expert_ids[g] : g;
                if (e >= 0 && e < num_experts) expert_ranges[2 * e] = r0, expert_ranges[2 * e + 1] = r1;
            }
        }
        const int incl = block_scan_inclusive(count, tid, totals[flip]);
        const int first = base + incl - count;
        for (int i = 0; i < count; i++) {
            TileDesc d;
            d.group = g, d.row_begin = r0 + i * bm, d.row_end = min(r1, r0 + (i + 1) * bm), d.expert = expert;
            tiles[first + i] = d;
        }
        base += totals[flip][0] + totals[flip][1] + totals[flip][2] + totals[flip][3];
        flip ^= 1;  // the next round's totals go to the other row: no barrier needed between the rounds
    }
    if (tid == 0) *tb.num_tiles[t] = base;
    TileDesc* by_size = tb.by_size[t];
    if (!by_size) return;
    // Stable bucket sort by the number of 32-row blocks, largest first: thread i takes the i-th contiguous share of the
    // table; the per-thread bucket counts are scanned over the threads, bucket after bucket.
    __syncthreads();  // the table written above is visible to the whole workgroup
    constexpr int kBuckets = 8;  // tiles of up to 256 rows
    __shared__ int bucket_totals[kBuckets][4];
    const int total = base;
    const int share = (total + 255) / 256, i0 = min(total, tid * share), i1 = min(total, i0 + share);
    int mine[kBuckets];
#pragma unroll
    for (int b = 0; b < kBuckets; b++) mine[b] = 0;
    for (int i = i0; i < i1; i++) {
        const int bucket = kBuckets - min(kBuckets, max(1, (tiles[i].row_end - tiles[i].row_begin + 31) >> 5));
#pragma unroll
        for (int b = 0; b < kBuckets; b++) mine[b] += bucket == b;
    }
    int at[kBuckets];  // position of this thread's first tile of bucket b
    int run = 0;
#pragma unroll
    for (int b = 0; b < kBuckets; b++) {
        const int incl = block_scan_inclusive(mine[b], tid, bucket_totals[b]);
        at[b] = run + incl - mine[b];
        run += bucket_totals[b][0] + bucket_totals[b][1] + bucket_totals[b][2] + bucket_totals[b][3];
    }
    for (int i = i0; i < i1; i++) {
        const TileDesc d = tiles[i];
        const int bucket = kBuckets - min(kBuckets, max(1, (d.row_end - d.row_begin + 31) >> 5));
        int pos = 0;
#pragma unroll
        for (int b = 0; b < kBuckets; b++) {
            if (bucket == b) pos = at[b];
            at[b] += bucket == b;
        }
        by_size[pos] = d;
    }
}

}  // namespace ggq
