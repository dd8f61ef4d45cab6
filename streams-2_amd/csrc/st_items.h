// st_items.h -- index arithmetic of the WENO work items of the one-pass stage
// (st_stage.hip): cell records, list segments and the numbering of the items,
// for the kernels and for host code.
#pragma once

#include "st_internal.h"

namespace st {

// Cell records, one per 64 cells of an interior row (row-major over j, k):
// words 2d and 2d+1 hold the lower-face and upper-face bits of direction d
// (words 6, 7 unused: a record is one 64-byte sector).
constexpr int kRecWords = 8;
constexpr int kItemSeg = 4096;  // list segments at most

// A launch numbers its items in pairs, a segment of an odd number ending in a
// blank.  A cell has up to three items: a grid of 2^31 points, the largest a
// solver takes, has 3.2e9 pairs at most, where the items themselves would not
// fit 32 bits.  (64-bit numbers in the kernel's search and prefix: 269 us for
// the 262 of this on 512 x 256 x 256, the masks of the step averaged in.)
using pair_t = unsigned;

__host__ __device__ __forceinline__ int rec_per_row(const Geo &g) { return (g.nx + 63) / 64; }

// The first cell of record wd, and with it of the segment that starts there.
__host__ __device__ __forceinline__ int seg_first_cell(const Geo &g, int nwx, int wd, int nwords) {
    return wd >= nwords ? (int)g.nint : (wd / nwx) * g.nx + 64 * (wd % nwx);
}

// Segments of 256 * wpt records, at most kItemSeg of them.
inline int item_segments(const Geo &g, int *wpt) {
    const long nwords = (long)rec_per_row(g) * g.ny * g.nz;
    long per = (nwords + 256L * kItemSeg - 1) / (256L * kItemSeg);
    if (per < 1) per = 1;
    *wpt = (int)per;
    return (int)((nwords + 256 * per - 1) / (256 * per));
}

// What a segment reports of its `total` items: their number where its list, of
// one slot a cell, holds them; otherwise the list stays empty, its items are
// all (cell, direction) pairs and the report is minus their number.
__host__ __device__ __forceinline__ int segment_report(int total, int cells) { return total > cells ? -3 * cells : total; }

__host__ __device__ __forceinline__ int segment_items(int report) { return report < 0 ? -report : report; }
__host__ __device__ __forceinline__ pair_t segment_pairs(int report) { return (pair_t)((segment_items(report) + 1) >> 1); }

// The segment of a pair: the last one that starts at or before it (pre[q] is
// the first pair of segment q, pre[nseg] their number).
__host__ __device__ __forceinline__ int pair_segment(const pair_t *pre, int nseg, pair_t e) {
    int lo = 0, hi = nseg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pre[mid] <= e) lo = mid;
        else hi = mid;
    }
    return lo;
}

}  // namespace st
