// The numbering of the WENO work items (st_items.h), built for the host: every
// segment's first, middle and last item must be found in it, and the waves of
// the item kernel must reach every pair of items, on grids up to the largest a solver
// takes and with segments that are all full, all listed or mixed.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../streams-2_amd/csrc/st_items.h"

using namespace st;

#define CHECK(c)                                                                                     \
    do {                                                                                             \
        if (!(c)) {                                                                                  \
            std::printf("%dx%dx%d pattern %d: %s (line %d)\n", g.nx, g.ny, g.nz, pat, #c, __LINE__); \
            return 1;                                                                                \
        }                                                                                            \
    } while (0)

// pattern 0: every cell has its three items; 1: full segments, lists and empty
// segments in turn; 2: every list as long as its room
static int run(int nx, int ny, int nz, int pat) {
    Geo g{};
    g.nx = nx; g.ny = ny; g.nz = nz; g.ng = 3;
    g.nint = (long long)nx * ny * nz;
    int wpt;
    const int nseg = item_segments(g, &wpt), nwx = rec_per_row(g), nwords = nwx * ny * nz;
    CHECK(nseg >= 1 && nseg <= kItemSeg);
    std::vector<int> counts(nseg);
    std::vector<pair_t> pre(nseg + 1);
    long long exact = 0;
    pair_t run = 0;
    for (int q = 0; q < nseg; q++) {
        const int s0 = seg_first_cell(g, nwx, q * 256 * wpt, nwords), s1 = seg_first_cell(g, nwx, (q + 1) * 256 * wpt, nwords);
        CHECK(s0 >= 0 && s1 > s0 && s1 <= g.nint && (q > 0 || s0 == 0) && (q < nseg - 1 || s1 == g.nint));
        CHECK(s1 - s0 < 1 << 24);  // an item's cell bits
        const int cells = s1 - s0, total = pat == 0 ? 3 * cells : (pat == 2 ? cells : (q % 3 == 0 ? 3 * cells : (q % 3 == 1 ? cells / 7 : 0)));
        counts[q] = segment_report(total, cells);
        CHECK(counts[q] == (total > cells ? -3 * cells : total));
        pre[q] = run;
        run += segment_pairs(counts[q]);
        exact += (segment_items(counts[q]) + 1) / 2;
    }
    pre[nseg] = run;
    CHECK((long long)run == exact);
    CHECK(pat != 0 || (2 * exact >= 3 * g.nint && 2 * exact <= 3 * g.nint + nseg));
    long long at = 0;
    for (int q = 0; q < nseg; q++) {
        const int n = segment_items(counts[q]), s0 = seg_first_cell(g, nwx, q * 256 * wpt, nwords);
        for (int x : {0, n / 2, n - 1}) {
            if (n == 0) continue;
            const pair_t e = (pair_t)(at + x / 2);
            CHECK(pair_segment(pre.data(), nseg, e) == q);
            CHECK(2 * (int)(e - pre[q]) + x % 2 == x);
            if (counts[q] < 0) CHECK(s0 + x / 3 < g.nint);
        }
        at += (n + 1) / 2;
    }
    // 512 workgroups of four waves, 31 pairs a wave and round
    const unsigned nwaves = 2048;
    for (unsigned wave : {0u, 1u, nwaves / 2, nwaves - 1}) {
        long long rounds = 0, want = (exact - 31LL * wave + 31LL * nwaves - 1) / (31LL * nwaves);
        for (pair_t base = wave * 31; base < run && rounds <= want; base += nwaves * 31) rounds++;
        CHECK(rounds == (want > 0 ? want : 0));
    }
    return 0;
}

int main() {
    const int grids[][3] = {{3, 3, 3}, {64, 17, 8}, {131, 97, 90}, {3, 8000, 8000}, {894, 894, 894}, {897, 897, 897},
                            {1024, 1024, 1024}, {1264, 1264, 1264}};
    int bad = 0;
    for (auto &n : grids)
        for (int pat = 0; pat < 3; pat++) bad += run(n[0], n[1], n[2], pat);
    return bad ? 1 : 0;
}
