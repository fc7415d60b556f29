// lsmp_ccd_plan.h -- which CCD solve a pass over the lines of a direction takes
// and how many block sums it leaves.  The launcher, the size of the block sums'
// buffer and the check before a mass correction's launches all ask here.  Plain C++:
// the host tests build it too.
#pragma once
#include <algorithm>

namespace lsmp {

constexpr int KCC = 17;   // CCD rows per lane at most (9 up to 284 cells, 17 up to 540 with 32 lanes per line, 1084 with 64)

// every line of a direction goes through the partitioned (one wave or 32
// lanes per line) solves up to this count of y or z lines (x lines have none).  The
// nine solves of the energy integrals, one lane per line, then with 32 lanes
// along x only, then along y and z as well: 96^3 497, 393, 273 us; 160x96x128 663,
// 456, 372 (FP32 611, -, 271); 192^3 (36,864 lines) 1003, 835, 799 (FP32 889, 680,
// 565); 256^3 1546, 1380, 1583 (FP32 1272, 1038, 1061); 400x400x30 (160,000 z
// lines) 1358, 860, 937.
constexpr int PART_MAX_CCD_STRIDED = 40960;

// listed band lines solved with 32 lanes per line up to these counts (x lines
// are contiguous; y and z lines are strided, and 32 lanes on one of them read
// 32 separate cache lines per row)
#ifndef LSMP_PART_LISTED_X
#define LSMP_PART_LISTED_X (1 << 30)
#endif
#ifndef LSMP_PART_LISTED_STRIDED
#define LSMP_PART_LISTED_STRIDED (1 << 30)
#endif
constexpr int PART_MAX_LISTED_X = LSMP_PART_LISTED_X, PART_MAX_LISTED_STRIDED = LSMP_PART_LISTED_STRIDED;

// lanes: 64 or 32 a line (k_ccd_part), or 1 (k_ccd_seg); blocks of 256 threads
struct CcdPlan {
    int lanes;
    long blocks;
};
inline CcdPlan ccd_plan(int dir, int n, long nlines, bool listed)
{
    const long part_max = dir == 0 ? PART_MAX_LISTED_X : listed ? PART_MAX_LISTED_STRIDED : PART_MAX_CCD_STRIDED;
    int lanes = 1;
    if (nlines <= part_max) lanes = n + 4 <= 32 * KCC ? 32 : n + 4 <= 64 * KCC ? 64 : 1;
    const long per = 256 / lanes;   // lines a block
    return {lanes, (nlines + per - 1) / per};
}

// mass and volume of the unlisted lines (k_line_hsums): each line in segments of
// at least 32 cells, a block per 256 lines and segment
constexpr int LINE_SEGMENTS = 8;
inline int hsum_segments(int n) { return std::max(1, std::min(LINE_SEGMENTS, n / 32)); }
inline long hsum_blocks(int n, long nlines) { return (nlines + 255) / 256 * hsum_segments(n); }

// block sums a mass correction leaves at most in its final pass (z, in 2D y): of
// every line, or of the unlisted ones and then of up to as many listed lines
inline long mass_sums(int dim, int nx, int ny, int nz)
{
    const int dir = dim == 3 ? 2 : 1, n = dim == 3 ? nz : ny;
    const long lines = dim == 3 ? (long)nx * ny : nx;
    long listed = ccd_plan(dir, n, lines, true).blocks;
    if (lines > PART_MAX_LISTED_STRIDED)   // fewer lines, more lanes each
        listed = std::max(listed, ccd_plan(dir, n, PART_MAX_LISTED_STRIDED, true).blocks);
    return std::max(ccd_plan(dir, n, lines, false).blocks, hsum_blocks(n, lines) + listed);
}

}  // namespace lsmp
