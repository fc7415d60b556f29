// lsmp_ccd_plan.h -- which CCD solve a pass over the lines of a direction takes
// and how many block sums it leaves.  The launcher, the size of the block sums'
// buffer and the check before a mass correction's launches all ask here.  Plain C++:
// the host tests build it too.
#pragma once
#include <algorithm>
#include <cstddef>

namespace lsmp {

constexpr int KCC = 17;   // CCD rows per lane at most (9 up to 284 cells, 17 up to 540 with 32 lanes per line, 1084 with 64)

// Lines of a direction, all of them solved, that go through the partitioned solve
// (32 or 64 lanes a line) at most.  It costs about as much for 4 cells as for 250,
// one lane a line (k_ccd_seg) a latency per cell until the chip is full, so the
// count grows with the length.  us of a solve of n cells x lines, 32 lanes against 1:
//   y, z FP64  24x5,184 12.3, 15.8; 24x16,384 22.8, 16.2; 64x16,384 26.0, 32.9;
//              64x40,000 53.7, 35.3; 100x19,881 44.2, 48.0; 100x29,929 63.3, 49.5;
//              160x29,929 64.1, 74.2; 160x40,000 83.0, 75.5; 256x40,000 88.9, 115
//   y, z FP32  32x16,384 17.3, 18.1; 64x40,000 36.1, 31.3; 128x40,000 47.4, 54.8
//   x FP64     24x5,184 11.7, 17.8; 24x16,384 21.9, 19.3; 80x40,000 55.8, 60.6;
//              80x160,000 189, 176; 128x160,000 217, 279; 128x810,000 1112, 1347
//   x FP32     24x16,384 15.2, 20.5; 32x40,000 30.1, 26.3; 48x810,000 426, 432
// Beyond 40,960 y or z lines 32 lanes on a line, each row another cache line, lose
// at any length (256x65,536 was measured).
//
// With 8 or 16 rows a lane (221-252, 477-508 and, of 64 lanes, 957-1,020 cells) the
// lanes of a line read the table from the same LDS banks: 240x19,881 115 against 105 us,
// 480x19,881 364 against 202 (x lines 368, 301), 1,000x10,000 566 against 859 and
// x19,600 1089 against 899.  Other lines of more than 540 cells (64 lanes) break even
// near 14,000 lines (700x19,600 677 against 584), except along x with the table in LDS
// (FP32, and FP64 to 624 cells): 700x40,000 FP32 185 against 380, 560x160,000 984
// against 1339.
constexpr int PART_MAX_CCD = 4096;   // up to these, 32 or 64 lanes always
constexpr int PART_MAX_CCD_STRIDED = 40960, PART_MAX_CCD_LONG = 13000;
constexpr long PART_CCD_ANY = 1L << 31;
inline long part_max_ccd(int dir, int n, size_t esz)
{
    const int lanes = n + 4 <= 32 * KCC ? 32 : 64, rows = (n + 4 + lanes - 1) / lanes;
    long m;
    if (rows % 8 == 0) m = rows % 16 == 0 ? 10000 : 16000;
    else if (lanes == 64) m = dir == 0 && 13 * (n + 6) * esz <= 65536 ? PART_CCD_ANY : PART_MAX_CCD_LONG;
    else if (dir == 0) m = n >= (esz == 4 ? 48 : 125) ? PART_CCD_ANY : 340L * n;
    else m = std::min<long>(PART_MAX_CCD_STRIDED, (esz == 4 ? 340L : 220L) * n);
    return std::max<long>(m, PART_MAX_CCD);
}

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
inline CcdPlan ccd_plan(int dir, int n, long nlines, bool listed, size_t esz)
{
    const long part_max = !listed ? part_max_ccd(dir, n, esz) : dir == 0 ? PART_MAX_LISTED_X : PART_MAX_LISTED_STRIDED;
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
inline long mass_sums(int dim, int nx, int ny, int nz, size_t esz)
{
    const int dir = dim == 3 ? 2 : 1, n = dim == 3 ? nz : ny;
    const long lines = dim == 3 ? (long)nx * ny : nx;
    long listed = ccd_plan(dir, n, lines, true, esz).blocks;
    if (lines > PART_MAX_LISTED_STRIDED)   // fewer lines, more lanes each
        listed = std::max(listed, ccd_plan(dir, n, PART_MAX_LISTED_STRIDED, true, esz).blocks);
    return std::max(ccd_plan(dir, n, lines, false, esz).blocks, hsum_blocks(n, lines) + listed);
}

}  // namespace lsmp
