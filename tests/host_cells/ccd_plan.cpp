// Host build of the CCD passes' plan (lsmp_ccd_plan.h of the library) for
// tests/test_ccd_plan_host.py.  Test infrastructure only.
#include "../../mass-preserving-level-set-method_amd/csrc/lsmp_ccd_plan.h"

extern "C" {
int hc_ccd_plan(int dir, int n, long nlines, int listed, int esz, long *blocks)
{
    const lsmp::CcdPlan p = lsmp::ccd_plan(dir, n, nlines, listed != 0, (size_t)esz);
    *blocks = p.blocks;
    return p.lanes;
}
int hc_hsum_segments(int n) { return lsmp::hsum_segments(n); }
long hc_hsum_blocks(int n, long nlines) { return lsmp::hsum_blocks(n, nlines); }
long hc_mass_sums(int dim, int nx, int ny, int nz, int esz) { return lsmp::mass_sums(dim, nx, ny, nz, (size_t)esz); }
}
