// bin_rows.h - which bins of a stencil row a list build reads.
#pragma once
#include <math.h>

#ifdef __HIPCC__
#define MDX_HD __host__ __device__ __forceinline__
#else
#define MDX_HD inline
#endif

namespace mdx {

// Bins x0 .. x1 of a row that lie within wb bins of an atom at tx bins, of the
// s bins on either side of its own bin ix.  The own bin is always among them,
// whatever tx is: an atom outside a box that is not periodic is reported by
// the build's flags, which the host reads after the list pass, so its place
// (far outside, infinite or NaN) must not choose bins the row does not have.
MDX_HD void row_bins(int ix, int s, float tx, float wb, int &x0, int &x1) {
  x0 = (int)fmaxf((float)(ix - s), fminf((float)ix, ceilf(tx - 1.0f - wb)));
  x1 = (int)fminf((float)(ix + s), fmaxf((float)ix, floorf(tx + wb)));
}

}  // namespace mdx
