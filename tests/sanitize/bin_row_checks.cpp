// The bins that a list build's row reads, for atoms inside the row (the plain
// expression) and outside it (never a bin that the row does not have).
#include <cstdio>
#include <initializer_list>
#include <limits>

#include "bin_rows.h"

int main() {
  const int s = 2;
  const float inf = std::numeric_limits<float>::infinity(), nan = std::numeric_limits<float>::quiet_NaN();
  long bad = 0;
  for (int n : {1, 2, 4, 5, 37, 1024})
    for (float wb : {0.0f, 1e-3f, 0.7f, 1.9f, 2.001f}) {
      for (float far : {0.0f, 0.5f, 1.0f, 17.25f, 1e6f, 1e9f, 3e9f, 1e30f, inf, nan})
        for (float tx : {-far, n + far}) {
          const int ix = tx > 0.0f && tx < n ? (int)tx : tx > 0.0f ? n - 1 : 0;
          int x0, x1;
          mdx::row_bins(ix, s, tx, wb, x0, x1);
          if (!(ix - s <= x0 && x0 <= ix && ix <= x1 && x1 <= ix + s)) {
            std::printf("%d bins, place %g, reach %g: bins %d to %d\n", n, tx, wb, x0, x1);
            bad++;
          }
        }
      for (int k = 0; k <= 64 * n; k++) {  // inside, the upper face included
        const float tx = k / 64.0f;
        const int ix = k == 64 * n ? n - 1 : k / 64;
        int x0, x1;
        mdx::row_bins(ix, s, tx, wb, x0, x1);
        const int lo = (int)ceilf(tx - 1.0f - wb), hi = (int)floorf(tx + wb);
        if (x0 != (lo > ix - s ? lo : ix - s) || x1 != (hi < ix + s ? hi : ix + s)) bad++;
      }
    }
  std::printf("%ld bad rows\n", bad);
  return bad ? 1 : 0;
}
