// nw_sell.h -- the columns that a sliced ELL product reads on slices in
// offset form (Sell in nw_internal.h).  Plain C++ as well as device code, so
// that the rule can be checked without a GPU.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define NW_SELL_HD __host__ __device__
#else
#define NW_SELL_HD
#endif

namespace nw {

// Column of offset `off` for the lane of row `row` in a matrix of n rows.  A
// partial last slice has lanes without a row; they read the last row's
// columns, which lie in [0, n) as every offset of a slice does for each of its
// rows (the slice is not in offset form otherwise).  row + off would not do:
// with one row in the slice its offsets are all <= 0, and the lanes behind it
// would read up to 63 entries past the vector.
NW_SELL_HD inline int dia_column(int row, int off, int n)
{
  return (row < n ? row : n - 1) + off;
}

}  // namespace nw
