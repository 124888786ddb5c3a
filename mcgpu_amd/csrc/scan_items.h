// How a scan numbers its candidates over the cells around a molecule (host and
// device).
#pragma once

#include "rng31.h"  // MCGPU_HD

namespace mcgpu {

constexpr int kScanEntries = 64;         // entries of a scan's cell table
constexpr int kMaxScanItems = 1 << 20;   // items a lane's division reaches (div_small)

// A scan's items are numbered `width` to an entry of its cell table, so that a
// lane finds its entry by one division; the lanes of free places idle.  A cell
// takes one entry of the largest occupancy while that costs at most two items a
// candidate (1.15 in a liquid) or no more than one pass.  Where the occupancies
// differ more, one full cell would make every other pay for it: the cells are
// then cut into pieces, the smallest that the table's free entries hold, sum /
// (64 - cells), which costs at most cells * (width - 1) free places.  us for the
// full energy of a box with a tenth of its molecules in one small cube, 4,096
// water 62.1 -> 33.4, mixture of 3,000 65.7 -> 41.3 (47.6 and 49.6 by an earlier
// kernel that mapped items by a prefix of the occupancies); of an even mixture
// of 20,000, which takes no pieces, 98.0 -> 98.8.
MCGPU_HD inline int scan_width(int cells, int largest, int sum, int pass) {
  const long long even = (long long)cells * largest;
  if (even <= pass || even <= 2ll * sum || cells >= kScanEntries) return largest;
  const int room = kScanEntries - cells;
  const int width = (sum + room - 1) / room;
  const long long cut = sum + (long long)cells * (width - 1);
  return cut < even && cut <= kMaxScanItems ? width : largest;
}

}  // namespace mcgpu
