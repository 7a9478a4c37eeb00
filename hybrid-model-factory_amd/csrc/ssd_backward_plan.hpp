// Host rules of the SSD backward's launches (plain C++, no device code).
#pragma once
#include <stdint.h>

#include <algorithm>

namespace hmx {
namespace ssdb {

// The states launch's cut of the table rows: blocks of `rows` rows, `blocks` of them.
// One block where the heads alone (`units` chains of a direction, head and 64 state rows)
// give a workgroup per CU, else as many as that takes, of no fewer than 8 rows: every
// further block costs the totals launch and a second read of x, dy, B and C.
struct StateBlocks { int rows, blocks; };
inline StateBlocks state_blocks(int nrows, int units, int cus) {
  const int want = std::min((cus + units - 1) / units, std::max(nrows / 8, 1));
  const int rows = std::max((nrows + want - 1) / want, 1);
  return {rows, std::max((nrows + rows - 1) / rows, 1)};
}

// Whether the group kernel takes the call: it shares C B^T and W's products over the heads
// (B and C grouped alike) and forms no y' (which only z needs); it is the faster one at
// every size measured (its comment), from one head per group on.  It addresses a chunk's
// 64 rows with 31-bit byte offsets (token strides of bf16 elements; dx rows of up to 4
// bytes an element) and stores dx in pieces of up to 16 bytes; the other kernel takes any
// stride, and dx at any element.
inline bool takes_group_kernel(int G, int GC, bool z, int64_t x_ts, int64_t dy_ts, int64_t b_ts,
                               int64_t c_ts, int64_t dx_ts, uintptr_t dx) {
  const int64_t lo = std::min({x_ts, dy_ts, b_ts, c_ts}), hi = std::max({x_ts, dy_ts, b_ts, c_ts});
  return G == GC && !z && lo >= 0 && hi < (1 << 24) && dx_ts < (1 << 23) && dx % 16 == 0;
}

}  // namespace ssdb
}  // namespace hmx
