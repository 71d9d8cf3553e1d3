// Which form of a prompt's attention kernel (fh_prefill.hip) takes a call.
#pragma once
#include "fh_common.h"

namespace fh {

constexpr int PA_BK = 64;  // keys a tile

// The keys split among a workgroup's waves: where its tiles of 32 rows are still one round of a workgroup a CU (past it,
// 32 heads of 128: 300 rows 13 -> 18 us, 512 19 -> 24) and there are enough key tiles that the longest wave's share takes less
// than all of them by the whole workgroup, which loads and converts a tile with four times the lanes. One rule for every
// cache format, so that a block float's results are bit for bit its values' in bf16: from 6 tiles of 128 (two tiles gain bf16
// 5% and lose a block float 21%, 10.1 -> 12.9 us; five, two for one wave, 10% and 12%, 16.4 -> 19.6; from six on bf16
// gains 13% and more, 64 rows after 1900 51 -> 30, and a block float 2 to 34%, 64 rows after 4000 in bfp8 140 -> 97, but for 320
// rows of four heads or fewer over exactly 6 or 9 tiles, which lose up to 8%, 18.7 -> 20.3) and 3 of 64 (two 7.9 -> 8.5 in bfp8; three 9.4
// -> 8.9, in bf16 7.7 -> 6.9).
inline bool prefill_splits_keys(int T, int heads, int head_dim, int64_t p0, int cus) {
  if ((int64_t)((T + 31) / 32) * heads > cus) return false;
  const int64_t tiles = (p0 + T - 1) / PA_BK + 1;
  return tiles >= (head_dim < 128 ? 3 : 6);
}

}  // namespace fh
