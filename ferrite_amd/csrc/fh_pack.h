// Which of fh_bfp_pack's kernels (fh_core.hip) takes a call.
#pragma once
#include "fh_common.h"

namespace fh {

// Along N, tiles of 64 rows by 16 runs in place of a thread a block: past ~2 MB of values (576 x 1536 takes 4.5 us a thread a
// block, 4.9 in tiles), from 8 rows (a tile's empty rows are idle threads: bf16 into bfp8 of 4M values in 1 row 10.2 us against
// 18.5, of 4 rows by 1M 5.4 against 6.8, 8 rows 10.9 against 9.2, 16 rows by 256K 10.2 against 5.2), and where the grid holds
// them (a grid's threads along x stay below 2^32, its y below 65536)
inline bool pack_in_tiles(int64_t K, int64_t runs) {
  return K >= 8 && K * runs >= 131072 && (runs + 15) / 16 < (1LL << 24) && (K + 63) / 64 <= 65535;
}

}  // namespace fh
