// Which decodes of the FP8 wire write their outputs with non-temporal stores (plain C++, host only).
#pragma once

#include <stdint.h>

namespace xgen {

// bytes: read and written by the call; cache: the last-level cache's; row_bytes: of one output row;
// lanes: per row, 16 bytes each; address_bits: the output bases and, strided, the destination strides
// in bytes, OR-ed together.
//
// Three conditions, each measured (bf16, 3 streams, 8 peers, 3 heads; us with ordinary -> non-temporal
// stores):
//  * The call passes the cache.  Below, what reads the outputs next would have found them there.
//  * Every store instruction writes whole 64-byte pieces of a row.  Non-temporal stores of less are not
//    merged on the way to memory: 270 MB of rows of 16, 40, 72 or 136 values 65 -> 80 to 134, rows of 128
//    values 16 bytes off 119 -> 242.
//  * Past 1.5 caches, contiguous outputs in whole 128-byte lines only.  The sum that counts is encode,
//    the exchange (a copy of the wire), decode and one read of the outputs: up to there it is 2% to 7%
//    lower (rows of 128 at 350 MB: 229 -> 222 contiguous, 233 -> 224 gathered), from there it is higher
//    for rows written in other pieces (420 MB: gathered 281 -> 296; 400 MB, rows of 64 contiguous
//    295 -> 313) and even for whole lines (420 / 512 / 900 MB: 280 -> 284, 338 -> 334, 598 -> 587), where
//    the decode itself (82 -> 69, 99 -> 85, 176 -> 179) and each shorter part of that sum are lower.
//    (Decode and read alone, of a wire that lay in the cache without an exchange, lose up to 1.5 caches:
//    gathered rows of 128 at 300 MB 95 -> 109.)
inline bool decode_stores_non_temporal(int64_t bytes, int64_t cache, int64_t row_bytes, int lanes, bool strided,
                                       uint64_t address_bits) {
  const uint64_t bits = address_bits | (uint64_t)row_bytes;
  if (bytes <= cache || lanes * 16 < 64 || bits % 64) return false;
  const bool whole_lines = !strided && lanes * 16 >= 128 && bits % 128 == 0;
  return whole_lines || bytes <= cache + cache / 2;
}

}  // namespace xgen
