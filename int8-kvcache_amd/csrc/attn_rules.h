// Which attention kernel a call runs, in a file of its own so that it also compiles for the host.
#pragma once
#include <stdint.h>

// verify_kernel (32-row wavefronts that share each K/V tile through LDS) or attn_kernel (16-row tiles), for `rows`
// (token, q head) rows per kv head, `pairs` (request, kv head) pairs and a call that may cut them into pieces
// (split buffers) or runs each whole. One row tile (decode) is attn_kernel's: 96 ragged requests 101 us against 114,
// 1 x 4,096 keys 14.9 against 16.8.
// Up to 32 rows, two row tiles of attn_kernel each stream and transpose every tile themselves, and verify_kernel's
// shared tiles pay where more than 16 pairs are cut (graph, us, attn_kernel and verify_kernel, 28 / 4 heads unless
// said: 64 x 4 tokens at 4,096 keys 85.3 and 63.5, 6 x 4 24.7 and 19.8, 5 x 4 23.2 and 19.1, 32 / 8 heads 3 x 5 at 30,000
// 73.8 and 50.2, 12 x 3 of 14 / 2 heads d64 at 8,192 21.6 and 19.1; at 1,000 keys 5 x 4 14.0 and 15.4).
// Not with fewer, which attn_kernel's pieces spread as well: 4 x 4 at 4,096 18.0 and 17.8, 2 x 5 of 32 / 8 at 30,000 43.1
// and 44.7, 4 x 4 at 1,000 13.8 and 15.2, 1 x 4 at 32,768 40.4 and 47.2, 1 row of 32 / 1 heads there 35.8 and 44.7.
// Not whole, where nothing waits for a merge and attn_kernel's key splits keep more tiles in flight: 64 x 4 at 4,096
// 72.8 and 76.1, 128 x 4 at 2,048 76.3 and 80.7, 256 decode rows of 32 / 1 heads at 4,096 73.4 and 79.1, 128 x 3 of 14 / 2
// heads d64 47.6 and 58.3; 64 x 4 at 16,384 270 and 271.
static inline int verify_rows(int64_t rows, int64_t pairs, int cut) {
  return rows > 32 || (rows > 16 && cut && pairs > 16);
}

// Shortest piece attn_kernel splits across a workgroup's key splits, in tiles (shorter ones go whole to one key split
// in turn: no barrier, no merge). Pieces of cut segments: 4 (graph, us, from 8 tiles on and from 4 on, 28 / 4 heads unless
// said, the shortest worker share lowered with it: 1 x 1,000 keys 12.6 and 11.6, 4 x 500 13.7 and 11.7, 8 x 2k 17.0 and
// 15.9, 16 x 100 12.7 and 11.8, 4 x 14k 27.2 and 26.0, c4's 96 ragged rows 99.2 and 98.7; 2 and 6 tiles time between the
// two). Segments run whole: 4 per key split, the key splits having other segments to take in the meantime (16 tiles
// at 2 key splits: 2 x 4 tokens of 14 / 2 heads d64 at up to 1,128 keys 11.5 -> 13.4, 69 x 4 at up to 463 13.0 -> 14.5).
static inline int coop_tiles(int cut, int ksplit) { return cut ? 4 : 4 * ksplit; }
