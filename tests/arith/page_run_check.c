/* run_fits(pages, page_bytes): where it holds, the 32-bit product key * row_bytes is the offset of every key of the
   run; where it does not, the last keys' is not. Pages of 16 to 4,096 slots, rows up to 2^31 / 16 bytes; keys at the
   run's ends and around every power of two. The reference product is summed from 16-bit halves in 128 bits. */
#include <stdio.h>

#include "../../int8-kvcache_amd/csrc/page_run.h"

static unsigned __int128 product(uint32_t a, uint32_t b) {
  unsigned __int128 s = 0;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j)
      s += (unsigned __int128)((a >> 16 * i) & 0xffff) * ((b >> 16 * j) & 0xffff) << 16 * (i + j);
  return s;
}

int main(void) {
  const uint32_t rows[] = {64, 128, 256, 1024, 4096, 8192, 16384, 65536, 1u << 20, (1u << 27) - 16, 1u << 27};
  long bad = 0, n = 0, fits = 0;
  for (unsigned r = 0; r < sizeof(rows) / sizeof(rows[0]); ++r)
    for (uint64_t bs = 16; bs <= 4096; bs *= 4) {
      const uint64_t page = bs * rows[r];
      if (page > 0xffffffffull) continue;
      const uint64_t edge = (1ull << 32) / page;      /* pages that end within 4 GiB */
      for (int64_t d = -2; d <= 3; ++d) {
        const int64_t pages = (int64_t)edge + d;
        if (pages < 1 || (uint64_t)pages * bs > 0x80000000ull) continue;
        const uint32_t last = (uint32_t)(pages * bs - 1);
        if (!run_fits((uint32_t)pages, (uint32_t)page)) {
          ++n;
          bad += product(last, rows[r]) + rows[r] <= (unsigned __int128)1 << 32;   /* refused needlessly */
          continue;
        }
        ++fits;
        for (int b = 0; b <= 31; ++b)
          for (int64_t e = -1; e <= 1; ++e) {
            int64_t key = (int64_t)(1ull << b) + e;
            if (b == 31) key = (int64_t)last + e - 1;
            if (key < 0 || key > last) continue;
            ++n;
            bad += (uint32_t)key * rows[r] != product((uint32_t)key, rows[r]);
          }
      }
    }
  printf("checked %ld, %ld runs fit, mismatched %ld\n", n, fits, bad);
  return bad != 0 || fits < 50;
}
