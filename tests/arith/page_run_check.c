/* run_offset(key, row_bytes) = key * row_bytes without wrapping, for the keys and row sizes a prefill call can
   have: keys below 2^31, rows up to 2^31 / 16 bytes (a page of 16 slots below 2^31 bytes). The reference product
   is summed from 16-bit halves in 128 bits. */
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
  long bad = 0, n = 0;
  for (unsigned r = 0; r < sizeof(rows) / sizeof(rows[0]); ++r) {
    const uint64_t wrap = (1ull << 32) / rows[r];   /* the first key 4 GiB away */
    uint64_t keys[80], nk = 0;
    for (int b = 0; b < 31; ++b) {
      keys[nk++] = 1ull << b;
      keys[nk++] = (1ull << b) - 1;
    }
    for (int d = -32; d <= 32; d += 16) keys[nk++] = wrap + d;
    keys[nk++] = 0x7fffffff;
    for (uint64_t i = 0; i < nk; ++i) {
      if (keys[i] > 0x7fffffff) continue;
      ++n;
      bad += run_offset((uint32_t)keys[i], rows[r]) != product((uint32_t)keys[i], rows[r]);
    }
  }
  printf("checked %ld mismatched %ld\n", n, bad);
  return bad != 0;
}
