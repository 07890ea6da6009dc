/* verify_rows and coop_tiles over the sizes a call can have: one line per mismatch with the rules as the kernels were
   measured. */
#include <stdio.h>

#include "../../int8-kvcache_amd/csrc/attn_rules.h"

int main(void) {
  long bad = 0, n = 0;
  for (int64_t rows = 1; rows <= 80; ++rows)
    for (int64_t pairs = 1; pairs <= 512; ++pairs)
      for (int cut = 0; cut < 2; ++cut, ++n) {
        int want = rows > 32 || (rows > 16 && cut && pairs > 16);
        if (verify_rows(rows, pairs, cut) != want && ++bad < 5)
          printf("rows %ld pairs %ld cut %d: %d\n", (long)rows, (long)pairs, cut, !want);
      }
  for (int ksplit = 1; ksplit <= 4; ++ksplit)
    for (int cut = 0; cut < 2; ++cut, ++n) {
      int want = cut ? 4 : 4 * ksplit;
      if (coop_tiles(cut, ksplit) != want && ++bad < 5) printf("ksplit %d cut %d: %d\n", ksplit, cut, coop_tiles(cut, ksplit));
    }
  printf("checked %ld mismatched %ld\n", n, bad);
  return bad != 0;
}
