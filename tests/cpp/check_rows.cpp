// Checks spark_rows.hpp: row_pad over box widths and guard depths (the first
// interior cell of every row starts a line or half line of 128 bytes, rows
// hold their cells, at most a third more memory), and pad_rows: a padded
// state fits into the memory that is free, also for widths whose padding is
// small, and takes at most 3/32 of it from the batches after it; div_pool
// likewise.  Prints "ok <cases>" or the first mismatch.
#include <cstdio>

#include "spark_rows.hpp"

int main() {
  long cases = 0;
  for (int ng = 0; ng <= 16; ng++)
    for (int nx = 1; nx <= 300; nx++) {
      const int NX = nx + 2 * ng;
      const spark::RowPad p = spark::row_pad(NX, ng);
      const int a = p.pitch % 16 == 0 ? 16 : 8;
      if (p.pitch < NX || p.lead < 0 || 3 * p.pitch > 4 * NX ||
          (p.pitch != NX && (p.pitch % a || (p.lead + ng) % a || p.lead >= a))) {
        std::printf("width %d guards %d: pitch %d lead %d\n", nx, ng, p.pitch, p.lead);
        return 1;
      }
      // a batch of these rows in ever less free memory: from where padding
      // fits easily to where the packed state just fits
      const int64_t rows = 1000000, fields = 58;
      const int64_t packed = rows * NX * fields * 8, padded = rows * p.pitch * fields * 8;
      for (int64_t free = 4 * packed; free >= packed; free -= packed / 16) {
        const bool pad = spark::pad_rows(rows * p.pitch, fields, free);
        if (pad && (padded > free || 32 * (padded - packed) > 3 * free)) {
          std::printf("width %d guards %d: %lld padded, %lld packed, %lld free\n", nx, ng, (long long)padded,
                      (long long)packed, (long long)free);
          return 1;
        }
        if (!pad && free == 4 * packed) {
          std::printf("width %d guards %d: not padded in four times its memory\n", nx, ng);
          return 1;
        }
        const int64_t left = free - (pad ? padded : packed), pool = rows * (pad ? p.pitch : NX) * 13;
        if (spark::div_pool(pool, left) && pool * 8 > left / 4) {
          std::printf("width %d guards %d: a pool of %lld doubles in %lld bytes\n", nx, ng, (long long)pool, (long long)left);
          return 1;
        }
        cases++;
      }
    }
  std::printf("ok %ld\n", cases);
  return 0;
}
