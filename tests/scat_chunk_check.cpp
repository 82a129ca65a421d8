// scat_chunk over the sizes that the scattered field meets
#include <cstdio>

#include "spk_scat.h"

int main() {
  const int64_t edges[] = {1, 5, 40, 176, 408, 736, 1680, 2640, 4720, 6256, 29800, 123840};
  const int64_t points[] = {1, 2, 7, 63, 64, 65, 181, 900, 1000, 4096, 20000, 131072, 131073, 1000000};
  const int64_t partials = 1 << 17;
  int bad = 0;
  for (int64_t n : edges)
    for (int64_t p : points) {
      const int64_t ns = 6 * n, tiles = (p + 63) / 64;
      int64_t nch = 0;
      const int64_t per = scat_chunk(ns, p, partials, &nch);
      const int64_t groups = (ns + 63) / 64 * tiles;
      // every source in one chunk, none empty, the sums in the workspace
      bool ok = nch >= 1 && per >= 1 && nch * per >= ns && (nch - 1) * per < ns;
      ok = ok && (nch == 1 || nch * p <= partials) && nch * tiles <= std::max<int64_t>(3072, tiles);
      // a wave does not walk through more sources than it has to wait for: 16 of
      // them where groups of 64 leave most of the chip idle
      if (groups < 512 && partials / p * 16 >= ns && 3072 / tiles * 16 >= ns) ok = ok && per <= 16;
      if (groups < 128) ok = ok && per <= 8;
      if (!ok) {
        std::printf("edges %lld points %lld: per %lld chunks %lld\n", (long long)n, (long long)p,
                    (long long)per, (long long)nch);
        ++bad;
      }
    }
  std::printf("bad %d\n", bad);
  return bad != 0;
}
