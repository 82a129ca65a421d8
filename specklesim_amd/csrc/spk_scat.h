// How the scattered field splits its sources (k_scattered): host code, also
// built by the CPU test.
#pragma once
#include <algorithm>
#include <cstdint>

// Sources per chunk for ns sources and npts points; *nch: the chunks.  Enough
// chunks for three waves on every SIMD (3072 workgroups of one wave), as long
// as their sums fit the workspace of `partials` points.  A chunk is whole
// groups of 64 sources, which a wave's lanes form together.  Where those are
// fewer than 512 workgroups in all, a call waits for a wave's walk through its
// group (0.35 us a source): there groups of 16, below 128 workgroups of 8.
// us a call with groups of 8, 16, 64 at (edges, points): (176, 1) 52, 53, 69;
// (176, 181) 54, 56, 71; (736, 1) 55, 56, 70; (736, 181) 66, 61, 72; (2640, 1)
// 68, 62, 72; (2640, 181) 78, 79, 76; (6256, 1) 80, 80, 76.
inline int64_t scat_chunk(int64_t ns, int64_t npts, int64_t partials, int64_t *nch) {
  const int64_t tiles = (npts + 63) / 64;
  const int64_t groups = (ns + 63) / 64 * tiles;
  const int64_t g = groups < 128 ? 8 : groups < 512 ? 16 : 64;
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(3072 / tiles, partials / npts));
  const int64_t per = ((ns + most - 1) / most + g - 1) / g * g;
  *nch = (ns + per - 1) / per;
  return per;
}
