// How the prefill attention (layers.hip) deals its keys. Host code alone,
// without HIP.
#pragma once

#include <algorithm>
#include <stddef.h>
#include <stdint.h>

namespace dnx {

// How the prefill attention deals its keys to workgroups: `splits` runs of
// tps tiles of kt keys each (1: the whole range, no workspace), and whether
// the combine can also write the fp6 panel of the output.
struct PrefillSplit {
  int splits, tps, kt;
  bool panel;
};

inline PrefillSplit prefill_split(int64_t position, int64_t n, int64_t heads, int64_t hd, int64_t window,
                           int gw) {
  // Tiles of `keys` keys that a block of `queries` tokens walks.
  auto tiles_of = [&](int64_t b, int64_t queries, int64_t keys) {
    const int64_t first = b * queries, last = (first + queries < n ? first + queries : n) - 1;
    const int64_t from = window > 0 && position + first - window + 1 > 0
                             ? position + first - window + 1 : 0;
    return (position + last + 1 - from + keys - 1) / keys;
  };
  // Calls with 512 or more blocks of 64 (query, head) pairs, or fewer than 4
  // tiles of 32 keys, keep their keys whole and need no workspace. The panel
  // is offered where those blocks, brought to 512 by splitting runs of at
  // least two such tiles, have at most 64 splits. The line does not follow the
  // tiles below: it is the one by which callers know which calls may allocate
  // and which write a panel.
  const int64_t q64 = 64 / gw, blocks64 = (n + q64 - 1) / q64;
  int64_t longest = 1;
  for (int64_t b = 0; b < blocks64; b++) longest = std::max(longest, tiles_of(b, q64, 32));
  const int64_t units = heads / gw * blocks64;
  int64_t splits32 = 1;
  if (units < 512 && longest >= 4) {
    splits32 = std::min((512 + units - 1) / units, longest / 2);
    const int64_t run = (longest + splits32 - 1) / splits32;
    splits32 = (longest + run - 1) / run;
    if (n * heads * splits32 * (hd + 4) * 4 > (1ll << 30) || splits32 > 4096) splits32 = 1;
  }
  // hd 64: tiles of 64 keys, but of 32 where the longest range is one or three
  // of those, half of whose last tile of 64 would be empty work (16 / 4 heads,
  // tiles of 32 against 64, us: 32 tokens from 0 4.9 against 6.1, 96 from 0
  // 8.1 against 9.2; two tiles of 32, 64 from 0: 6.5 against 6.2).
  const int kt = hd == 128 || longest == 1 || longest == 3 ? 32 : 64;
  const int64_t qb = 64 / gw, by = (n + qb - 1) / qb;   // 16 queries a wave
  int64_t tmax = 1, total = 0;
  for (int64_t b = 0; b < by; b++) {
    const int64_t t = tiles_of(b, qb, kt);
    tmax = std::max(tmax, t);
    total += t;
  }
  total *= heads / gw;
  if (splits32 == 1) return {1, (int)tmax, kt, false};
  // Runs of equal length that make about kTargetWorkgroups of them (two to a
  // CU; 256, 384, 640 .. 1536 were slower or equal at 17 shapes), at most 64
  // to a row (the row combine's lanes) and 1 GiB of partials.
  constexpr int64_t kTargetWorkgroups = 512;
  int64_t tps = (total + kTargetWorkgroups - 1) / kTargetWorkgroups;
  tps = std::max(tps, (tmax + 63) / 64);
  // A split a tile writes partials that cost more than they spread where they
  // are large: two tiles a split above 9 MB (at 18 MB, 89 tokens after 269, 32
  // / 4 heads, hd 128: 20.1 -> 14.6 us; at 12.3 and 16.9 MB 15.5 -> 14.3 and
  // 17.7 -> 15.5; at 8.8 and 5.4 MB 11.8 -> 13.2 and 12.5 -> 13.3).
  if (n * heads * tmax * (hd + 4) * 4 > 9000000) tps = std::max<int64_t>(tps, 2);
  if (tps >= tmax) tps = std::max<int64_t>(1, (tmax + 1) / 2);
  int64_t splits = (tmax + tps - 1) / tps;
  while (splits > 2 && n * heads * splits * (hd + 4) * 4 > (1ll << 30)) {
    tps *= 2;
    splits = (tmax + tps - 1) / tps;
  }
  return {(int)splits, (int)tps, kt, splits32 <= 64 && splits > 1};
}

// What the first call that splits its keys reserves: no later one needs more
// (about 512 workgroups of 64 rows, twice that where half of the longest range
// lies past the early queries' keys, and 512 blocks that are rounded up). The
// partials of a call do not grow with its position (8 tokens of 16 / 8 heads,
// hd 128: 43 splits after 4095 keys, 63 after 2000), so a reserve by size
// would let a call allocate after a longer one had run.
constexpr size_t kPrefillWorkspace = (size_t)1536 * 64 * (128 + 4) * 4;

}  // namespace dnx
