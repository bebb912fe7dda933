// Which tiles a product is cut into: plain arithmetic on its sizes, so that a host compiler can take it as well.
#pragma once

#include <algorithm>
#include <cmath>

namespace {

// Lanes whose vector lies past the end of a row are sent OUT_OF_RANGE bytes on, which has to lie past the extent
// of a tile's rows and to leave room for their offset in 31 bits: the rows of a tile span less than that.
constexpr int OUT_OF_RANGE = 0x40000000;

bool tile_rows_in_range(long long rows, long long K) { return rows * K * 2 < OUT_OF_RANGE; }

// Weights that the 256 MB behind L2 cannot hold are read with streaming (nontemporal) loads: they then push nothing out
// of it on their way, which costs 5 to 10 % (us, plain / streaming, operands changing from call to call: 64 groups of 2
// rows, 1024 x 2048, 268 MB 42.8 / 39.2, 2048 x 7168 134.9 / 119.7; 32 groups of 256 rows, 2048 x 4096 133.6 / 125.4,
// of 100 rows 97.0 / 86.2; 32 of 63, 7168 x 7168 574 / 546). Smaller ones may still be there from the call before,
// and streaming loads leave nothing behind: 32 groups, 1024 x 2048, 134 MB read again 20.2 / 25.6, 67 MB 12.4 / 14.4.
// Where a group has several rows of tiles L2 has to keep its weights between them: 32 of 1000, 7168 x 2048 828 / 835.
bool weights_past_the_cache(int groups, int N, int K) { return (double)groups * N * K * 2 >= 256.0 * (1 << 20); }

// How a grouped product is cut: the height of its tiles in bands of 32 rows (10, 8, 6: phased_gemm_kernel, 256
// columns; 4, 2: dense_gemm_kernel, 128 columns), 0 where rows of K are too long for any. `rows_hint` rows over all
// groups are taken to be spread as uniform routing spreads them: a group's number is normal around the average.
//
// A tile costs per step of K what its unit has to fetch, in rows of 128 bytes, about 3 ns each (32 groups of 256 rows,
// 2048 x 4096, tiles of 192 rows: 37 KB a microsecond and unit, 40 without the MFMAs; the MFMAs without the loads take
// 0.5 to 0.7 of the time on every tall tile). A step takes no less than HBM needs for the weights,
// which every round of tiles over the units asks for anew: 256 x 256 columns in the time of 490 rows, two
// workgroups of 128 columns on every unit in that of 530. What else was measured and stands in the factors: two
// workgroups on a unit fetch 1.3 times as slowly as one; tiles of 320 rows, which have room for half a step of weights
// beyond the next one, 1.15 times (30 KB a microsecond, 32 without the MFMAs); the first
// loads and the results of a tile take as long as six steps, of two with two workgroups on a unit, which overlap them.
// Factors and floors are those that lose least, and their neighbours lose hardly more: 697 shapes of 2 to 128 groups,
// 50 to 1024 rows, N and K of 512 to 8192, all five tiles timed on each. The choice is 1.5 % behind the best of them
// and the streaming kernel on average, more than a tenth on 31. (Counting rounds x (height + columns) alone, without
// the tile of 128 x 128, it was 6.4 % behind, and more than a tenth on 155.) Among them, us with 320 / 256 / 192 / 128 /
// 64 rows: 32 groups of 63 rows, 7168 x 7168 640 / 613 / 604 / 576 / 708; 8 of 64, 4096 x 4096 89 / 78 / 76 / 52 / 65;
// 32 of 100, 2048 x 4096 112 / 105 / 104 / 119 / 146; 32 of 256, 4096 x 2048 147 / 176 / 182 / 203 / 240.
struct GroupTiles {
  double each;    // tiles of a group, on average
  double surely;  // as many as nearly every group has
  double height;  // rows of a tall one
};

GroupTiles tiles_of_groups(double rows, int groups, int high) {
  if (rows > 16.0 * high) return {rows / high + 0.5, rows / high, (double)high};
  const double deviation = std::max(1e-3, std::sqrt(rows * (1.0 - 1.0 / groups)));
  GroupTiles t = {1.0, 1.0, 0.0};
  for (int k = 1;; ++k) {
    const double need_more = 0.5 * std::erfc(((double)k * high + 0.5 - rows) / (deviation * std::sqrt(2.0)));
    if (need_more > 0.95) t.surely = k + 1;
    if (need_more < 1e-3) break;
    t.each += need_more;
  }
  t.height = std::min((double)high, (rows + deviation) / t.surely);
  return t;
}

int grouped_tile_bands(long long rows_hint, int groups, int N, int K) {
  constexpr double UNITS = 256, FEW = 0.01;  // (of a round: tiles that only some draws of the rows have)
  const double rows = (double)rows_hint / groups, steps = (K + 63) / 64;
  int best_bands = 0;
  double best = 0;
  for (const int bands : {6, 8, 2, 4, 10}) {  // (where two cost the same the first is faster, by up to 3 and 13 %)
    const int high = bands * 32, wide = bands <= 4 ? 128 : 256;
    if (!tile_rows_in_range(std::max(high, 256), K)) continue;
    const GroupTiles t = tiles_of_groups(rows, groups, high);
    const double one_each = (double)groups * ((N + wide - 1) / wide) / UNITS;
    const double rounds = std::max(t.surely * one_each, t.each * one_each - FEW);
    double cost;
    if (wide == 256) {  // one workgroup per unit
      const double fetch = (t.height + 256) * (bands == 10 ? 1.15 : 1.0), weights = 490 / t.each;
      const double whole = std::floor(rounds), rest = rounds - whole;
      cost = whole * std::max(fetch, weights) + (rest > 0 ? std::max(fetch, rest * weights) : 0);
      cost *= 1 + 6 / steps;
    } else {  // two per unit, and one in the last round if they are odd
      const double each = std::ceil(rounds), pairs = std::floor(each / 2);
      cost = pairs * std::max(1.3 * 2 * (t.height + 128), 530 / t.each) + (each - 2 * pairs) * (t.height + 128);
      cost *= 1 + 2 / steps;
    }
    if (!best_bands || cost < best) {
      best = cost;
      best_bands = bands;
    }
  }
  return best_bands;
}

}  // namespace
