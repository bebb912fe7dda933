// Which tiles a product is cut into: plain arithmetic on its sizes, so that a host compiler can take it as well.
#pragma once

#include <limits.h>

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
// What counts is what is read: no more groups than there are rows. Where that is three quarters of the cache or more,
// reading it again gains little, and other weights in between cost the most (groups, N x K, rows: the same groups call
// after call, other groups, another matrix in between): 64, 1024 x 2048, 24 rows, 96 MB 20.4 / 25.9, 20.6 / 26.6, 26.5 /
// 26.8; 8 rows 18.1 / 18.3, 18.4 / 23.5, 21.6 / 23.5; 128, 1024 x 4096, 16 rows, 128 MB 33.9 / 43.5, 45.5 / 45.2, 46.0 /
// 45.5; but 64, 1024 x 2048, 48 rows, 192 MB 30.9 / 31.9, 31.2 / 32.1, 36.3 / 32.8; 63 rows 39.1 / 40.7, 39.3 / 40.8, 46.0 /
// 41.7; and against the rule 64, 2048 x 7168, 8 rows, 224 MB 56.6 / 75.3, 77.6 / 76.7, 78.2 / 76.9; 256, 1024 x 1024, 64
// rows, 128 MB 24.3 / 22.2, 24.2 / 24.0, 25.0 / 24.4.
// Where a group has several rows of tiles L2 has to keep its weights between them: 32 of 1000, 7168 x 2048 828 / 835.
bool weights_past_the_cache(int groups, long long rows_hint, int N, int K) {
  constexpr double CACHE = 256.0 * (1 << 20);
  const double group = (double)N * K * 2;
  return groups * group >= CACHE && (double)std::min<long long>(groups, rows_hint) * group >= CACHE * 3 / 4;
}

// How a grouped product is cut: the height of its tiles in bands of 32 rows (10, 8, 6: phased_gemm_kernel, 256
// columns; 4: dense_gemm_kernel, 2: sliced_gemm_kernel, 128 columns; grouped_slices has some of the others too), 0 where rows of K are too long
// for any. `rows_hint` rows over all groups are taken to be spread as uniform routing spreads them: a group's number is normal around the average.
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

// Whether expert_gemm_kernel has so few blocks (32 rows on 64 columns, at most two per unit) that each looks four steps ahead.
// They are counted as uniform routing would have it: the groups that get a row, or half a block on top of whole ones.
bool streams_far_ahead(long long rows_hint, int groups, int N) {
  const double average = (double)rows_hint / groups;
  return groups * std::max(1.0 - std::exp(-average), average / 32 + 0.5) * ((N + 63) / 64) <= 512;
}

// Tiles of a ring of steps (rows x columns), or none, for a grouped product: those of 32 rows are ring_gemm_kernel's, those of 64, which it had when the
// times below were taken, sliced_gemm_kernel's by now (grouped_slices). Groups with a row, and their row tiles, are
// counted as uniform routing would have them, and `of_*` is how many tiles that makes per unit.
//
// As long as every unit has one tile at most a ring is ahead of expert_gemm_kernel, on 32 x 32 up to 40 rows per group, on 32 x 64
// where those are too many, and from 56 rows on of dense_gemm_kernel, on 64 x 64 and then 64 x 128 (of which nearly a unit's worth pays
// from 40 rows on). With more tiles the kernel that streams the weights looks four steps ahead up to two blocks per unit and is as fast
// or faster. Beyond, where it does not, walks of K that are long beside the start of a ring are ahead: of 48 steps with up to three
// tiles per unit (just above that the last round, of two tiles on a unit, is nearly empty), of 24 with five or more, of 32 with just under
// two (few rows in many groups: 36 in 78, 960 x 2496 31.1 / 26.2 on 32 x 64, 12 in 61, 2528 x 2400 30.6 / 25.7), on 32 x 64 up to 24 rows per group
// and on 64 x 64 up to 44: tiles of 32 rows would there read most groups' weights twice, under skewed routing (a group of 300 rows
// in ten tiles) and uniform routing alike. us, the others / 32 x 32 / 32 x 64 / 64 x 64 / 64 x 128 (rows, groups, N x K):
//    1 each in 5 of 41, 576 x 3520  19.8 / 10.5 / 12.3 / 15.0 / 22.2     9, 43, 2240 x 2752          123 / 92.4 / 86.5 / 88.7 / 110
//   22, 7, 768 x 6656               35.8 / 19.6 / 27.1 / 30.8 / 45.5     46, 8, 1024 x 3648          22.7 / 21.0 / 18.0 / 22.3 / 32.1
//   35, 48, 512 x 2432              39.2 / 40.4 / 40.6 / 30.4 / 28.3     52, 9, 2304 x 5568          66.4 / 76.9 / 64.7 / 61.5 / 53.2
//  143, 6, 960 x 2400               27.2 / 28.2 / 22.8 / 17.7 / 27.3     282, 4, 1472 x 4992         46.0 / 72.6 / 58.8 / 42.8 / 37.9
// and where the others stay: 40, 8, 7168 x 7168 (skewed) 144 / - / 182 / 165 / 143; 28, 8, 7168 x 1536 (skewed) 37.9 / - / 47.5 / 40.4 /
// 42.8; 40, 128, 1792 x 7168 587 / - / 719 / 566 / 537; 28, 128, 4096 x 2880 516 / - / 611 / 532 / 542; 4, 8, 7168 x 2048 39.7 / - / 44.1 /
// 45.7 / 46.6; 2, 53, 2240 x 512 23.3 / 35.8 / 29.4; 68, 41, 512 x 640 12.7 / 23.1 / 17.1 / 16.0 / 19.7.
// A ring is filled whatever the walk: with fewer than five steps of K (three on 32 x 32, eight on 64 x 128) that takes longer than the
// others' whole product: 57, 5, 2816 x 8 4.9 / 6.8 on 64 x 128 and 48, 10, 896 x 360 8.2 / 9.8; but 25, 11, 512 x 216 5.5 / 4.9 on 32 x 32.
// Over 12204 products (4 to 128 groups, 0.06 to 400 rows per group, N and K of 512 to 14000, half of them with Zipf's routing, exponent
// 1.2) the choice takes 0.907 of the others' time (geometric mean; the best of all five 0.88) and is more than 5 % behind them on 1.3 %.
enum RingTile { NO_RING = 0, RING_32x32, RING_32x64, RING_64x64, RING_64x128 };

RingTile grouped_ring(long long rows_hint, int groups, int N, int K) {
  constexpr double UNITS = 256;
  if (!tile_rows_in_range(128, K)) return NO_RING;
  const int steps = (K + 63) / 64;
  if (steps < 3) return NO_RING;
  const double rows = (double)rows_hint / groups, hit = 1.0 - std::exp(-rows);
  auto per_unit = [&](int high, int wide) {
    const double of_a_group = rows < 0.7 ? hit : std::max(hit, rows / high + 0.5);
    return of_a_group * groups * ((N + wide - 1) / wide) / UNITS;
  };
  if (rows <= 40 && per_unit(32, 32) <= 1) return RING_32x32;
  if (steps < 5) return NO_RING;
  const double of_32 = per_unit(32, 64), of_64 = per_unit(64, 64), of_128 = per_unit(64, 128);
  const bool one_per_unit = steps >= 8 && of_128 <= 0.9;
  if (rows >= 56) return of_64 <= 1 ? RING_64x64 : one_per_unit ? RING_64x128 : NO_RING;
  if (rows > 40 && of_128 >= 0.6 && one_per_unit) return RING_64x128;
  const bool far_ahead = streams_far_ahead(rows_hint, groups, N);
  // (few rows hit now more groups, now less; where nothing else is under way either, more than a tile per unit is still ahead)
  if (of_32 <= (rows < 2 && far_ahead ? 0.9 : rows < 1 ? 1.5 : 1.0)) return RING_32x64;
  if (far_ahead) return rows > 24 && of_64 >= 0.75 && of_64 <= 0.95 ? RING_64x64 : NO_RING;
  if (rows > 24 && of_64 <= 2) return RING_64x64;
  const double tiles = rows <= 24 ? of_32 : of_64;
  const bool long_walk = (steps >= 24 && tiles >= 5) || (steps >= 48 && (tiles < 3 || tiles >= (rows <= 24 ? 3.5 : 4.0))) ||
                         (steps >= 32 && tiles <= 1.9);
  if (rows > 44 || !long_walk) return NO_RING;
  return rows <= 24 ? RING_32x64 : RING_64x64;
}

// The kernel of a plain product [M, N, K].
//
// Up to 160 tiles of 256 x 256 a product takes, per step of K, what its workgroups wait for (about the same for every
// round of them over the 256 units, and the longer the larger the tile) and what all of them fetch, in rows of 128
// bytes, 0.7 ns for one row on every unit: rounds x `wait` + rows fetched. Small tiles fetch more and wait less. The
// waits are those that lose least over 510 shapes (65 to 1500 rows, N 1024 to 8192, K 256 to 8192, all five timed on
// each): the choice is 0.5 % behind the best of the five on average, by more than a tenth on 5 shapes; on 180 that had no
// part in the fit (to 20000 rows, N from 32 to 36000) 0.4 %, on 2 shapes. By the number of tiles alone (64 x 128 up to
// 256 of them, then 128 x 128) it was 13 % behind, by more than a quarter on 103. Among them, us with SPLIT_32 / SPLIT_64 /
// 64 x 128 / 128 x 128 / PHASED_128:
//   112 x 1920 x 1832   7.3 /  9.4 / 13.8 / 18.9 / 21.0     255 x 1728 x 3968  19.4 / 14.4 / 23.1 / 26.7 / 37.0
//   867 x 1216 x 6104  70.0 / 61.1 / 43.5 / 56.1 / 63.9     547 x 2688 x 5376  61.1 / 44.2 / 31.3 / 35.0 / 49.2
//   825 x 2624 x 1792  40.2 / 35.5 / 18.5 / 15.5 / 19.5     1586 x 2688 x 1536 phased / 128 x 128 21.9 / 24.1
// Up to 64 rows the two that split K are ahead of the others as far as SPLIT_MAX_TILES, and the same comparison picks the
// height: 59 x 512 x 4448 7.9 / 11.2, 59 x 896 x 6728 16.2 / 22.2 (60 shapes of 33 to 64 rows: 1 % behind the better one,
// 64 rows high for all of them 13 %, more than a quarter on 15).
//
// Between 256 tiles of 128 x 128 and 160 of 256 x 256 what counts is how many tiles the fullest unit has. 192 x 128 (192 +
// 128 rows fetched, one workgroup per unit) makes one round of up to 384 tiles of 128 x 128, of which a quarter to a half
// of the units would have two, and 256 x 256 one of those that would be three rounds of 128 x 128. Their waits (680, 1380)
// lose least over 130 shapes of 360 to 8192 rows there (0.14 % behind the best of five on average, more than a tenth
// on none; without these two 6.9 %, on 29; any 640 to 720 and 1300 to 1400 do as well). us with 128 x 128 / PHASED_128 /
// PHASED_192 / PHASED_256:
//   2048 x 2880 x 360    12.7 / 11.3 /  9.9 / 15.2     3532 x 1408 x 3824   69.5 / 67.9 / 46.5 / 73.3
//   1586 x 2688 x 1536   23.4 / 21.7 / 20.1 / 29.2      685 x 7232 x 2800   49.5 / 46.2 / 33.5 / 53.1
//   2048 x 4096 x 1024   21.4 / 19.1 / 29.0 / 23.3     1646 x 5056 x 2800   76.9 / 76.6 / 67.5 / 54.2
//   1024 x 8192 x 2048   36.7 / 32.1 / 49.5 / 39.3     4225 x 2176 x 1896   58.4 / 57.1 / 51.8 / 42.4
// From 160 tiles on 256 x 256 win, whose rate per unit is half as high again as that of 128 x 128: with 256 / 128 rows
// 4096 x 4096 x 512 (256) 22.2 / 27.4; 8192 x 8192 x 3696 (1024) 407 / 622.
enum LinearWay {
  SPLIT_32, SPLIT_64,                  // skinny_gemm_kernel, 32 or 64 rows x 32 columns
  TILES_64x128, TILES_128x128,         // sliced_gemm_kernel (linear_slices), dense_gemm_kernel
  PHASED_128, PHASED_192, PHASED_256,  // phased_gemm_kernel, 128 x 128, 192 x 128 or 256 x 256
  STREAM_WEIGHTS                       // expert_gemm_kernel, as one group
};

// `*least_cost`: what the choice costs by that comparison, where there was one.
LinearWay linear_way(long long M, long long N, long long K, long long* least_cost = nullptr) {
  constexpr long long UNITS = 256, SPLIT_MIN_STEPS = 8;  // (two for each of four waves)
  constexpr long long SPLIT_MAX_TILES = 192;             // of 128 columns, up to 64 rows
  // (sizes of tiles as powers of two: a small product waits for every division here)
  auto tiles = [&](int rows, int columns) { return ((M + (1 << rows) - 1) >> rows) * ((N + (1 << columns) - 1) >> columns); };
  const bool can_split = (K + 63) / 64 >= SPLIT_MIN_STEPS;
  const bool only_split = can_split && M <= 64 && (N + 127) / 128 < SPLIT_MAX_TILES;
  if (!tile_rows_in_range(only_split ? 128 : 256, K)) return STREAM_WEIGHTS;
  if (!only_split && tiles(8, 8) > UNITS * 5 / 8) return PHASED_256;
  auto cost_of = [&](long long n, int rows_fetched, int wait, int more) {
    return ((n + UNITS - 1) / UNITS * wait + more) * UNITS + n * rows_fetched;
  };
  auto cost = [&](int rows, int columns, int wait, int more) {
    return cost_of(tiles(rows, columns), (1 << rows) + (1 << columns), wait, more);
  };
  LinearWay best = PHASED_128;
  long long least = LLONG_MAX;
  auto consider = [&](LinearWay way, long long c) {
    if (c < least) {
      least = c;
      best = way;
    }
  };
  if (can_split) {
    consider(SPLIT_32, cost(5, 5, 120, 0));
    consider(SPLIT_64, cost(6, 5, 190, 0));
  }
  if (!only_split) {
    consider(TILES_64x128, cost(6, 7, 380, 0));
    consider(TILES_128x128, cost(7, 7, 550, 0));
    consider(PHASED_128, cost(7, 7, 380, 280));
    consider(PHASED_192, cost_of((M + 191) / 192 * ((N + 127) >> 7), 192 + 128, 680, 0));
    consider(PHASED_256, cost(8, 8, 1380, 0));
  }
  if (least_cost) *least_cost = least;
  return best;
}

// Whether a plain product goes to a ring of steps instead (ring_gemm_kernel's when the times below were taken, sliced_gemm_kernel's by now). With K
// too short to be split it is ahead on tiles of 32 x 32 as long as every unit has one at most, but for walks that end before the ring is filled: 1 to 7
// steps take 1.11, 1.07, 1.05, 1.01, 0.99, 0.96 and 0.93 of the others' time (284 products). Above, tiles of 64 x 64, which it has under way for longer
// than dense_gemm_kernel and which fetch no more than skinny_gemm_kernel does, fill a gap between those two; a wait of 300 in the comparison
// above finds them (280 to 320 choose the same of 95 shapes), from 12 steps on (shorter ones are as fast elsewhere). us, linear_way's choice / here:
//   137 x 4320 x 5440  47.9 / 25.7     200 x 4096 x 4096  36.9 / 21.4     82 x 6592 x 2816  27.1 / 16.9
//   494 x 2048 x 2176  20.1 / 13.4     128 x 8192 x 2048  21.2 / 14.9    195 x 3008 x 832    7.7 /  7.5
// and on 32 x 32: 15 x 5888 x 448 5.5 / 4.7, 80 x 2176 x 448 5.6 / 4.8, 4 x 7104 x 280 5.0 / 4.4; but 33 x 4608 x 352 5.3 / 5.5.
// Elsewhere the others stay: 255 x 1728 x 3968 14.7 / 21.6, 349 x 4032 x 2752 26.8 / 25.4, 358 x 6976 x 2096 27.7 / 39.0.
RingTile linear_ring(long long M, long long N, long long K) {
  constexpr long long UNITS = 256, WAIT = 300;
  const long long steps = (K + 63) / 64;
  if (steps < 8) return steps >= 5 && (M + 31) / 32 * ((N + 31) / 32) <= UNITS ? RING_32x32 : NO_RING;
  if (steps < 12 || M <= 64) return NO_RING;
  const long long n = (M + 63) / 64 * ((N + 63) / 64);
  long long least = 0;  // (more than a unit's tile each, or one of the largest tiles: not compared)
  if (n > UNITS || linear_way(M, N, K, &least) == STREAM_WEIGHTS) return NO_RING;
  return WAIT * UNITS + n * (64 + 64) < least ? RING_64x64 : NO_RING;
}

// Tiles of sliced_gemm_kernel (rows x columns), or none.
enum SlicedTile { NO_SLICES = 0, SLICES_32x64, SLICES_64x64, SLICES_64x128, SLICES_128x128, SLICES_192x128, SLICES_64x32 };
int sliced_rows(SlicedTile t) { return t == SLICES_32x64 ? 32 : t <= SLICES_64x128 || t == SLICES_64x32 ? 64 : t == SLICES_128x128 ? 128 : 192; }
int sliced_cols(SlicedTile t) { return t == SLICES_64x32 ? 32 : t <= SLICES_64x64 ? 64 : 128; }

// For a grouped product; `ring` and `bands`: what grouped_ring and (from 56 rows per group on, else 0) grouped_tile_bands have chosen. It takes 64 x
// 64 and 64 x 128 over from both: of 500 products (4 to 64 groups, 1 to 3500 rows per group, N and K of 512 to 7168, a third of them with Zipf's
// routing) those of 64 x 128 of a ring take 0.85 and of dense_gemm_kernel 0.67 of the others' time, of 64 x 64 0.94 (2 of 26 more than 3 % behind).
//
// Taller tiles have a workgroup per unit, and a few tiles past a round make a second one. Skewed routing has more of them than uniform routing: by
// Zipf's a group adds 0.6 of a tile to those that its rows fill (the median; nine of ten at most 0.7 of 128 rows, 0.75 of 192). So 128 x 128
// from dense_gemm_kernel and 192 x 128 from 192 x 256 go there where such tiles fit a round, and uniform routing's 0.9 of one. Where 128 x 128 do not,
// 192 x 128 do as well as dense_gemm_kernel while that has one round, and are up to 1.7 times as fast where it begins another. us, the kernel
// before / here, with uniform and with Zipf's routing: 27 groups of 173, 864 x 2536, whose 192 x 128 are 0.79 of a round and 1.18, 47.8 / 37.0, 43.9 /
// 67.3 (they stay); 30 of 152, 736 x 536, 1.4 rounds of 128 x 128, 20.6 / 13.0, 18.2 / 23.0; 8 of 214, 1984 x 6688 with a popularity that falls with
// the root of the rank 106.6 / 73.7; 7 of 166, 2048 x 2576, 0.87 of a round of 128 x 128, on 192 x 128 30.3 / 33.7, 28.7 / 33.4 (128 x 128 it is).
// Of 600 products (2 to 64 groups, 56 to 1500 rows per group, N and K of 512 to 7168, uniform routing's tiles 1.15 rounds at most), each with these three
// kinds of routing, the choice takes 0.920 of the time of the kernels before, 22 of 1800 more than 3 % behind, by 26 % at most (with 0.8 of a round
// for uniform routing as the only line 0.934, 57, 53 %; the fastest of the three tiles 0.865).
// With fewer rows expert_gemm_kernel stays, whose small blocks read weights from HBM as fast: 42 groups of 25, 1280 x 896, on
// 64 x 128 23.6 / 23.4 us, 896 x 1280 28.2 / 30.2, and where those are few 41.9 / 54.7 (20 of 23, 768 x 6464).
SlicedTile grouped_slices(RingTile ring, int bands, long long rows_hint, int groups, int N) {
  constexpr double UNITS = 256;
  if (ring) return ring == RING_64x64 ? SLICES_64x64 : ring == RING_64x128 ? SLICES_64x128 : NO_SLICES;
  if (bands == 2) return SLICES_64x128;
  if (bands != 4 && bands != 6) return NO_SLICES;
  const double columns = (N + 127) / 128;
  auto uniform = [&](int high) { return tiles_of_groups((double)rows_hint / groups, groups, high).each * groups * columns / UNITS; };
  auto skewed = [&](int high, double of_group) { return ((double)rows_hint / high + of_group * groups) * columns / UNITS; };
  if (bands == 6) return uniform(192) <= 0.9 && skewed(192, 0.7) <= 1 ? SLICES_192x128 : NO_SLICES;
  if (uniform(128) <= 0.9 && skewed(128, 0.7) <= 1) return SLICES_128x128;
  const bool second_round = uniform(128) > 0.95 && uniform(192) <= 0.8;
  return second_round || (skewed(128, 1.0) > 1 && uniform(192) <= 0.9 && skewed(192, 0.8) <= 1) ? SLICES_192x128 : NO_SLICES;
}

// For a plain product; `ring` and `way`: what linear_ring and, without one, linear_way have chosen. It takes over all of the ring's tiles, all of 64 x
// 128 (on the smallest tiles of which every unit has one at most, else as they are), and of the products split over K those of 33 to 96 rows that
// give nearly every unit a tile: up to 64 rows, with weights that the L2s hold, of 64 x 32, which read every weight once (walks of eight steps, the
// shortest that are split, of 32 x 64 as above), and of 32 x 64 above, from 14 steps on. Of 300 products (16 to 8192 rows, N 1024 to 8192, K 256 to
// 8192) 98, at 0.86 of the others' time, none behind. us, 37 x 7808 x 448 on 64 x 128 / 64 x 64 / 32 x 64: 5.59 / 4.82 / 4.76; 148 x 3680 x 448 (87,
// 174 and 290 tiles) 5.71 / 4.92 / 5.86; 500 x 2976 x 448 (192, 376, 752) 5.86 / 6.56 / 8.28.
// Up to 64 rows, split over K / 32 x 64, of which two wait for the same weights / 64 x 32, calls with the same weights and with others out of HBM: 64 x
// 7168 x 2304 (31.5 MiB) 9.1 / 8.8 / 8.7, 12.2 / 12.3 / 11.9; 60 x 7616 x 1688 8.3 / 7.2 / 7.1, 12.1 / 12.7 / 12.2; 52 x 7904 x 1592 7.5 / 6.9 / 6.8,
// 11.0 / 11.5 / 10.9; 64 x 8192 x 1024 6.1 / 5.9 / 5.9, 7.8 / 7.7 / 7.5. In a graph: 62 x 6976 x 1960 8.7 / 7.6 / 7.7, 12.9 / 13.4 / 12.7; 33 x 7168 x
// 1432 6.6 / 6.2 / 6.0, 9.5 / 8.7 / 8.2; 63 x 8160 x 568 4.6 / 4.2 / 4.2, 6.3 / 6.1 / 6.0; 33 x 7008 x 512 3.9 / 3.8 / 3.8, 5.0 / 4.8 / 4.7; over 33
// products of 33 to 64 rows 64 x 32 takes 0.91 and 0.93 of the split's time, at worst 0.99 and 1.01. But larger weights out of HBM 64 x 7008 x 3008
// 14.3 / 15.2 / 14.7 in calls.
// Above, in a graph, split / 32 x 64: 88 x 5056 x 2432 10.4 / 8.8, 13.9 / 12.3; 90 x 4480 x 6000 26.0 / 20.7, 32.2 / 30.7; of short walks 70 x 4704 x
// 688 4.38 / 4.56, 5.74 / 5.82, 65 x 5056 x 568 4.12 / 4.18, 5.20 / 5.39; 66 x 5312 x 872 5.15 / 4.99, 6.63 / 6.63. With fewer tiles or more rows
// splitting K stays ahead: 52 x 5824 x 3624 (182 tiles) 0.99 of its time here, 183 x 1120 x 960 (108) 1.24, 295 x 1536 x 8000 (240) 1.12.
// 192 x 128 stay phased_gemm_kernel's: launched one after the other in a graph they are up to 4 % ahead here, in calls of their own 2 to 3 % behind
// (2048 x 2880 x 360 9.98 / 10.16, 1399 x 3904 x 3016 42.6 / 43.8).
SlicedTile linear_slices(RingTile ring, LinearWay way, long long M, long long N, long long K) {
  constexpr long long UNITS = 256;
  auto tiles = [&](int rows, int columns) { return (M + rows - 1) / rows * ((N + columns - 1) / columns); };
  if (ring == RING_64x64) return SLICES_64x64;
  if (ring || way == TILES_64x128) return tiles(32, 64) <= UNITS ? SLICES_32x64 : tiles(64, 64) <= UNITS ? SLICES_64x64 : SLICES_64x128;
  if ((way != SPLIT_32 && way != SPLIT_64) || M <= 32 || M > 96) return NO_SLICES;
  const long long of_round = M <= 64 ? tiles(64, 32) : tiles(32, 64);
  if (of_round < 200 || of_round > UNITS) return NO_SLICES;
  const long long steps = (K + 63) / 64;
  if (M <= 64) return N * K * 2 > 32 << 20 ? NO_SLICES : steps > 8 ? SLICES_64x32 : SLICES_32x64;
  return steps >= 14 ? SLICES_32x64 : NO_SLICES;
}

}  // namespace
