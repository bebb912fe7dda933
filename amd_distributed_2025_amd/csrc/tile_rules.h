// Which tiles a product is cut into: plain arithmetic on its sizes, so that a host compiler can take it as well.
#pragma once

#include <algorithm>
#include <cmath>

namespace {

// Lanes whose vector lies past the end of a row are sent OUT_OF_RANGE bytes on, which has to lie past the extent
// of a tile's rows and to leave room for their offset in 31 bits: the rows of a tile span less than that.
constexpr int OUT_OF_RANGE = 0x40000000;

bool tile_rows_in_range(long long rows, long long K) { return rows * K * 2 < OUT_OF_RANGE; }

// How a grouped product with `rows` rows in an average group is cut: the height of its tiles in bands of 32
// rows (10, 8, 6: phased_gemm_kernel, 256 columns; 2: dense_gemm_kernel, 64 x 128), 0 where rows of K are too long
// for any. A tile costs what a compute
// unit has to fetch for it, (rows + columns) x 128 bytes per step of K: that, and not the matrix cores, bounds
// these kernels (measured on 32 groups of 256 rows, 137 GFLOP: 163 us, 145 without the MFMAs, 119 without the
// loads; a unit fetches about 49 KB a microsecond). Tiles run in rounds over the units. A group is taken to have
// one standard deviation of uniform routing more rows than the average: it decides how many tiles most groups
// need. 320 rows leave room for two buffers of each operand only and get 15 % on top.
// Measured, us (rows: 320, 256, 192, 64 x 128): 32 groups x 256 rows, N 2048, K 4096: 156 188 171 -; N 4096, K
// 2048: 164 173 183 -; 512 rows: 266 276 259 -; 128 rows: 133 111 108 -; 16 x 1024 rows, N 4096, K 2048: 261 254
// 260 -; 8 x 200, N 7168, K 2048: 73 62 88 -; 16 x 150, 2880 x 2880: 87 73 71 136; 8 x 64, N 2048, K 7168: 168 117
// 112 75; 4 x 300, N 2048, K 4096: 97 64 58 43; 4 x 1000, N 512, K 7168: 169 119 104 70.
int grouped_tile_bands(long long rows, int groups, int N, int K) {
  constexpr long long UNITS = 256;
  const long long most = std::max<long long>(1, rows + (long long)std::sqrt((double)rows));
  int best_bands = 0;
  double best = 0;
  for (const int bands : {8, 6, 10, 2}) {
    const long long high = bands * 32, wide = bands == 2 ? 128 : 256, n = (most + high - 1) / high;
    if (!tile_rows_in_range(std::max<long long>(high, 256), K)) continue;
    const long long height = std::min(high, ((most + n - 1) / n + 31) / 32 * 32);
    const long long rounds = (n * groups * ((N + wide - 1) / wide) + UNITS - 1) / UNITS;
    const double cost = (double)rounds * (height + wide) * (bands == 10 ? 1.15 : 1.0);
    if (!best_bands || cost < best) {
      best = cost;
      best_bands = bands;
    }
  }
  return best_bands;
}

}  // namespace
