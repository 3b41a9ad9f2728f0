// Host side of the k-split contractions' tile choice, shared by
// l2c_qgemm_ksplit.hip and l2c_scgemm_ksplit.hip.
#pragma once

#include <algorithm>

#include "l2c_common.h"

namespace l2c {

// One tile: 16 mf batch rows x 16 nf weight rows by `waves` waves, `lds` bytes of
// LDS a workgroup.
struct KsplitTile {
  int mf, nf, waves, lds;
};

inline long long ksplit_tiles(const KsplitTile &t, int batch, int rows) {
  return static_cast<long long>((batch + 16 * t.mf - 1) / (16 * t.mf)) * ((rows + 16 * t.nf - 1) / (16 * t.nf));
}

inline bool ksplit_launchable(const KsplitTile &t, int batch, int rows) {
  return launchable(ksplit_tiles(t, batch, rows), 64 * t.waves);
}

// What the busiest CU does, in bytes staged: its tiles' X and W rows (x_bytes
// and w_bytes a k), eight times the waves' partial sums that meet in LDS, and
// 10000 for every k-step (`step` k) of a wave's chain, once for each group of
// workgroups that fit the CU together. The first term rules at long K, the
// other two at short K, where small tiles on two waves, several of them on a CU,
// are up to 1.8 times faster than large ones. Fitted to the GPU times of 27
// tiles on 56 shapes of 1 to 1024 x 256 to 16384 x 288 to 11008 in six formats:
// the choice among twelve tiles is 3 to 6% slower than the best of the 27 in
// the mean.
inline double ksplit_cost(const KsplitTile &t, double x_bytes, double w_bytes, int step, int batch, int cols,
                          int rows) {
  const double bm = 16.0 * t.mf, bn = 16.0 * t.nf;
  const long long per_cu = (ksplit_tiles(t, batch, rows) + 255) / 256;
  const long long together =
      std::max(1LL, std::min(per_cu, static_cast<long long>(std::min(160 * 1024 / t.lds, 2048 / (64 * t.waves)))));
  const int chain = (cols / step + t.waves - 1) / t.waves;
  return static_cast<double>(per_cu) * (cols * (x_bytes * bm + w_bytes * bn) + 8.0 * bm * bn * t.waves) +
         1e4 * static_cast<double>((per_cu + together - 1) / together) * chain;
}

}  // namespace l2c
