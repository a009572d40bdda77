// Which tile of gemm_rows.hip takes a product, and its launch.
#pragma once

#include <cmath>

#include "gemm_rows.hip"

// What a round of a tile's workgroups costs beside its stages and what a stage of 64 of K
// costs, us; a round is 256 workgroups.
struct RowsCost {
  int bm, bn, wk;
  float round, stage;
};

struct RowsPlan {
  int tile = -1, splits = 1;
  float us = INFINITY;
};

// Whether splits of `per` of K columns begin in the same channels of memory: rows of W
// and their splits are multiples of 4 KiB apart, so that all workgroups read from few
// channels at a time. It counts where W from memory is what bounds a product. us, splits
// of that kind and others: 8192 x 8192, 33 rows 38.6 with 4, 32.0 with 3; 16384 x 4096, 64
// rows 38.9 with 2, 34.1 with 4; 8192 x 28672, 17 rows 106 with 2, 85 with 4; 3072 x 24576,
// 16 rows 38.2 with 4, 33.5 with 5. Where K is no multiple of 4 KiB there is no such
// difference (4032 x 16320, 34 rows: 5% the other way), nor beyond 128 rows.
static bool same_channels(long K, long per) { return K % 2048 == 0 && per % 2048 == 0; }

// The tile and the splits of K that take least by these figures: small results are split
// so that all CUs take part, which a fold pays for. whole: no splits; turned: sums run
// over rows of W, whose splits are apart by whole rows.
static RowsPlan rows_best(const RowsCost* tiles, int n, long M, long N, long K,
                          bool whole, bool turned = false) {
  RowsPlan best;
  for (int i = 0; i < n; ++i) {
    const RowsCost& t = tiles[i];
    if (K % (64 * t.wk) || (whole && t.wk > 1)) continue;
    const long wgs = ldiv_up(M, t.bm) * ldiv_up(N, t.bn), all = K / (64 * t.wk);
    for (int s = 1; s <= (whole ? 1 : 16); ++s) {
      if (s > 1 && (wgs * s > 300 || all / s < 6)) break;
      float us = ldiv_up(wgs * s, 256) * (t.round + ldiv_up(all, s) * t.wk * t.stage) +
                 (s > 1 ? 3.f + s * (M * N) * 1.6e-6f : 0.f);
      if (s > 1 && M <= 128 && !turned && same_channels(K, ldiv_up(all, s) * t.wk * 64))
        us *= 1.3f;
      if (us < best.us) best = {i, s, us};
    }
  }
  best.us += (N + M) * K / 9.8e6f;   // memory, a quarter of it not hidden
  return best;
}

template <typename K, typename... Args>
static void rows_launch(K kernel, long grid, int threads, int lds, hipStream_t stream,
                        const Args&... a) {
  HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  kernel<<<grid, threads, lds, stream>>>(a...);
  HIP_OK(hipGetLastError());
}
