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

// The tile and the splits of K that take least by these figures: small results are split
// so that all CUs take part, which a fold pays for.
static RowsPlan rows_best(const RowsCost* tiles, int n, long M, long N, long K,
                          bool whole) {
  RowsPlan best;
  for (int i = 0; i < n; ++i) {
    const RowsCost& t = tiles[i];
    if (K % (64 * t.wk) || (whole && t.wk > 1)) continue;
    const long wgs = ldiv_up(M, t.bm) * ldiv_up(N, t.bn), all = K / (64 * t.wk);
    for (int s = 1; s <= (whole ? 1 : 16); ++s) {
      if (s > 1 && (wgs * s > 300 || all / s < 6)) break;
      const float us = ldiv_up(wgs * s, 256) * (t.round + ldiv_up(all, s) * t.wk * t.stage) +
                       (s > 1 ? 3.f + s * (M * N) * 1.6e-6f : 0.f);
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
