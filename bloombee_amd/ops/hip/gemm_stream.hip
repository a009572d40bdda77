// Products of a few rows with a weight matrix, C(M,N) = A(M,K) @ W(N,K)^T, M <= 32, in
// one launch with what follows them in a decoder layer:
//   EPI_SUM     [+ bias] [+ residual]
//   EPI_SWIGLU  silu(gate) * up of a fused [gate | up] projection
//   EPI_ROPE    rotations and paged K/V of a fused [q | k | v] projection
// and with the RMS norm of the rows ahead of them (its weight folded into W).
//
// The weights are streamed once and bound it. A workgroup owns 16 rows of W (two sets
// of 16 where the epilogue pairs columns) over all of K: its eight waves take every
// eighth piece of 128 columns and add up in LDS, so that no partial sums go through
// memory and nothing has to be folded by another launch. In a decode step a launch
// costs about 5 us whatever it does (code, arguments and first loads miss caches that
// the weights swept), which is why the layer's small steps ride here.
// Every wave keeps DP pieces of W in flight in registers; rows of A come from L2 in
// fragments, W being the wider of the two streams.
// A row's sum of squares for the norm is the diagonal of A A^T, made by the matrix
// cores from the fragments at hand.

#pragma once
#include "common.h"

enum { EPI_SUM, EPI_SWIGLU, EPI_ROPE };

struct StreamArgs {
  const unsigned short* A;     // (M, K)
  const unsigned short* W;     // (N, K)
  const unsigned short* R;     // EPI_SUM: (M, N) residual or null
  const unsigned short* bias;  // EPI_SUM: (N,) or null
  unsigned short* C;           // EPI_SUM, EPI_ROPE: (M, N), EPI_SWIGLU: (M, N / 2)
  int M, N, K;
  float eps;                   // of the norm
  // EPI_ROPE: row m is token m % T of sequence m / T
  const float* cos_t;          // (max_pos, D / 2)
  const float* sin_t;
  const int* pos;              // (M,) or null: start + token
  const int* start;            // (M / T,)
  const int* table;            // (M / T, maxp)
  unsigned short* k_pages;     // (np, Hkv, P, D)
  unsigned short* v_pages;     // (np, Hkv, D, P)
  int T, Hq, Hkv, D, P, maxp, max_pos;
};

// Columns d and d + D / 2 of head h of a fused [q | k | v] projection, row m: q turned
// to its place in C, k turned and v as it is to their page slots.
DEVINL void rope_kv_store(const StreamArgs& a, int h, int d, int m, float v, float u) {
  const int b = m / a.T, at = a.start[b] + m % a.T;
  const int slot = at % a.P;
  const long page = h < a.Hq ? 0 : a.table[b * a.maxp + at / a.P];
  if (h >= a.Hq + a.Hkv) {
    unsigned short* vp =
        a.v_pages + ((page * a.Hkv + h - a.Hq - a.Hkv) * a.D + d) * a.P + slot;
    vp[0] = f2bf(v);
    vp[(long)(a.D / 2) * a.P] = f2bf(u);
    return;
  }
  const int p = min(max(a.pos ? a.pos[m] : at, 0), a.max_pos - 1);
  const float cs = a.cos_t[(long)p * (a.D / 2) + d];
  const float sn = a.sin_t[(long)p * (a.D / 2) + d];
  unsigned short* dst =
      h < a.Hq ? a.C + (long)m * a.N + h * a.D + d
               : a.k_pages + ((page * a.Hkv + h - a.Hq) * a.P + slot) * a.D + d;
  dst[0] = f2bf(v * cs - u * sn);
  dst[a.D / 2] = f2bf(u * cs + v * sn);
}

// Folds the splits of such a projection, (ksplit, M, N) f32: a thread a pair of
// columns, grid M * N / 2 / 256.
__global__ __launch_bounds__(256) void rope_kv_fold_kernel(
    StreamArgs a, const float* __restrict__ part, int ksplit) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.M * (a.N / 2)) return;
  const int m = i / (a.N / 2), c = i % (a.N / 2);
  const int h = c / (a.D / 2), d = c % (a.D / 2);
  const float* p = part + (long)m * a.N + h * a.D + d;
  const long step = (long)a.M * a.N;
  float v = 0.f, u = 0.f;
#pragma unroll 8
  for (int s = 0; s < ksplit; ++s) {
    v += p[s * step];
    u += p[s * step + a.D / 2];
  }
  rope_kv_store(a, h, d, m, v, u);
}

// NW waves; RT sets of 16 rows of W (EPI_SUM: side by side), MT of 16 rows of A.
template <int EPI, int RT, int MT, bool NORM, int NW, int DP>
__global__ __launch_bounds__(NW * 64, NW / 4) void gemm_stream_kernel(StreamArgs a) {
  static_assert(EPI == EPI_SUM || RT == 2, "pairs");
  __shared__ __attribute__((aligned(16))) float sums[NW][RT * MT * 256];
  __shared__ float squares[NW][MT * 16];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int li = lane & 15, hi = lane >> 4;

  // neighbouring tiles on one XCD: each streams a stretch of W of its own
  int tile = blockIdx.x;
  {
    const int n = gridDim.x, xcd = tile % 8, q = n / 8, r = n % 8;
    if (n >= 8)
      tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + tile / 8;
  }
  int row0[RT];
  if (EPI == EPI_SUM) {
#pragma unroll
    for (int t = 0; t < RT; ++t) row0[t] = (tile * RT + t) * 16;
  } else if (EPI == EPI_SWIGLU) {
    row0[0] = tile * 16;
    row0[RT - 1] = a.N / 2 + tile * 16;
  } else {
    const int per = a.D / 32;
    row0[0] = tile / per * a.D + tile % per * 16;
    row0[RT - 1] = row0[0] + a.D / 2;
  }

  // a lane's place: 32-bit byte offsets to uniform bases, which move along K
  const unsigned wofs = (unsigned)(li * a.K + hi * 8) * 2;
  unsigned xofs[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    xofs[t] = (unsigned)(min(t * 16 + li, a.M - 1) * a.K + hi * 8) * 2;
  auto load = [](const unsigned short* base, unsigned ofs, bool once) {
    const short8* p =
        reinterpret_cast<const short8*>(reinterpret_cast<const char*>(base) + ofs);
    return as_bf16x8(once ? __builtin_nontemporal_load(p) : *p);
  };

  bf16x8 w[DP][RT][4], x[DP][MT][4];
  f32x4 acc[RT][MT], sq[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    sq[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  const int count = (a.K / 128 - wave + NW - 1) / NW;
  auto issue = [&](int d, int i) {
    const int k = (i * NW + wave) * 128;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
        w[d][t][u] = load(a.W + (long)row0[t] * a.K + k, wofs + u * 64, true);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        x[d][m][u] = load(a.A + k, xofs[m] + u * 64, false);
    }
  };
#pragma unroll
  for (int d = 0; d < DP; ++d)
    if (d < count) issue(d, d);
  for (int i = 0; i < count; i += DP) {
#pragma unroll
    for (int d = 0; d < DP; ++d) {
      if (i + d < count) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int t = 0; t < RT; ++t)
              acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  w[d][t][u], x[d][m][u], acc[t][m], 0, 0, 0);
            if (NORM)
              sq[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  x[d][m][u], x[d][m][u], sq[m], 0, 0, 0);
          }
        // keep the loads that follow above the next piece's products
        __builtin_amdgcn_sched_barrier(0);
        if (i + d + DP < count) issue(d, i + d + DP);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // acc[t][m] holds W rows hi * 4 .. +3 of A row li
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      *reinterpret_cast<f32x4*>(
          &sums[wave][(t * MT + m) * 256 + li * 16 + hi * 4]) = acc[t][m];
  if (NORM) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (hi * 4 + e == li) squares[wave][m * 16 + li] = sq[m][e];
  }
  __syncthreads();
  auto total = [&](int at) {
    float v = sums[0][at];
#pragma unroll
    for (int i = 1; i < NW; ++i) v += sums[i][at];
    return v;
  };
  constexpr int OUT = (EPI == EPI_SUM ? RT : 1) * MT * 256;
#pragma unroll
  for (int o = 0; o < (OUT + NW * 64 - 1) / (NW * 64); ++o) {
    const int at = o * NW * 64 + tid;
    const int m = at % (MT * 256) / 16, n = at & 15;
    if (at >= OUT || m >= a.M) continue;
    float r = 1.f;
    if (NORM) {
      float s = squares[0][m];
#pragma unroll
      for (int i = 1; i < NW; ++i) s += squares[i][m];
      r = rsqrtf(s / a.K + a.eps);
    }
    float v = total(at) * r;
    if (EPI == EPI_SUM) {
      const long c = (long)m * a.N + row0[RT == 1 ? 0 : at / (MT * 256)] + n;
      if (a.bias) v += bf2f(a.bias[row0[RT == 1 ? 0 : at / (MT * 256)] + n]);
      if (a.R) v += bf2f(a.R[c]);
      a.C[c] = f2bf(v);
      continue;
    }
    const float u = total(MT * 256 + at) * r;
    if (EPI == EPI_SWIGLU) {
      const float s = v / (1.f + fast_expf(-v));
      a.C[(long)m * (a.N / 2) + row0[0] + n] = f2bf(s * u);
      continue;
    }
    rope_kv_store(a, row0[0] / a.D, row0[0] % a.D + n, m, v, u);
  }
}
