// Products of a few rows with a weight matrix, C(M,N) = A(M,K) @ W(N,K)^T, M <= 32, in
// one launch with what follows them in a decoder layer:
//   EPI_SUM     [+ bias] [+ residual]
//   EPI_SWIGLU  silu(gate) * up of a fused [gate | up] projection
//   EPI_ROPE    rotations and paged K/V of a fused [q | k | v] projection
// and with the RMS norm of the rows ahead of them (its weight folded into W).
//
// The weights are streamed once and bound it. A workgroup owns 16 rows of W (two sets
// of 16 where the epilogue pairs columns) over all of K: its waves take pieces of 128
// columns in turns and add up in LDS, so that no partial sums go through memory and
// nothing has to be folded by another launch. In a decode step a launch costs about
// 5 us whatever it does (code, arguments and first loads miss caches that the weights
// swept), which is why the layer's small steps ride here.
//
// W goes straight to registers, DP pieces ahead. All of A is read by every workgroup, as
// many bytes as of W at 16 rows: it comes from L2 to a piece of LDS of the wave's own,
// in whole lines and without registers on the way (fragments straight from L2 took
// 51 us where this takes 35: 32 rows, 14336 x 4096).
// Loads of W as nontemporal cost 15% (29.5 us for 25.6: one row, 14336 x 4096): these are
// half lines. By whole ones past the caches the tiles of gemm_rows.hip are faster, and take
// what they are built for.
//
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

// Folds the splits of such a projection, (ksplit, M, N) f32, and the rows' squares,
// (ksplit, 32): a thread a pair of columns, grid M * N / 2 / 256.
__global__ __launch_bounds__(256) void rope_kv_fold_kernel(
    StreamArgs a, const float* __restrict__ part, const float* __restrict__ squares,
    int ksplit) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.M * (a.N / 2)) return;
  const int m = i / (a.N / 2), c = i % (a.N / 2);
  const int h = c / (a.D / 2), d = c % (a.D / 2);
  const float* p = part + (long)m * a.N + h * a.D + d;
  const long step = (long)a.M * a.N;
  float v = 0.f, u = 0.f, sq = 0.f;
#pragma unroll 8
  for (int s = 0; s < ksplit; ++s) {
    v += p[s * step];
    u += p[s * step + a.D / 2];
    sq += squares[s * 32 + m];
  }
  const float r = rsqrtf(sq / a.K + a.eps);
  rope_kv_store(a, h, d, m, v * r, u * r);
}

// NW waves; RT sets of 16 rows of W (EPI_SUM: side by side), MT of 16 rows of A, of
// which XN * 4 are there.
template <int EPI, int RT, int MT, int XN, bool NORM, int NW, int DP>
__global__ __launch_bounds__(NW * 64, NW / 4) void gemm_stream_kernel(StreamArgs a) {
  static_assert(EPI == EPI_SUM || RT == 2, "pairs");
  static_assert(XN <= MT * 4, "rows");
  constexpr int XB = MT * 4096;        // bytes of a piece of A
  constexpr int XT = NW * DP * XB, ST = NW * RT * MT * 1024;
  __shared__ __attribute__((aligned(16))) unsigned char lds[XT > ST ? XT : ST];
  __shared__ float squares[NW][MT * 16];
  float* sums = reinterpret_cast<float*>(lds);   // [NW][RT * MT * 256]
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
  // load t of a piece of A is rows 4 t .. +3, 16 B pieces c of row r at c ^ r: sixteen
  // rows read at one piece cover all banks
  unsigned xofs[XN];
#pragma unroll
  for (int t = 0; t < XN; ++t) {
    const int row = t * 4 + (lane >> 4), col = (lane & 15) ^ (row & 15);
    xofs[t] = (unsigned)(min(row, a.M - 1) * a.K + col * 8) * 2;
  }
  auto at_byte = [](const unsigned short* base, unsigned ofs) {
    return reinterpret_cast<const unsigned short*>(
        reinterpret_cast<const char*>(base) + ofs);
  };

  bf16x8 w[DP][RT][4];
  f32x4 acc[RT][MT], sq[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    sq[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  const int count = (a.K / 128 - wave + NW - 1) / NW;
  unsigned char* mine = lds + wave * (DP * XB);
  auto issue = [&](int d, int i) {
    const int k = (i * NW + wave) * 128;
#pragma unroll
    for (int t = 0; t < XN; ++t)
      copy16_to_lds(at_byte(a.A + k, xofs[t]), mine + d * XB + t * 1024);
    // ahead of W in every respect: whoever has waited for W has waited for these
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < RT; ++t)
        w[d][t][u] = as_bf16x8(*reinterpret_cast<const short8*>(
            at_byte(a.W + (long)row0[t] * a.K + k, wofs + u * 64)));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto consume = [&](int d) {
    // W arrives here, and with it the rows of A that were asked for before it: loads of
    // a wave return in order
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < RT; ++t) asm volatile("" : "+v"(w[d][t][u]));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const bf16x8 x = as_bf16x8(*reinterpret_cast<const short8*>(
            mine + d * XB + (m * 16 + li) * 256 + (((u * 4 + hi) ^ li) << 4)));
#pragma unroll
        for (int t = 0; t < RT; ++t)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[d][t][u], x,
                                                              acc[t][m], 0, 0, 0);
        if (NORM)
          sq[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, x, sq[m], 0, 0, 0);
      }
    // the loads that take this piece's place stay behind its products
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // The steady part has no conditions on the way, so that the wait for a piece counts
  // the loads behind it and leaves them in flight.
  int i = 0;
  if (count >= 2 * DP) {
#pragma unroll
    for (int d = 0; d < DP; ++d) issue(d, d);
    for (; i + 2 * DP <= count; i += DP)
#pragma unroll
      for (int d = 0; d < DP; ++d) {
        consume(d);
        issue(d, i + d + DP);
      }
  } else {
#pragma unroll
    for (int d = 0; d < DP; ++d)
      if (d < count) issue(d, d);
  }
  for (; i < count; i += DP)
#pragma unroll
    for (int d = 0; d < DP; ++d)
      if (i + d < count) {
        consume(d);
        if (i + d + DP < count) issue(d, i + d + DP);
      }
  __syncthreads();   // the sums take the place of the rows

  // acc[t][m] holds W rows hi * 4 .. +3 of A row li
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      *reinterpret_cast<f32x4*>(
          &sums[(wave * RT * MT + t * MT + m) * 256 + li * 16 + hi * 4]) = acc[t][m];
  if (NORM) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (hi * 4 + e == li) squares[wave][m * 16 + li] = sq[m][e];
  }
  __syncthreads();
  auto total = [&](int at) {
    float v = sums[at];
#pragma unroll
    for (int i = 1; i < NW; ++i) v += sums[i * RT * MT * 256 + at];
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

// EPI_SUM of up to RW = 16 / PARTS rows without a norm, where W has too few rows for
// workgroups of 16 to fill the chip: a workgroup owns RW rows of W, and what would be
// sixteen rows of an operand are RW of each in PARTS parts of K. Products of unequal
// parts are nobody's; those of part p are where p = li / RW = hi * 4 / RW. A wave takes 32
// * PARTS columns at a time, whole lines of each row, four such pieces on their way; A
// comes to registers, bias and residual ahead of it all.
// What a CU takes in bounds small products: with 64 of them at work 1024 x 3072 takes 5.6
// us, with all 256, each a quarter of the bytes, 4.0, of which 3 are the launch.
template <int PARTS, int NW>
__global__ __launch_bounds__(NW * 64) void gemm_stream_parts_kernel(StreamArgs a) {
  constexpr int DP = 4, RW = 16 / PARTS, STEP = 32 * PARTS, GROUPS = 64 / (RW * RW);
  __shared__ __attribute__((aligned(16))) float sums[NW * PARTS * RW * RW];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int li = lane & 15, hi = lane >> 4, part = li / RW;
  const int row0 = blockIdx.x * RW, count = a.K / STEP;
  const int m = lane % (RW * RW) / RW, n = row0 + lane % RW;   // of the way out
  const bool mine = wave == 0 && lane < RW * RW && m < a.M;
  unsigned short bias = 0, res = 0;
  if (mine && a.bias) bias = a.bias[n];
  if (mine && a.R) res = a.R[(long)m * a.N + n];
  const unsigned short* w = a.W + (long)(row0 + li % RW) * a.K + part * 32 + hi * 8;
  const unsigned short* x = a.A + (long)min(li % RW, a.M - 1) * a.K + part * 32 + hi * 8;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i = wave; i < count; i += NW * DP) {
    short8 wf[DP], xf[DP];
#pragma unroll
    for (int d = 0; d < DP; ++d) {
      const int k = min(i + d * NW, count - 1) * STEP;
      wf[d] = *reinterpret_cast<const short8*>(w + k);
      xf[d] = *reinterpret_cast<const short8*>(x + k);
    }
#pragma unroll
    for (int d = 0; d < DP; ++d) {
      if (i + d * NW >= count) wf[d] = xf[d] = short8{};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wf[d]), as_bf16x8(xf[d]),
                                                    acc, 0, 0, 0);
    }
  }
  // [wave and part][row of A][row of W]
  if (hi * 4 / RW == part)
    *reinterpret_cast<f32x4*>(
        &sums[((wave * PARTS + part) * RW + li % RW) * RW + hi * 4 % RW]) = acc;
  __syncthreads();
  if (wave) return;
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < NW * PARTS / GROUPS; ++i)
    v += sums[(lane / (RW * RW) * (NW * PARTS / GROUPS) + i) * (RW * RW) +
              lane % (RW * RW)];
#pragma unroll
  for (int o = RW * RW; o < 64; o *= 2) v += __shfl_xor(v, o);
  if (mine) a.C[(long)m * a.N + n] = f2bf(v + bf2f(bias) + bf2f(res));
}
