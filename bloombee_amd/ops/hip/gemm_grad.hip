// The gradient of a frozen projection's input, C(M,K) = A(M,N) @ W(N,K), W as the
// projection has it: sums run over rows of W, whose fragments are read from LDS by
// columns (transposing reads).
//
// Rows of W that come in 64s take the tiles of gemm_rows.hip, TURNED (28672 x 4096: 33
// rows 45 us, 450 112, where this takes 53 and 157); this is for the others, N % 32 == 0.
//
// A 128 x 256 tile a workgroup, 32 of N a step, two buffers filled by DMA; a wave holds
// all rows of 64 columns. The sum along N is split over workgroups so that two run on
// every CU, each leaving f32 sums that a second kernel folds. Reads of LDS, of A by all
// four waves, bound large ones.

#pragma once
#include "attn_train.hip"

struct GemmGradArgs {
  const unsigned short* A;   // (M, N)
  const unsigned short* W;   // (N, K)
  unsigned short* C;         // (M, K), or null:
  float* part;               // (splits, M, K)
  int M, N, K, splits;
};

// Place of 16 B piece c of a 64 B row: the lanes that read together cover all banks.
DEVINL int grad_piece(int r, int c) {
  const int g = (r >> 2) & 3;
  return c ^ ((g & 1) << 1) ^ ((g >> 1) * 3);
}

// grid: row tiles * column tiles * splits; N % 32 == 0, K % 256 == 0
__global__ __launch_bounds__(256, 2) void gemm_grad_kernel(GemmGradArgs a) {
  constexpr int BM = 128, BN = 32, MT = BM / 32, NT = 2;
  constexpr int AB = BM * BN * 2, SUB = BN * 256;   // bytes: A, 128 columns of W
  constexpr int AI = AB / 4096, WI = 2 * SUB / 4096;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2][AB + 2 * SUB];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int li = lane & 31, hi = lane >> 5;

  // the row tiles of a column tile side by side on one XCD: they share W
  const int mt = (a.M + BM - 1) / BM, ct = a.K / 256;
  int id = blockIdx.x;
  {
    const int n = gridDim.x, q = n / 8, r = n % 8, x = id % 8;
    id = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + id / 8;
  }
  const int m0 = id % mt * BM, c0 = id / mt % ct * 256, split = id / mt / ct;
  const int steps = a.N / BN, per = (steps + a.splits - 1) / a.splits;
  const int n0 = split * per * BN, n1 = min(a.N, n0 + per * BN);

  const unsigned short* ap[AI];
  const unsigned short* wp[WI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int at = (i * 4 + wave) * 64 + lane, r = at / 4;
    ap[i] = a.A + (long)min(m0 + r, a.M - 1) * a.N + grad_piece(r, at % 4) * 8;
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int at = (i * 4 + wave) * 64 + lane, sub = at / (BN * 16), r = at / 16 % BN;
    wp[i] = a.W + (long)r * a.K + c0 + sub * 128 +
            ((at % 16) ^ TrainTile<128>::swizzle(r)) * 8;
  }
  auto issue = [&](int n, int buf) {
#pragma unroll
    for (int i = 0; i < AI; ++i)
      copy16_to_lds(ap[i] + n, lds[buf] + (i * 4 + wave) * 1024);
#pragma unroll
    for (int i = 0; i < WI; ++i)
      copy16_to_lds(wp[i] + (long)n * a.K, lds[buf] + AB + (i * 4 + wave) * 1024);
  };

  f32x16 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x16{};
  if (n0 < n1) issue(n0, 0);
  int buf = 0;
  for (int n = n0; n < n1; n += BN) {
    __syncthreads();
    if (n + BN < n1) issue(n + BN, buf ^ 1);
    const unsigned char* wt = lds[buf] + AB + (wave >> 1) * SUB;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      bf16x8 wf[NT];
#pragma unroll
      for (int c = 0; c < NT; ++c)
        wf[c] = col_frag<128>(wt, u * 16, (wave & 1) * 2 + c, lane);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int r = m * 32 + li;
        const bf16x8 af = as_bf16x8(*reinterpret_cast<const short8*>(
            lds[buf] + r * (BN * 2) + grad_piece(r, u * 2 + hi) * 16));
#pragma unroll
        for (int c = 0; c < NT; ++c)
          acc[m][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[c], af, acc[m][c], 0,
                                                              0, 0);
      }
    }
    buf ^= 1;
  }

  // a lane holds columns q * 8 + hi * 4 .. +3 of row li
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m0 + m * 32 + li;
    if (row < a.M) {
#pragma unroll
      for (int c = 0; c < NT; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const long at = (long)row * a.K + c0 + wave * 64 + c * 32 + q * 8 + hi * 4;
          if (a.C) {
            short4v v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (short)f2bf(acc[m][c][q * 4 + e]);
            *reinterpret_cast<short4v*>(a.C + at) = v;
          } else {
            *reinterpret_cast<f32x4*>(a.part + (long)split * a.M * a.K + at) =
                f32x4{acc[m][c][q * 4], acc[m][c][q * 4 + 1], acc[m][c][q * 4 + 2],
                      acc[m][c][q * 4 + 3]};
          }
        }
    }
  }
}

// Folds the splits, eight columns a thread; n = M * K.
__global__ __launch_bounds__(256) void gemm_grad_fold_kernel(
    const float* __restrict__ part, unsigned short* __restrict__ out, long n,
    int splits) {
  const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (at >= n) return;
  float v[8] = {};
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(part + s * n + at);
    const f32x4 y = *reinterpret_cast<const f32x4*>(part + s * n + at + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] += x[j];
      v[j + 4] += y[j];
    }
  }
  store_bf16x8(out + at, v);
}
