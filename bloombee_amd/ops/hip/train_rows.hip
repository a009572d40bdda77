// Row steps of the training path with their gradients: RMS norm ahead of a
// projection, SiLU-gated product behind one.

#pragma once
#include "common.h"

// Gradient of y = x / sqrt(mean(x^2) + eps) * w, plus what reaches x past the norm:
//   dx = gx + r (w gy) - x r^3 mean(w gy x),   r = 1 / sqrt(mean(x^2) + eps)
// One workgroup a row, one pass over memory: x and w gy stay in registers
// (ITERS * 2048 columns). Bytes bound it: 8 B an element with gx; 3998 rows of 4096
// 21 us, 6.3 TB/s.
template <int ITERS>
__global__ __launch_bounds__(256) void rms_norm_grad_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ gy, const unsigned short* __restrict__ gx,
    unsigned short* __restrict__ dx, int H, float eps) {
  const long at = (long)blockIdx.x * H;
  // Loads at once and not under conditions, those of gx while the sums meet (us in a graph,
  // before and now: 97 rows of 4096 3.7, 3.25; 333 4.3, 3.85; 3998 22.1, 20.9; gx with the
  // others 3.0, 3.75 and 20.5, but 8.6 for 1400 rows, 7.7 else)
  short8 xs[ITERS], gs[ITERS], ws[ITERS], o[ITERS];
  auto load = [&](const unsigned short* p, int i) {
    const int d = (i * 256 + threadIdx.x) * 8;
    return *reinterpret_cast<const short8*>(p + (d < H ? d : 0));
  };
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    xs[i] = load(x + at, i);
    gs[i] = load(gy + at, i);
    ws[i] = load(w, i);
  }
  auto f = [](short8 v, int j) { return bf2f((unsigned short)v[j]); };
  float g[ITERS][8], ss = 0.f, sg = 0.f;
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    if ((i * 256 + (int)threadIdx.x) * 8 >= H) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float xv = f(xs[i], j);
      g[i][j] = f(gs[i], j) * f(ws[i], j);
      ss += xv * xv;
      sg += g[i][j] * xv;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < ITERS; ++i) o[i] = gx ? load(gx + at, i) : short8{};
  __builtin_amdgcn_sched_barrier(0);
  __shared__ float part[2][256 / WAVE];
  ss = wave_reduce_sum(ss);
  sg = wave_reduce_sum(sg);
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    part[0][threadIdx.x / WAVE] = ss;
    part[1][threadIdx.x / WAVE] = sg;
  }
  __syncthreads();
  ss = part[0][0] + part[0][1] + part[0][2] + part[0][3];
  sg = part[1][0] + part[1][1] + part[1][2] + part[1][3];
  const float r = rsqrtf(ss / (float)H + eps);
  const float c = sg / (float)H * r * r * r;
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int d = (i * 256 + threadIdx.x) * 8;
    if (d >= H) continue;
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      y[j] = f(o[i], j) + (g[i][j] * r - f(xs[i], j) * c);
    store_bf16x8(dx + at + d, y);
  }
}

// Gradient of silu(gate) * up with gate and up side by side, (N, 2 I). Bytes bound
// it: 10 B a product; 3998 rows of 14336 96 us, 6.0 TB/s.
__global__ __launch_bounds__(256) void swiglu_grad_kernel(
    const unsigned short* __restrict__ gu, const unsigned short* __restrict__ gm,
    unsigned short* __restrict__ dgu, long N, long I) {
  const long per = I / 8;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < N * per;
       i += gridDim.x * 256L) {
    const long row = i / per, col = i % per * 8;
    float g[8], u[8], m[8], dg[8], du[8];
    load_bf16x8(gu + row * 2 * I + col, g);
    load_bf16x8(gu + row * 2 * I + I + col, u);
    load_bf16x8(gm + row * I + col, m);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s = 1.f / (1.f + fast_expf(-g[j]));
      du[j] = m[j] * g[j] * s;
      dg[j] = m[j] * u[j] * (s * (1.f + g[j] * (1.f - s)));
    }
    store_bf16x8(dgu + row * 2 * I + col, dg);
    store_bf16x8(dgu + row * 2 * I + I + col, du);
  }
}
