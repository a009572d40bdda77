// Row steps around the routed experts of a layer with softmax routing.

#pragma once
#include "common.h"

static constexpr int ROUTE_MAX_E = 64;

// Ahead of the experts: h = a + res, y = RMS norm of h, router logits of y, the `top`
// largest and the softmax over them. Sum, norm, logits and weights are bf16 results. Without
// norm_w the rows a are taken as they are (res, h and y null). A workgroup
// a row; a row's products with the router (64 KB for 8 x 4096) come from L2. One
// launch where norm, GEMM, conversion, top-k, sort and softmax were ten.
template <int ITERS>
__global__ __launch_bounds__(256) void norm_route_kernel(
    const unsigned short* __restrict__ a, const unsigned short* __restrict__ res,
    const unsigned short* __restrict__ norm_w,
    const unsigned short* __restrict__ router,   // (E, H)
    unsigned short* __restrict__ h, unsigned short* __restrict__ y,
    int* __restrict__ ids, float* __restrict__ wts, int H, int E, int top,
    float eps) {
  __shared__ float part[4], dots[4][ROUTE_MAX_E];
  const long at = (long)blockIdx.x * H;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid & (WAVE - 1);
  float v[ITERS][8], ss = 0.f;
#pragma unroll
  for (int i = 0; i < ITERS; ++i) {
    const int d = (i * 256 + tid) * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    if (d >= H) continue;
    load_bf16x8(a + at + d, v[i]);
    if (!norm_w) continue;
    float r[8];
    load_bf16x8(res + at + d, r);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] = bf2f(f2bf(v[i][j] + r[j]));
      ss += v[i][j] * v[i][j];
    }
    store_bf16x8(h + at + d, v[i]);
  }
  if (norm_w) {
    ss = wave_reduce_sum(ss);
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / (float)H + eps);
#pragma unroll
    for (int i = 0; i < ITERS; ++i) {
      const int d = (i * 256 + tid) * 8;
      if (d >= H) continue;
      float w[8];
      load_bf16x8(norm_w + d, w);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = bf2f(f2bf(v[i][j] * r * w[j]));
      store_bf16x8(y + at + d, v[i]);
    }
  }
  // eight experts at a time, so that their loads overlap
  for (int e0 = 0; e0 < E; e0 += 8) {
    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.f;
#pragma unroll
    for (int i = 0; i < ITERS; ++i) {
      const int d = (i * 256 + tid) * 8;
      if (d >= H) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float w[8];
        load_bf16x8(router + (long)min(e0 + e, E - 1) * H + d, w);
#pragma unroll
        for (int j = 0; j < 8; ++j) s[e] += v[i][j] * w[j];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e] = wave_reduce_sum(s[e]);
      if (lane == 0 && e0 + e < E) dots[wave][e0 + e] = s[e];
    }
  }
  __syncthreads();
  if (wave != 0) return;
  // a lane an expert; larger keys win, NaN of either sign above all, of equal ones (both
  // zeros are) the first
  float logit = 0.f;
  unsigned long long key = 0;   // taken, or no expert
  if (lane < E) {
    logit = bf2f(f2bf(dots[0][lane] + dots[1][lane] + dots[2][lane] + dots[3][lane]));
    const unsigned b = __float_as_uint(logit);
    const unsigned u = logit != logit ? 0xffffffffu
                       : logit == 0.f ? 0x80000000u
                       : (b >> 31)    ? ~b
                                      : b | 0x80000000u;
    key = ((unsigned long long)u + 1) << 8 | (unsigned)(ROUTE_MAX_E - lane);
  }
  float first = 0.f, mine = 0.f, sum = 0.f;
  int chosen = 0;
  for (int k = 0; k < top; ++k) {
    unsigned long long best = key;
#pragma unroll
    for (int m = 1; m < WAVE; m <<= 1) {
      const unsigned long long o = __shfl_xor(best, m);
      best = o > best ? o : best;
    }
    const int e = ROUTE_MAX_E - (int)(best & 255);
    const float l = __shfl(logit, e);
    if (k == 0) first = l;
    const float x = expf(l - first);
    sum += x;
    if (lane == k) {
      mine = x;
      chosen = e;
    }
    if (lane == e) key = 0;
  }
  if (lane < top) {
    ids[(long)blockIdx.x * top + lane] = chosen;
    wts[(long)blockIdx.x * top + lane] = bf2f(f2bf(mine / sum));
  }
}

// Behind them: out = h (or nothing) + the sum of a row's `top` weighted expert outputs,
// bf16 sums. Bytes bound it.
__global__ __launch_bounds__(256) void add_experts_kernel(
    const unsigned short* __restrict__ h, const unsigned short* __restrict__ y,
    unsigned short* __restrict__ out, long n, int W, int top) {
  for (long i = (blockIdx.x * 256L + threadIdx.x) * 8; i < n;
       i += gridDim.x * 2048L) {
    const long row = i / W, c = i % W;
    float v[8], s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = s[j] = 0.f;
    if (h) load_bf16x8(h + i, v);
    for (int k = 0; k < top; ++k) {
      float u[8];
      load_bf16x8(y + (row * top + k) * W + c, u);
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = bf2f(f2bf(s[j] + u[j]));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += s[j];
    store_bf16x8(out + i, v);
  }
}
