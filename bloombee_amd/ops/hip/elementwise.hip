// Fused elementwise / normalization kernels for gfx950.
//
// rmsnorm_kernel       — fused (optional residual-add) + RMSNorm, fp32 accum
//                        (replaces reference flexgen_utils/pytorch_backend.py:111-120;
//                        fused per SURVEY.md: HBM3E-bound ops get one pass).
// layernorm_kernel     — LayerNorm for bloom/falcon-family blocks.
// rope_kernel          — rotary embedding with arbitrary position ids
//                        (ref pytorch_backend.py:59-110), host-precomputed
//                        cos/sin tables (guide Appendix B: no device trig).
// swiglu_kernel        — SiLU(gate) * up from a fused gate_up GEMM output
//                        (ref mlp_llama, pytorch_backend.py:1033-1048).
// gelu_mul / bias ops  — falcon/bloom variants.
//
// All bf16 I/O is vectorized 16 B/lane (guide G13: scalar bf16 ~2x slower).

#include "common.h"

// ---------------------------------------------------------------------------
// RMSNorm: one workgroup per row. ITERS*BLOCK*8 >= H.
// If `res` != nullptr: h = x + res is written to out_h and normalized.
// ---------------------------------------------------------------------------

template <int BLOCK, int ITERS>
__global__ __launch_bounds__(BLOCK) void rmsnorm_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ res,
    const unsigned short* __restrict__ w, unsigned short* __restrict__ out_h,
    unsigned short* __restrict__ out_y, int H, float eps) {
  const long row = blockIdx.x;
  const unsigned short* xr = x + row * (long)H;
  const unsigned short* rr = res ? res + row * (long)H : nullptr;

  // Every load at once, the weights' as well: what it waits for bounds a row. us in a
  // graph, with loads under conditions and weights behind the barrier, and so: 25 rows of
  // 4096 2.65, 2.35; 333 3.9, 3.4; 3998 14.5, 12.9; 16 of 16384 6.2, 4.0; with a residual
  // 333 rows 4.9, 4.45.
  float v[ITERS][8], wv[ITERS][8];
  short8 r[ITERS];
  float ssq = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int d = (it * BLOCK + threadIdx.x) * 8, c = d < H ? d : 0;
    load_bf16x8(xr + c, v[it]);
    load_bf16x8(w + c, wv[it]);
    if (rr) r[it] = *reinterpret_cast<const short8*>(rr + c);
  }
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int d = (it * BLOCK + threadIdx.x) * 8;
    if (d < H) {
      if (rr) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[it][j] = bf2f(f2bf(v[it][j] + bf2f((unsigned short)r[it][j])));
        if (out_h) store_bf16x8(out_h + row * (long)H + d, v[it]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ssq += v[it][j] * v[it][j];
    }
  }
  // wave reduce then cross-wave via LDS
  ssq = wave_reduce_sum(ssq);
  __shared__ float warp_ssq[BLOCK / WAVE];
  if ((threadIdx.x & (WAVE - 1)) == 0) warp_ssq[threadIdx.x / WAVE] = ssq;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < BLOCK / WAVE; ++i) total += warp_ssq[i];
  const float inv = rsqrtf(total / (float)H + eps);

#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    int d = (it * BLOCK + threadIdx.x) * 8;
    if (d < H) {
      float o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[it][j] * inv * wv[it][j];
      store_bf16x8(out_y + row * (long)H + d, o);
    }
  }
}

// ---------------------------------------------------------------------------
// LayerNorm (bloom/falcon). Same structure, mean+var in fp32.
// ---------------------------------------------------------------------------

template <int BLOCK, int ITERS>
__global__ __launch_bounds__(BLOCK) void layernorm_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ res,
    const unsigned short* __restrict__ w, const unsigned short* __restrict__ b,
    unsigned short* __restrict__ out_h, unsigned short* __restrict__ out_y,
    int H, float eps) {
  const long row = blockIdx.x;
  const unsigned short* xr = x + row * (long)H;
  const unsigned short* rr = res ? res + row * (long)H : nullptr;

  float v[ITERS][8];
  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    int d = (it * BLOCK + threadIdx.x) * 8;
    if (d < H) {
      load_bf16x8(xr + d, v[it]);
      if (rr) {
        float r[8];
        load_bf16x8(rr + d, r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[it][j] += r[j];
        if (out_h) store_bf16x8(out_h + row * (long)H + d, v[it]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) { s1 += v[it][j]; s2 += v[it][j] * v[it][j]; }
    }
  }
  s1 = wave_reduce_sum(s1);
  s2 = wave_reduce_sum(s2);
  __shared__ float ws1[BLOCK / WAVE], ws2[BLOCK / WAVE];
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    ws1[threadIdx.x / WAVE] = s1;
    ws2[threadIdx.x / WAVE] = s2;
  }
  __syncthreads();
  float t1 = 0.f, t2 = 0.f;
#pragma unroll
  for (int i = 0; i < BLOCK / WAVE; ++i) { t1 += ws1[i]; t2 += ws2[i]; }
  const float mu = t1 / (float)H;
  const float inv = rsqrtf(t2 / (float)H - mu * mu + eps);

#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    int d = (it * BLOCK + threadIdx.x) * 8;
    if (d < H) {
      float wv[8], bv[8], o[8];
      load_bf16x8(w + d, wv);
      if (b) load_bf16x8(b + d, bv);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o[j] = (v[it][j] - mu) * inv * wv[j] + (b ? bv[j] : 0.f);
      }
      store_bf16x8(out_y + row * (long)H + d, o);
    }
  }
}

// ---------------------------------------------------------------------------
// RoPE (half-split convention), in place on q and k.
// q: (B, Hq, T, D)  k: (B, Hkv, T, D)  pos: (B, T) int32
// cos/sin: (max_pos, D/2) f32, precomputed on host.
// grid: (B*T, Hq + Hkv), block: 64.
// ---------------------------------------------------------------------------

__global__ void rope_kernel(
    unsigned short* __restrict__ q, unsigned short* __restrict__ k,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    const int* __restrict__ pos, int B, int Hq, int Hkv, int T, int D,
    int max_pos) {
  const int bt = blockIdx.x;
  const int b = bt / T, t = bt % T;
  const int h = blockIdx.y;
  unsigned short* base =
      (h < Hq) ? q + (((long)b * Hq + h) * T + t) * D
               : k + (((long)b * Hkv + (h - Hq)) * T + t) * D;
  // clamp: positions past the rope table (model max_position_embeddings)
  // must not read out of bounds — the python layer guards the supported
  // range, this is the device-safety net
  const int p = min(max(pos[b * T + t], 0), max_pos - 1);
  const float* c = cos_t + (long)p * (D / 2);
  const float* s = sin_t + (long)p * (D / 2);
  for (int i = threadIdx.x; i < D / 2; i += blockDim.x) {
    float x1 = bf2f(base[i]), x2 = bf2f(base[i + D / 2]);
    float cc = c[i], ss = s[i];
    base[i] = f2bf(x1 * cc - x2 * ss);
    base[i + D / 2] = f2bf(x2 * cc + x1 * ss);
  }
}

// ---------------------------------------------------------------------------
// SwiGLU: out[n, i] = silu(gu[n, i]) * gu[n, I + i];  gu: (N, 2I)
// ---------------------------------------------------------------------------

__global__ void swiglu_kernel(const unsigned short* __restrict__ gu,
                              unsigned short* __restrict__ out, long N, long I) {
  const long nvec = N * (I / 8);
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < nvec;
       idx += (long)gridDim.x * blockDim.x) {
    const long row = idx / (I / 8);
    const long col = (idx % (I / 8)) * 8;
    float g[8], u[8], o[8];
    load_bf16x8(gu + row * 2 * I + col, g);
    load_bf16x8(gu + row * 2 * I + I + col, u);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float s = g[j] / (1.f + fast_expf(-g[j]));
      o[j] = s * u[j];
    }
    store_bf16x8(out + row * I + col, o);
  }
}

// gelu(tanh approx)(x) * 1.0 — falcon/bloom MLP activation, out-of-place.
__global__ void gelu_kernel(const unsigned short* __restrict__ x,
                            unsigned short* __restrict__ out, long n) {
  const long nvec = n / 8;
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < nvec;
       idx += (long)gridDim.x * blockDim.x) {
    float v[8], o[8];
    load_bf16x8(x + idx * 8, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float t = tanhf(0.7978845608028654f * (v[j] + 0.044715f * v[j] * v[j] * v[j]));
      o[j] = 0.5f * v[j] * (1.f + t);
    }
    store_bf16x8(out + idx * 8, o);
  }
}

// residual add: out = a + b (bf16), used where no norm fusion applies
__global__ void add_kernel(const unsigned short* __restrict__ a,
                           const unsigned short* __restrict__ b,
                           unsigned short* __restrict__ out, long n) {
  const long nvec = n / 8;
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < nvec;
       idx += (long)gridDim.x * blockDim.x) {
    float va[8], vb[8], o[8];
    load_bf16x8(a + idx * 8, va);
    load_bf16x8(b + idx * 8, vb);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = va[j] + vb[j];
    store_bf16x8(out + idx * 8, o);
  }
}

// ---------------------------------------------------------------------------
// Fused RoPE + paged-KV write on the raw QKV GEMM output (B, T, (Hq+2Hkv)*D).
// q heads: rotary in place. k heads: rotary -> k_pages (never written back).
// v heads: straight copy -> v_pages. One launch replaces rope + kv_write and
// removes every transpose copy between the QKV GEMM and attention.
// q_norm, k_norm: weights of an RMS norm of every head ahead of its rotation, or null;
// neither without NORM, whose code costs others 0.1 of 2.4 us.
// grid: (B*T, Hq+2Hkv), block: 64.
// ---------------------------------------------------------------------------

template <bool NORM>
__global__ void rope_kv_write_kernel(
    unsigned short* __restrict__ qkv, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, const int* __restrict__ pos,
    unsigned short* __restrict__ k_pages, unsigned short* __restrict__ v_pages,
    const int* __restrict__ page_table, const int* __restrict__ start_pos,
    int B, int Hq, int Hkv, int T, int D, int P, int maxp, int max_pos,
    const unsigned short* __restrict__ q_norm,
    const unsigned short* __restrict__ k_norm, float eps) {
  const int bt = blockIdx.x;
  const int b = bt / T, t = bt % T;
  const int h = blockIdx.y;
  const int X = Hq + 2 * Hkv;
  unsigned short* base = qkv + (((long)b * T + t) * X + h) * D;

  const int abspos = start_pos[b] + t;
  if (h >= Hq + Hkv) {  // v head: copy to pages (d-major V layout: transpose
    const int hv = h - Hq - Hkv;  // on write, scattered 2 B stores, once/token)
    const int page = page_table[b * maxp + abspos / P];
    const int slot = abspos % P;
    unsigned short* dst = v_pages + ((long)page * Hkv + hv) * D * P + slot;
    for (int i = threadIdx.x; i < D; i += blockDim.x)
      dst[(long)i * P] = base[i];
    return;
  }
  const int p = min(max(pos ? pos[b * T + t] : abspos, 0), max_pos - 1);
  const float* c = cos_t + (long)p * (D / 2);
  const float* s = sin_t + (long)p * (D / 2);
  unsigned short* dst = base;
  if (h >= Hq) {  // k head: write rotated values to pages only
    const int hk = h - Hq;
    const int page = page_table[b * maxp + abspos / P];
    dst = k_pages + (((long)page * Hkv + hk) * P + (abspos % P)) * D;
  }
  const unsigned short* nw = NORM ? h < Hq ? q_norm : k_norm : nullptr;
  float r = 1.f;
  if (nw) {
    float sq = 0.f;
    for (int i = threadIdx.x; i < D; i += blockDim.x) {
      const float x = bf2f(base[i]);
      sq += x * x;
    }
    r = rsqrtf(wave_reduce_sum(sq) / (float)D + eps);
  }
  for (int i = threadIdx.x; i < D / 2; i += blockDim.x) {
    float x1 = bf2f(base[i]), x2 = bf2f(base[i + D / 2]);
    if (nw) {
      x1 *= r * bf2f(nw[i]);
      x2 *= r * bf2f(nw[i + D / 2]);
    }
    float cc = c[i], ss = s[i];
    dst[i] = f2bf(x1 * cc - x2 * ss);
    dst[i + D / 2] = f2bf(x2 * cc + x1 * ss);
  }
}

// The same for many tokens, D = 16 L: memory bounds it, so a lane takes eight elements
// of both halves of a head, and values go to their pages as eight tokens of a page row,
// gathered from as many rows of the projection. 4 x 4096 tokens of 32, 8 and 8 heads of
// 128: 70 us, 5.8 TB/s (two bytes at a time 233). grid: qk_blocks of 256 / L heads,
// then 256 pairs of columns of an octet of tokens each, octs octets a sequence and head.
template <int L>
__global__ __launch_bounds__(256) void rope_kv_rows_kernel(
    unsigned short* __restrict__ qkv, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, const int* __restrict__ pos,
    unsigned short* __restrict__ k_pages, unsigned short* __restrict__ v_pages,
    const int* __restrict__ page_table, const int* __restrict__ start_pos,
    int B, int Hq, int Hkv, int T, int P, int maxp, int max_pos,
    const unsigned short* __restrict__ q_norm,
    const unsigned short* __restrict__ k_norm, float eps, int qk_blocks, int octs) {
  constexpr int D = 16 * L, H2 = D / 2;
  const long row = (long)(Hq + 2 * Hkv) * D;
  if ((int)blockIdx.x < qk_blocks) {
    const long item = ((long)blockIdx.x * 256 + threadIdx.x) / L;
    const int i = threadIdx.x % L * 8;
    const long bt = item / (Hq + Hkv);
    const int h = (int)(item - bt * (Hq + Hkv));
    if (bt >= (long)B * T) return;
    const int b = (int)(bt / T), at = start_pos[b] + (int)(bt - (long)b * T);
    unsigned short* src = qkv + bt * row + h * D + i;
    float x1[8], x2[8];
    load_bf16x8(src, x1);
    load_bf16x8(src + H2, x2);
    const unsigned short* nw = h < Hq ? q_norm : k_norm;
    if (nw) {
      float sq = 0.f, w1[8], w2[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sq += x1[j] * x1[j] + x2[j] * x2[j];
#pragma unroll
      for (int o = 1; o < L; o <<= 1) sq += __shfl_xor(sq, o);
      const float r = rsqrtf(sq / (float)D + eps);
      load_bf16x8(nw + i, w1);
      load_bf16x8(nw + i + H2, w2);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x1[j] *= r * w1[j];
        x2[j] *= r * w2[j];
      }
    }
    const int p = min(max(pos ? pos[bt] : at, 0), max_pos - 1);
    const float* cs = cos_t + (long)p * H2 + i;
    const float* sn = sin_t + (long)p * H2 + i;
    float o1[8], o2[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float c = cs[j], s = sn[j];
      o1[j] = x1[j] * c - x2[j] * s;
      o2[j] = x2[j] * c + x1[j] * s;
    }
    unsigned short* dst = src;
    if (h >= Hq) {
      const long page = page_table[(long)b * maxp + at / P];
      dst = k_pages + ((page * Hkv + h - Hq) * P + at % P) * D + i;
    }
    store_bf16x8(dst, o1);
    store_bf16x8(dst + H2, o2);
    return;
  }
  const long idx = (long)(blockIdx.x - qk_blocks) * 256 + threadIdx.x;
  const int d = (int)(idx % H2) * 2;
  long rest = idx / H2;
  const int o = (int)(rest % octs);
  rest /= octs;
  const int h = (int)(rest % Hkv), b = (int)(rest / Hkv);
  if (b >= B) return;
  const int start = start_pos[b], p0 = (start / 8 + o) * 8;
  if (p0 >= start + T) return;
  const unsigned short* src = qkv + (long)b * T * row + (Hq + Hkv + h) * D + d;
  unsigned v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = *reinterpret_cast<const unsigned*>(
        src + min(max(p0 + j - start, 0), T - 1) * row);
  const long page = page_table[(long)b * maxp + p0 / P];
  unsigned short* dst = v_pages + ((page * Hkv + h) * D + d) * P + p0 % P;
  if (p0 >= start && p0 + 8 <= start + T) {
    short8 lo, hi;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      lo[j] = (short)(v[j] & 0xffff);
      hi[j] = (short)(v[j] >> 16);
    }
    *reinterpret_cast<short8*>(dst) = lo;
    *reinterpret_cast<short8*>(dst + P) = hi;
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (p0 + j >= start && p0 + j < start + T) {
      dst[j] = (unsigned short)(v[j] & 0xffff);
      dst[P + j] = (unsigned short)(v[j] >> 16);
    }
}
