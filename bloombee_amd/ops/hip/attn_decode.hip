// Decode-attention support kernels for gfx950.
//
// attn_decode_combine_kernel — folds the per-split (m, l, acc) partials of
// the flash-decode MFMA kernel (attn_decode_mfma.hip) into the final output
// (softmax merge identical to the reference fp32 semantics,
// pytorch_backend.py:919-934).
// kv_stream_probe_kernel     — pure-streaming bandwidth probe of the KV walk.

#include "common.h"

typedef __attribute__((ext_vector_type(4))) short short4_v;
typedef __attribute__((ext_vector_type(2))) short short2_v;

template <int E>
DEVINL void load_bf16_e(const unsigned short* p, float* out) {
  if constexpr (E == 2) {
    short2_v v = *reinterpret_cast<const short2_v*>(p);
    out[0] = bf2f((unsigned short)v[0]);
    out[1] = bf2f((unsigned short)v[1]);
  } else if constexpr (E == 4) {
    short4_v v = *reinterpret_cast<const short4_v*>(p);
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = bf2f((unsigned short)v[j]);
  } else {
#pragma unroll
    for (int c = 0; c < E / 8; ++c) {
      short8 v = *reinterpret_cast<const short8*>(p + c * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) out[c * 8 + j] = bf2f((unsigned short)v[j]);
    }
  }
}

// Combine n_split partials: a wave a row (unit, head of the chunk), grid
// ceil(units * maxg / 4). Lanes read the splits' maxima and sums at once and share
// out the weights, so that the loads of the values do not wait for one another
// (32 splits: 15 us in a decode step when they did, about 5 now, which is a launch).
// cuts: of equal shares (attn_decode_even_kernel), a context's first one and how many.
template <int D>
__global__ __launch_bounds__(256) void attn_decode_combine_kernel(
    const float* __restrict__ part_ml, const float* __restrict__ part_acc,
    unsigned short* __restrict__ out, int units, int Hkv, int G, int nch, int maxg,
    int n_split, const int2* __restrict__ cuts, long out_sb, long out_sh) {
  constexpr int E = D >= 128 ? D / 64 : 1;   // columns of a lane
  const int row = blockIdx.x * 4 + threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);
  const int bh = row / maxg, g = row % maxg;   // bh: (b, kvh, chunk)
  if (bh >= units) return;
  const int b = bh / (Hkv * nch);
  const int rem = bh % (Hkv * nch);
  const int kvh = rem / nch;
  const int g0 = (rem % nch) * maxg;
  if (g0 + g >= G) return;
  long first = (long)bh * n_split;   // the unit's rows, `step` apart
  int step = maxg;
  if (cuts) {
    first = (long)(cuts[b].x + b) * (Hkv * nch) + rem;
    n_split = cuts[b].y;
    step = Hkv * nch * maxg;
    if (n_split == 1) return;        // is in `out`
  }
  const float* ml = part_ml + (first * maxg + g) * 2;
  float m = NEG_BIG;
  for (int s = lane; s < n_split; s += WAVE)
    if (ml[(long)s * step * 2 + 1] != 0.f) m = fmaxf(m, ml[(long)s * step * 2]);
  m = wave_reduce_max(m);
  float l = 0.f, acc[E];
#pragma unroll
  for (int j = 0; j < E; ++j) acc[j] = 0.f;
  const int col = min(lane * E, D - E);
  const float* pa = part_acc + (first * maxg + g) * D + col;
  for (int s0 = 0; s0 < n_split; s0 += WAVE) {
    const int s = s0 + lane;
    float w = 0.f, ls = 0.f;
    if (s < n_split) ls = ml[(long)s * step * 2 + 1];
    if (ls != 0.f) {
      w = fast_exp2(ml[(long)s * step * 2] - m);
      l += w * ls;
    }
    // splits beyond the context, or ahead of the window, have no sum: values are read
    // from the first to the last that has one (a window of 1024 in 4096 tokens, 8 of 32
    // splits of 256: 7.9 -> 4.9 us)
    const unsigned long long live = __builtin_amdgcn_ballot_w64(ls != 0.f);
    if (live == 0) continue;
    const int end = WAVE - __builtin_clzll(live);
#pragma unroll 8
    for (int i = __builtin_ctzll(live); i < end; ++i) {
      const float wi = __shfl(w, i);
#pragma unroll
      for (int j = 0; j < E; ++j)
        acc[j] += wi * pa[(long)(s0 + i) * step * D + j];
    }
  }
  l = wave_reduce_sum(l);
  if (lane * E >= D) return;
  const float inv = (l > 0.f) ? 1.f / l : 0.f;
  unsigned short* o = out + (long)b * out_sb + (kvh * G + g0 + g) * out_sh + col;
#pragma unroll
  for (int j = 0; j < E; ++j) o[j] = f2bf(acc[j] * inv);
}

// Pure-streaming probe: same grid/walk/loads as attn_decode_kernel but no
// softmax/acc — measures the access pattern's bandwidth ceiling. NT variant
// uses nontemporal loads (KV is read-once-per-step; keep L2 for weights).
template <int D, bool NT>
__global__ __launch_bounds__(256) void kv_stream_probe_kernel(
    const unsigned short* __restrict__ k_pages,
    const unsigned short* __restrict__ v_pages,
    const int* __restrict__ page_table, const int* __restrict__ ctx_lens,
    float* __restrict__ out, int B, int Hkv, int P, int maxp, int n_split) {
  constexpr int E = D / 16;
  const int bh = blockIdx.x;
  const int split = blockIdx.y;
  const int b = bh / Hkv, kvh = bh % Hkv;
  const int ctx = ctx_lens[b];
  const int pages_total = (ctx + P - 1) / P;
  const int pages_per_split = (pages_total + n_split - 1) / n_split;
  const int c0 = split * pages_per_split * P;
  const int c1 = min(ctx, c0 + pages_per_split * P);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = threadIdx.x / WAVE;
  const int group_id = wave * 4 + lane / 16;
  const int li = lane & 15;
  const long head_slab = (long)kvh * P * D;
  float acc = 0.f;
  for (int pos = c0 + group_id; pos < c1; pos += 16) {
    const int page = page_table[b * maxp + pos / P];
    const long off =
        ((long)page * Hkv) * P * D + head_slab + (long)(pos % P) * D + li * E;
    const short8* kp8 = reinterpret_cast<const short8*>(k_pages + off);
    const short8* vp8 = reinterpret_cast<const short8*>(v_pages + off);
#pragma unroll
    for (int c = 0; c < E / 8; ++c) {
      short8 kv = NT ? __builtin_nontemporal_load(kp8 + c) : kp8[c];
      short8 vv = NT ? __builtin_nontemporal_load(vp8 + c) : vp8[c];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += bf2f((unsigned short)kv[j]) + bf2f((unsigned short)vv[j]);
    }
  }
  acc = wave_reduce_sum(acc);
  if (lane == 0) out[(blockIdx.y * gridDim.x + blockIdx.x) * 4 + wave] = acc;
}
