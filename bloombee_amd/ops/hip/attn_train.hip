// Causal attention of whole sequences with its gradients, rotations included.
//
//  rope_rows_kernel        rotates queries and keys of a fused [q | k | v] projection
//                          into a buffer of their own.
//  attn_train_kernel       the attention; keeps the 32-bit result and each row's
//                          log-sum for the gradients.
//  attn_train_dq_kernel    gradients of the queries, turned back; a row's
//                          sum(dO * O) on the way, for the next kernel.
//  attn_train_dkv_kernel   gradients of keys (turned back) and values, summed over
//                          the heads of a group in registers.
//
// Rows are (token, head of the group) pairs. All products are
// v_mfma_f32_32x32x16_bf16. Scores and weights never reach memory: the gradient
// kernels make them anew, the first with a row a lane (S^T, what it adds up is over
// keys), the second with a key a lane (S, what it adds up is over rows), so that each
// finds its second products' operand in its registers: the keys (rows) of a product
// are taken in an order, bits 2 and 3 of their number swapped, in which the 16
// results of a lane are the eight consecutive ones it hands to each of two products.
// The other operand has to be read by columns, which the transposing LDS reads do.
// No atomics; every sum has a fixed order.
//
// Weights and their gradients are 32-bit. They enter the second products as a sum of
// two bf16 (the value and what its rounding lost); queries, keys, values and dO are
// bf16 already. So a product loses no more than 2^-17 of a term. Errors against 64 bits
// over 12 sizes of 33 to 1999 tokens, inputs of scale 1 and 3, beside those of weights
// kept in 32 bits (torch operations): results 0.0021 to 0.0077, the same; gradients of
// queries 0.0027 to 0.0140 (0.0031 to 0.0141), keys 0.0028 to 0.0141 (0.0035 to 0.0143),
// values 0.0022 to 0.0077 (0.0028 to 0.0079): a group's heads are summed in 32 bits here.
//
// 3, 4 and 6 products of 32 x 32 x D a tile. Two sequences of 1999, 32 heads on 8 of 128:
// 132, 167 and 234 us (743, 784 and 840 TF/s of the visible half); as float32 torch
// operations a layer's attention took 9.2 ms both ways. The first two keep the matrix cores
// busy for 37 and 39% of that, and the vector units, which weigh and split, for as much; the
// third is described where it stands.

#pragma once
#include "common.h"

struct TrainAttnArgs {
  const unsigned short* qk;    // (B, T, Hq + Hkv, D) rotated
  const unsigned short* qkv;   // (B, T, Hq + 2 Hkv, D)
  const unsigned short* dout;  // (B, T, Hq, D)
  const float* cos_t;          // (positions, D / 2)
  const float* sin_t;
  unsigned short* out;         // (B, T, Hq, D)
  float* out32;                // the same, or null: no gradients wanted
  float* lse;                  // (B * Hkv, T * G) log2 units
  float* delta;                // (B * Hkv, T * G)
  unsigned short* dqkv;        // (B, T, Hq + 2 Hkv, D)
  int B, T, Hkv, G, start;
  float scale;
};

template <int D>
struct TrainTile {
  static constexpr int RC = D / 8;                // 16 B pieces of a row
  static constexpr int BYTES = 64 * D * 2;        // 64 rows
  static constexpr int NI = BYTES / 1024 / 4;     // loads of a wave
  // piece c of row r lies at c ^ swizzle(r). Sixteen rows read at one piece, and
  // four rows read at four consecutive pieces, cover all banks.
  DEVINL static int swizzle(int r) {
    return RC >= 16 ? ((r & 3) << 2) | ((r >> 2) & 3)
                    : ((r & 2) << 1) | ((r >> 2) & 3);
  }
};

typedef __attribute__((address_space(3))) short4v train_lds4;

// MFMA row -> row of the tile it stands for.
DEVINL int swap23(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

// Eight elements of row `row` from kk * 16 + hi * 8.
template <int D>
DEVINL bf16x8 row_frag(const unsigned char* tile, int row, int kk, int hi) {
  return as_bf16x8(*reinterpret_cast<const short8*>(
      tile + row * (D * 2) + (((kk * 2 + hi) ^ TrainTile<D>::swizzle(row)) << 4)));
}

// Column n * 32 + (lane & 31) of rows r0 + (lane >> 5) * 8 .. +7; r0 % 16 == 0.
template <int D>
DEVINL bf16x8 col_frag(const unsigned char* tile, int r0, int n, int lane) {
  const int i = lane & 15, row = r0 + (lane >> 5) * 8 + (i >> 2);
  const int piece = n * 4 + ((lane >> 4) & 1) * 2 + ((i >> 1) & 1);
  short8 v;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = row + q * 4;
    const short4v c = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (train_lds4*)(tile + r * (D * 2) +
                      ((piece ^ TrainTile<D>::swizzle(r)) << 4) + (i & 1) * 8));
#pragma unroll
    for (int e = 0; e < 4; ++e) v[q * 4 + e] = c[e];
  }
  return as_bf16x8(v);
}

DEVINL void split_pair(const float* p, bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    hi[j] = (__bf16)p[j];
    lo[j] = (__bf16)(p[j] - (float)hi[j]);
  }
}

// Rows of two (token, head) tensors that a workgroup's kernels read.
struct RowMap {
  const unsigned short* base;
  long ld;      // of a token
  int G;        // heads taken in turns
  DEVINL const unsigned short* at(int row, int D) const {
    return base + (long)(row / G) * ld + row % G * D;
  }
};

// 64 rows from r0 to LDS, rows beyond `last` repeat it.
template <int D>
DEVINL void stage_rows(const RowMap& m, int r0, int last, unsigned char* tile,
                       int wave, int lane) {
  using Tile = TrainTile<D>;
#pragma unroll
  for (int i = 0; i < Tile::NI; ++i) {
    const int at = (wave + i * 4) * 64 + lane;
    const int r = at / Tile::RC, c = (at % Tile::RC) ^ Tile::swizzle(r);
    dma16_to_lds(m.at(min(r0 + r, last), D) + c * 8, tile + (wave + i * 4) * 1024);
  }
}

// The same for tiles that begin at multiples of 64. Where the heads of a group divide 64
// and no row is beyond `last`, a lane's offsets from the tile's first row are those of any
// tile, and nothing is calculated (a division and a 64-bit product a load otherwise).
template <int D>
struct RowStage {
  using Tile = TrainTile<D>;
  RowMap m;
  long step;               // from a tile's first row to the next one's
  int last, wave, lane;
  unsigned ofs[Tile::NI];
  DEVINL RowStage(const RowMap& rows, int last_, int wave_, int lane_)
      : m(rows), step(64 % rows.G ? 0 : 64 / rows.G * rows.ld), last(last_),
        wave(wave_), lane(lane_) {
#pragma unroll
    for (int i = 0; i < Tile::NI; ++i) {
      const int at = (wave + i * 4) * 64 + lane;
      const int r = at / Tile::RC, c = (at % Tile::RC) ^ Tile::swizzle(r);
      ofs[i] = (unsigned)((r / m.G * m.ld + r % m.G * D + c * 8) * 2);
    }
  }
  DEVINL void operator()(int r0, unsigned char* tile) const {
    if (step == 0 || r0 + 63 > last) {
      stage_rows<D>(m, r0, last, tile, wave, lane);
      return;
    }
    const unsigned short* base = m.base + (r0 >> 6) * step;
#pragma unroll
    for (int i = 0; i < Tile::NI; ++i)
      dma16(base, ofs[i],
            (unsigned)(unsigned long)(lptr_t)(tile + (wave + i * 4) * 1024));
  }
};

// grid: ceil(B * T * (Hq + Hkv) * D / 16 / 256); a thread turns eight pairs
__global__ __launch_bounds__(256) void rope_rows_kernel(
    const unsigned short* __restrict__ qkv, unsigned short* __restrict__ qk,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, long tokens,
    int T, int heads, int X, int D, int start) {
  const int per = D / 16;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= tokens * heads * per) return;
  const int c = (int)(i % per) * 8;
  const int h = (int)(i / per % heads);
  const long t = i / per / heads;
  const unsigned short* src = qkv + (t * X + h) * D + c;
  unsigned short* dst = qk + (t * heads + h) * D + c;
  const long p = (long)(start + (int)(t % T)) * (D / 2) + c;
  float x[8], y[8], u[8], v[8];
  load_bf16x8(src, x);
  load_bf16x8(src + D / 2, y);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float cs = cos_t[p + j], sn = sin_t[p + j];
    u[j] = x[j] * cs - y[j] * sn;
    v[j] = y[j] * cs + x[j] * sn;
  }
  store_bf16x8(dst, u);
  store_bf16x8(dst + D / 2, v);
}

// grid (B * Hkv, row tiles of 128); four waves of 32 rows
template <int D>
__global__ __launch_bounds__(256, 2) void attn_train_kernel(TrainAttnArgs a) {
  using Tile = TrainTile<D>;
  constexpr int KT = 64, NKK = D / 16, ND = D / 32;
  __shared__ __attribute__((aligned(16))) unsigned char lds[4 * Tile::BYTES];
  const int b = blockIdx.x / a.Hkv, g = blockIdx.x % a.Hkv;
  const int G = a.G, R = a.T * G, Hq = a.Hkv * G;
  const int base = (int)(gridDim.y - 1 - blockIdx.y) * 128;  // long rows first
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int li = lane & 31, hi = lane >> 5;
  const long ldq = (long)(Hq + a.Hkv) * D, ldx = (long)(Hq + 2 * a.Hkv) * D;
  const unsigned short* qb = a.qk + (long)b * a.T * ldq;
  const RowMap keys{qb + (long)(Hq + g) * D, ldq, 1};
  const RowMap vals{a.qkv + (long)b * a.T * ldx + (long)(Hq + a.Hkv + g) * D, ldx, 1};
  const RowMap rows{qb + (long)g * G * D, ldq, G};

  const int row = base + wave * 32 + li;
  const int r = min(row, R - 1), tok = r / G;
  bf16x8 qf[NKK];
  const unsigned short* qp = rows.at(r, D) + hi * 8;
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)
    qf[kk] = as_bf16x8(*reinterpret_cast<const short8*>(qp + kk * 16));
  const float sc2 = a.scale * LOG2E;
  const int kend = (min(base + 128, R) - 1) / G + 1;
  const int w0 = base + wave * 32;
  const int wlast = w0 >= R ? -1 : min(w0 + 31, R - 1) / G;
  const int wfull = w0 / G;    // keys up to here are seen by all rows of the wave
  const int krow = swap23(li);

  float m = NEG_BIG, l = 0.f;
  f32x16 acc[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) acc[n] = f32x16{};

  stage_rows<D>(keys, 0, kend - 1, lds, wave, lane);
  stage_rows<D>(vals, 0, kend - 1, lds + Tile::BYTES, wave, lane);
  wait_loads<0>();
  __syncthreads();
  int buf = 0;
  for (int kb = 0; kb < kend; kb += KT) {
    if (kb + KT < kend) {
      unsigned char* next = lds + (buf ^ 1) * 2 * Tile::BYTES;
      stage_rows<D>(keys, kb + KT, kend - 1, next, wave, lane);
      stage_rows<D>(vals, kb + KT, kend - 1, next + Tile::BYTES, wave, lane);
    }
    const unsigned char* kt = lds + buf * 2 * Tile::BYTES;
    if (kb <= wlast) {
      f32x16 s[2];
      s[0] = s[1] = f32x16{};
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
        for (int n = 0; n < 2; ++n)
          s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              row_frag<D>(kt, n * 32 + krow, kk, hi), qf[kk], s[n], 0, 0, 0);
      // s[n][j] is key kb + n * 32 + (j & 8) * 2 + hi * 8 + (j & 7)
      if (kb + KT - 1 > wfull) {
        const int d0 = tok - kb - hi * 8;
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (n * 32 + (j & 8) * 2 + (j & 7) > d0) s[n][j] = NEG_BIG;
      }
      float mx = m;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s[n][j]);
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      if (__builtin_amdgcn_ballot_w64(mx > m)) {
        const float corr = fast_exp2((m - mx) * sc2);
        l *= corr;
#pragma unroll
        for (int n = 0; n < ND; ++n)
#pragma unroll
          for (int j = 0; j < 16; ++j) acc[n][j] *= corr;
        m = mx;
      }
      const float ref = m > 0.5f * NEG_BIG ? m * sc2 : 0.f;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float p[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            p[e] = fast_exp2(fmaf(s[n][j * 8 + e], sc2, -ref));
            l += p[e];
          }
          bf16x8 ph, pl;
          split_pair(p, ph, pl);
#pragma unroll
          for (int d = 0; d < ND; ++d) {
            const bf16x8 vf =
                col_frag<D>(kt + Tile::BYTES, n * 32 + j * 16, d, lane);
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, ph, acc[d], 0, 0, 0);
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pl, acc[d], 0, 0, 0);
          }
        }
    }
    wait_loads<0>();
    __syncthreads();
    buf ^= 1;
  }

  l += __shfl_xor(l, 32);
  if (row >= R) return;
  const float inv = 1.f / l;
  const long at = (((long)b * a.T + tok) * Hq + g * G + r % G) * D + hi * 4;
  if (a.out32 && hi == 0)
    a.lse[(long)blockIdx.x * R + r] = m * sc2 + __log2f(l);
#pragma unroll
  for (int n = 0; n < ND; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 o;
      short4v u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = acc[n][j * 4 + e] * inv;
        u[e] = (short)f2bf(o[e]);
      }
      *reinterpret_cast<short4v*>(a.out + at + n * 32 + j * 8) = u;
      if (a.out32) *reinterpret_cast<f32x4*>(a.out32 + at + n * 32 + j * 8) = o;
    }
}

// grid and rows as above
template <int D>
__global__ __launch_bounds__(256, 2) void attn_train_dq_kernel(TrainAttnArgs a) {
  using Tile = TrainTile<D>;
  constexpr int KT = 64, NKK = D / 16, ND = D / 32;
  __shared__ __attribute__((aligned(16))) unsigned char lds[4 * Tile::BYTES];
  const int b = blockIdx.x / a.Hkv, g = blockIdx.x % a.Hkv;
  const int G = a.G, R = a.T * G, Hq = a.Hkv * G;
  const int base = (int)(gridDim.y - 1 - blockIdx.y) * 128;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int li = lane & 31, hi = lane >> 5;
  const long ldq = (long)(Hq + a.Hkv) * D, ldx = (long)(Hq + 2 * a.Hkv) * D;
  const unsigned short* qb = a.qk + (long)b * a.T * ldq;
  const RowMap keys{qb + (long)(Hq + g) * D, ldq, 1};
  const RowMap vals{a.qkv + (long)b * a.T * ldx + (long)(Hq + a.Hkv + g) * D, ldx, 1};
  const RowMap rows{qb + (long)g * G * D, ldq, G};

  const int row = base + wave * 32 + li;
  const int r = min(row, R - 1), tok = r / G;
  const long at = (((long)b * a.T + tok) * Hq + g * G + r % G) * D;
  bf16x8 qf[NKK], of[NKK];
  const unsigned short* qp = rows.at(r, D) + hi * 8;
  float del = 0.f;
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    qf[kk] = as_bf16x8(*reinterpret_cast<const short8*>(qp + kk * 16));
    const long c = at + kk * 16 + hi * 8;
    of[kk] = as_bf16x8(*reinterpret_cast<const short8*>(a.dout + c));
#pragma unroll
    for (int e = 0; e < 8; ++e) del += (float)of[kk][e] * a.out32[c + e];
  }
  del += __shfl_xor(del, 32);
  const float lse = a.lse[(long)blockIdx.x * R + r];
  if (hi == 0 && row < R) a.delta[(long)blockIdx.x * R + r] = del;
  const float sc2 = a.scale * LOG2E;
  const int kend = (min(base + 128, R) - 1) / G + 1;
  const int w0 = base + wave * 32;
  const int wlast = w0 >= R ? -1 : min(w0 + 31, R - 1) / G;
  const int wfull = w0 / G;
  const int krow = swap23(li);

  f32x16 acc[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) acc[n] = f32x16{};

  stage_rows<D>(keys, 0, kend - 1, lds, wave, lane);
  stage_rows<D>(vals, 0, kend - 1, lds + Tile::BYTES, wave, lane);
  wait_loads<0>();
  __syncthreads();
  int buf = 0;
  for (int kb = 0; kb < kend; kb += KT) {
    if (kb + KT < kend) {
      unsigned char* next = lds + (buf ^ 1) * 2 * Tile::BYTES;
      stage_rows<D>(keys, kb + KT, kend - 1, next, wave, lane);
      stage_rows<D>(vals, kb + KT, kend - 1, next + Tile::BYTES, wave, lane);
    }
    const unsigned char* kt = lds + buf * 2 * Tile::BYTES;
    if (kb <= wlast) {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        f32x16 s = f32x16{}, dp = f32x16{};
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
          s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              row_frag<D>(kt, n * 32 + krow, kk, hi), qf[kk], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              row_frag<D>(kt + Tile::BYTES, n * 32 + krow, kk, hi), of[kk], dp, 0, 0,
              0);
        }
        const int d0 = tok - kb - hi * 8;
        const bool edge = kb + KT - 1 > wfull;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float ds[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float p = fast_exp2(fmaf(s[j * 8 + e], sc2, -lse));
            ds[e] = p * (dp[j * 8 + e] - del);
            if (edge && n * 32 + j * 16 + e > d0) ds[e] = 0.f;
          }
          bf16x8 dh, dl;
          split_pair(ds, dh, dl);
#pragma unroll
          for (int d = 0; d < ND; ++d) {
            const bf16x8 kf = col_frag<D>(kt, n * 32 + j * 16, d, lane);
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, dh, acc[d], 0, 0, 0);
            acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, dl, acc[d], 0, 0, 0);
          }
        }
      }
    }
    wait_loads<0>();
    __syncthreads();
    buf ^= 1;
  }

  if (row >= R) return;
  // back through the rotation: element d turned with element d + D / 2
  unsigned short* dq = a.dqkv + ((long)b * a.T + tok) * ldx +
                       (long)(g * G + r % G) * D + hi * 4;
  const long p = (long)(a.start + tok) * (D / 2) + hi * 4;
#pragma unroll
  for (int n = 0; n < ND / 2; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      short4v x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float cs = a.cos_t[p + n * 32 + j * 8 + e];
        const float sn = a.sin_t[p + n * 32 + j * 8 + e];
        const float u = acc[n][j * 4 + e] * a.scale;
        const float v = acc[n + ND / 2][j * 4 + e] * a.scale;
        x[e] = (short)f2bf(u * cs + v * sn);
        y[e] = (short)f2bf(v * cs - u * sn);
      }
      *reinterpret_cast<short4v*>(dq + n * 32 + j * 8) = x;
      *reinterpret_cast<short4v*>(dq + D / 2 + n * 32 + j * 8) = y;
    }
}

DEVINL void dma4(const void* base, unsigned ofs, unsigned l) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :: "s"(l), "v"(ofs), "s"(base) : "m0");
}

// Where the tiles of 64 rows wait: one is worked on, the next one's rows are read as well,
// two are on their way.
template <int D>
struct TrainRing {
  static constexpr int DEPTH = 4;
  static constexpr int SLOT = 2 * TrainTile<D>::BYTES + 1024;
  static constexpr int LOADS = 2 * TrainTile<D>::NI + 1;   // of a wave and tile
  static constexpr int BYTES = DEPTH * SLOT;
};

// grid (B * Hkv, tiles of 64 keys); waves 0 and 1 own 32 keys each, waves 2 and 3 the
// same keys: the two pairs take the two halves of a tile of 64 rows and add up at the
// end. 192 accumulator and operand registers leave room for one wave a SIMD; tiles of
// 64 keys and not 128 make twice as many workgroups with half as long a chain.
//
// With one wave a SIMD nothing overlaps but what the wave's own order lets: the products
// of a tile run beside the vector work and the LDS reads of its neighbours. 16 products of
// the last tile's second half hide the reads of this one's numbers and the next one's rows,
// the next one's 16 score products half of the weights (about ten instructions an element)
// and the reads of columns, 16 products of the first half the rest. Two sequences of 1999,
// 32 heads on 8 of 128: products and vector work one after the other, every read waited
// for, 410 us; reads at once, addresses of constant offsets 291; tiles three ahead 288; the
// order above 262; sums exchanged both ways at the end, rotation tables read at once 252, all
// in one session (234 in later ones; the wait for reads of LDS ahead of the barrier costs
// nothing). 600 tokens: 103 us, now 60. What is left: a tile's 48 products take 770 ns of
// 1900, its LDS traffic (160 KB a workgroup) about 600.
template <int D>
__global__ __launch_bounds__(256, 1) void attn_train_dkv_kernel(TrainAttnArgs a) {
  using Tile = TrainTile<D>;
  constexpr int NKK = D / 16, ND = D / 32;
  using Ring = TrainRing<D>;
  extern __shared__ __attribute__((aligned(16))) unsigned char train_lds[];
  const int b = blockIdx.x / a.Hkv, g = blockIdx.x % a.Hkv;
  const int G = a.G, R = a.T * G, Hq = a.Hkv * G;
  const int k0 = blockIdx.y * 64;                // early keys are seen most
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int li = lane & 31, hi = lane >> 5;
  const int half = (wave >> 1) * 32;
  const long ldq = (long)(Hq + a.Hkv) * D, ldx = (long)(Hq + 2 * a.Hkv) * D;
  const unsigned short* qb = a.qk + (long)b * a.T * ldq;
  const RowMap rows{qb + (long)g * G * D, ldq, G};
  const RowMap outs{a.dout + ((long)b * a.T * Hq + (long)g * G) * D, (long)Hq * D, G};
  const float* lse = a.lse + (long)blockIdx.x * R;
  const float* delta = a.delta + (long)blockIdx.x * R;

  const int key = k0 + (wave & 1) * 32 + li;
  bf16x8 kf[NKK], vf[NKK];
  {
    const long t = (long)b * a.T + min(key, a.T - 1);
    const unsigned short* kp = a.qk + t * ldq + (long)(Hq + g) * D + hi * 8;
    const unsigned short* vp = a.qkv + t * ldx + (long)(Hq + a.Hkv + g) * D + hi * 8;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      kf[kk] = as_bf16x8(*reinterpret_cast<const short8*>(kp + kk * 16));
      vf[kk] = as_bf16x8(*reinterpret_cast<const short8*>(vp + kk * 16));
    }
  }
  const float sc2 = a.scale * LOG2E;
  const int first = key * G;                     // rows from here on see the key
  const int full = (k0 + (wave & 1) * 32 + 31) * G;   // ... all keys of the wave
  const int qrow = half + swap23(li);

  f32x16 dk[ND], dv[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) {
    dk[n] = dv[n] = f32x16{};
    // known zeros would be carried through the loop as 16 numbers each, and copied
    asm volatile("" : "+a"(dk[n]), "+a"(dv[n]));
  }

  const int r0 = (k0 * G) & ~63;
  const RowStage<D> row_tile(rows, R - 1, wave, lane);
  const RowStage<D> out_tile(outs, R - 1, wave, lane);
  // a tile's rows, and of each wave its log-sums (waves 0 and 2) or sums of dO * O
  auto ask = [&](int t) {
    unsigned char* to = train_lds + t % Ring::DEPTH * Ring::SLOT;
    const int rb = r0 + t * 64;
    row_tile(rb, to);
    out_tile(rb, to + Tile::BYTES);
    dma4(wave & 1 ? delta : lse, (unsigned)min(rb + lane, R - 1) * 4,
         (unsigned)(unsigned long)(lptr_t)(to + 2 * Tile::BYTES + wave * 256));
  };
  const int tiles = (R - r0 + 63) / 64;
  for (int t = 0; t < min(tiles, Ring::DEPTH - 1); ++t) ask(t);
  // these have arrived: what is waited for from here on are the tiles alone
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) asm volatile("" : "+v"(kf[kk]), "+v"(vf[kk]));
  // tiles of which this wave's half sees keys of its own
  const int seen = max(0, (k0 + (wave & 1) * 32) * G - half - 31 - r0 + 63) / 64;
  const int rest = (R - half - r0 + 63) / 64;

  // of a tile: the scores and dO V^T, ahead of the rest by one tile
  f32x16 s, dp, s1, dp1;
  bf16x8 qa[NKK], oa[NKK], oc[2][ND], qc[2][ND], ph[2], pl[2], dh[2], dl[2];
  f32x4 ls[4], de[4];
  float p[8], ds[8];
  auto weigh = [&](int e) {      // element e, of the one before it as well the splits
    const int j = e >> 3, i = e & 7;
    p[i] = fast_exp2(fmaf(s[e], sc2, -ls[e >> 2][e & 3]));
    ds[i] = p[i] * (dp[e] - de[e >> 2][e & 3]);
    if (i & 1) {
#pragma unroll
      for (int c = i - 1; c <= i; ++c) {
        ph[j][c] = (__bf16)p[c];
        dh[j][c] = (__bf16)ds[c];
        pl[j][c] = (__bf16)(p[c] - (float)ph[j][c]);
        dl[j][c] = (__bf16)(ds[c] - (float)dh[j][c]);
      }
    }
  };
  auto add = [&](int j, int d) {
    dv[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ph[j], oc[j][d], dv[d], 0, 0, 0);
    dk[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dh[j], qc[j][d], dk[d], 0, 0, 0);
    dv[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pl[j], oc[j][d], dv[d], 0, 0, 0);
    dk[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dl[j], qc[j][d], dk[d], 0, 0, 0);
  };
  auto turn = [&](int t) {
    if (tiles - t > 2) wait_loads<Ring::LOADS>();
    else wait_loads<0>();
    // everybody's loads of this tile and the next, and everybody is done with the one
    // before, whose place another takes
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + Ring::DEPTH - 1 < tiles) ask(t + Ring::DEPTH - 1);
  };
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    oc[1][d] = qc[1][d] = bf16x8{};
    asm volatile("" : "+v"(oc[1][d]), "+v"(qc[1][d]));
  }
  ph[1] = pl[1] = dh[1] = dl[1] = bf16x8{};
  asm volatile("" : "+v"(ph[1]), "+v"(pl[1]), "+v"(dh[1]), "+v"(dl[1]));
  int t = 0;
  for (; t < min(seen, tiles); ++t) turn(t);
  if (t < rest) {
    turn(t);
    const unsigned char* qt = train_lds + t % Ring::DEPTH * Ring::SLOT;
    s = dp = f32x16{};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(qt, qrow, kk, hi), kf[kk],
                                                  s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          row_frag<D>(qt + Tile::BYTES, qrow, kk, hi), vf[kk], dp, 0, 0, 0);
    }
  }
  while (t < rest) {
    const unsigned char* qt = train_lds + t % Ring::DEPTH * Ring::SLOT;
    const unsigned char* ot = qt + Tile::BYTES;
    const unsigned char* qn = train_lds + (t + 1) % Ring::DEPTH * Ring::SLOT;
    const unsigned char* on = qn + Tile::BYTES;
    const float* stat =
        reinterpret_cast<const float*>(qt + 2 * Tile::BYTES) + (wave & 2) * 64;
    __builtin_amdgcn_sched_barrier(0);
    auto numbers = [&](int j) {
      const int rr = half + (j >> 1) * 16 + hi * 8 + (j & 1) * 4;
      ls[j] = *reinterpret_cast<const f32x4*>(stat + rr);
      de[j] = *reinterpret_cast<const f32x4*>(stat + 64 + rr);
    };
    auto next_rows = [&](int kk) {
      qa[kk] = row_frag<D>(qn, qrow, kk, hi);
      oa[kk] = row_frag<D>(on, qrow, kk, hi);
    };
    // what is left of the tile before; meanwhile this one's numbers and the next's rows
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      add(1, d);
#pragma unroll
      for (int j = d * 4 / ND; j < (d + 1) * 4 / ND; ++j) numbers(j);
      next_rows(d * 2);
      next_rows(d * 2 + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // element j of a lane is row w0 + (j & 8) * 2 + hi * 8 + (j & 7); rows that do not see
    // the key get weights of zero, whatever their log-sum
    const int w0 = r0 + t * 64 + half;
    if (w0 < full || w0 + 31 >= R) {
      const int q0 = w0 + hi * 8;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int q = q0 + (j & 8) * 2 + (j & 7);
        if (q < first || q >= R) {
          s[j] = 0.f;
          ls[j >> 2][j & 3] = __builtin_inff();
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next tile's scores; meanwhile half of this one's weights
    s1 = dp1 = f32x16{};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qa[kk], kf[kk], s1, 0, 0, 0);
      dp1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(oa[kk], vf[kk], dp1, 0, 0, 0);
      if (kk & 1) qc[0][kk >> 1] = col_frag<D>(qt, half, kk >> 1, lane);
      else oc[0][kk >> 1] = col_frag<D>(ot, half, kk >> 1, lane);
#pragma unroll
      for (int e = kk * 8 / NKK; e < (kk + 1) * 8 / NKK; ++e) weigh(e);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the products of this half; meanwhile the other half
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      add(0, d);
      oc[1][d] = col_frag<D>(ot, half + 16, d, lane);
      qc[1][d] = col_frag<D>(qt, half + 16, d, lane);
#pragma unroll
      for (int e = d * 8 / ND; e < (d + 1) * 8 / ND; ++e) weigh(8 + e);
      __builtin_amdgcn_sched_barrier(0);
    }
    s = s1;
    dp = dp1;
    if (++t < rest) turn(t);
  }
  for (; t < tiles; ++t) turn(t);
#pragma unroll
  for (int d = 0; d < ND; ++d) add(1, d);
  __syncthreads();

  // waves 0 and 1 finish the keys, 2 and 3 the values: each pair hands the other what it
  // has of these, through LDS
  auto place = [&](int w) { return reinterpret_cast<float*>(train_lds) + w * 32 * D; };
  auto hand = [&](const f32x16 (&x)[ND]) {
    float* to = place(wave ^ 2);
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int j = 0; j < 16; ++j) to[(n * 16 + j) * 64 + lane] = x[n][j];
  };
  if (wave >> 1) hand(dk);
  else hand(dv);
  __syncthreads();
  const float* other = place(wave);
  // element j of a lane is key j % 4 + j / 4 * 8 + hi * 4
  const int t0 = k0 + (wave & 1) * 32 + hi * 4;
  unsigned short* kx = a.dqkv + ((long)b * a.T + t0) * ldx + (long)(Hq + g) * D + li;
  if (wave >> 1) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int d = (j & 3) + (j >> 2) * 8;
      if (t0 + d >= a.T) continue;
#pragma unroll
      for (int n = 0; n < ND; ++n)
        kx[(long)a.Hkv * D + d * ldx + n * 32] =
            f2bf(other[(n * 16 + j) * 64 + lane] + dv[n][j]);
    }
    return;
  }
  float cs[16][ND / 2], sn[16][ND / 2];   // all at once: one latency
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int t = min(t0 + (j & 3) + (j >> 2) * 8, a.T - 1);
    const long at = (long)(a.start + t) * (D / 2) + li;
#pragma unroll
    for (int n = 0; n < ND / 2; ++n) {
      cs[j][n] = a.cos_t[at + n * 32];
      sn[j][n] = a.sin_t[at + n * 32];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int d = (j & 3) + (j >> 2) * 8;
    if (t0 + d >= a.T) continue;
#pragma unroll
    for (int n = 0; n < ND / 2; ++n) {
      const int m = n + ND / 2;
      const float u = (dk[n][j] + other[(n * 16 + j) * 64 + lane]) * a.scale;
      const float v = (dk[m][j] + other[(m * 16 + j) * 64 + lane]) * a.scale;
      kx[d * ldx + n * 32] = f2bf(u * cs[j][n] + v * sn[j][n]);
      kx[d * ldx + D / 2 + n * 32] = f2bf(v * cs[j][n] - u * sn[j][n]);
    }
  }
}
