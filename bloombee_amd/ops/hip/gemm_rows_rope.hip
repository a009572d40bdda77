// [q | k | v] = A @ W^T of a fused projection on a tile of gemm_rows.hip, with q turned in
// C and k, v in their page slots, for the rows that one tile takes (rope_kv_store of
// gemm_stream.hip, four columns at a time).
//
// W by whole lines past the caches is what bounds it, and below some 8000 columns the few
// workgroups that are left. us in a graph, W from memory, with gemm_stream.hip, which takes W
// by half lines and all of A again for every 16 rows of it, and here: 6144 x 4096: 1 row
// 13.8, 13.4; 8 rows 15.2, 13.5; 32 rows 20.2, 16.3. 24576 x 8192: 78.6, 72.0; 106, 73.5.

#pragma once
#include "gemm_rows.hip"
#include "gemm_stream.hip"

typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef short4v short4_any __attribute__((aligned(2)));

// A strip of 16 rows of the tile is eight columns of a head and the eight half a head on,
// so that every lane has both of a pair (as gates and ups in gemm_rows_glu_kernel). grid:
// tiles of BN / 2 of N / 2 columns; D / 2 % 8 == 0.
template <typename T>
__global__ __launch_bounds__(T::THREADS, T::MINW) void gemm_rows_rope_kernel(StreamArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & (WAVE - 1), li = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int half = a.D / 2, columns = a.N / 2;
  const int n = gridDim.x, q = n / 8, r = n % 8, x = blockIdx.x % 8;
  const int tile = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + blockIdx.x / 8;
  const int n0 = tile * (T::BN / 2);
  // the row of W that column c of the first halves of all heads is
  auto row_of = [&](int c) { return c / half * a.D + c % half; };
  const int base = row_of(n0);

  unsigned ofs[T::LPW];
#pragma unroll
  for (int j = 0; j < T::LPW; ++j) {
    const int t = T::load_row(j, wave, lane);
    const int row = j < T::AJ ? min(t, a.M - 1)
                              : row_of(min(n0 + t / 16 * 8 + t % 8, columns - 1)) - base;
    ofs[j] = (unsigned)row * (unsigned)(a.K * 2) + T::load_byte(j, wave, lane);
  }
  // asked for ahead of it all: each lane's rows' sequences begin where
  int b[T::MI], start[T::MI];
#pragma unroll
  for (int m = 0; m < T::MI; ++m) {
    b[m] = min(T::row0() + m * 16 + li, a.M - 1) / a.T;
    start[m] = a.start[b[m]];
  }
  typename T::Acc acc;
  T::template run<true, true>(
      ofs, a.A, a.W + (long)base * a.K, a.K / T::BK, lds, acc,
      [&](int j) { return (long)(T::load_row(j, wave, 0) / 8 % 2) * half * a.K; }, T::BK,
      a.eps, rows_begin(a.K / T::BK));

  constexpr int NO = T::COLS / 16, S = (NO + 1) / 2;
  const int c0 = n0 + T::col0() / 2;
#pragma unroll
  for (int m = 0; m < T::MI; ++m) {
    const int row = T::row0() + m * 16 + li;
    const bool there = row < a.M;
    const int at = start[m] + min(row, a.M - 1) - b[m] * a.T, slot = at % a.P;
    const int p = min(max(a.pos ? a.pos[min(row, a.M - 1)] : at, 0), a.max_pos - 1);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      f32x4 v, u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = acc[m][2 * s][e];
        const float y = 2 * s + 1 < NO ? acc[m][2 * s + 1 < NO ? 2 * s + 1 : 0][e] : 0.f;
        const auto w = __builtin_amdgcn_permlane32_swap(
            __builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y), false, false);
        v[e] = __builtin_bit_cast(float, (unsigned)w[0]);
        u[e] = __builtin_bit_cast(float, (unsigned)w[1]);
      }
      const int local = s * 16 + hi * 4, c = c0 + local;
      if (!there || local >= NO * 8 || c >= columns) continue;
      const int h = c / half, d = c % half;
      if (h >= a.Hq + a.Hkv) {
        const long page = a.table[b[m] * a.maxp + at / a.P];
        unsigned short* vp =
            a.v_pages + ((page * a.Hkv + h - a.Hq - a.Hkv) * a.D + d) * a.P + slot;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vp[(long)e * a.P] = f2bf(v[e]);
          vp[(long)(half + e) * a.P] = f2bf(u[e]);
        }
        continue;
      }
      const f32x4 cs = *reinterpret_cast<const f32x4_any*>(a.cos_t + (long)p * half + d);
      const f32x4 sn = *reinterpret_cast<const f32x4_any*>(a.sin_t + (long)p * half + d);
      unsigned short* dst = a.C + (long)row * a.N + h * a.D + d;
      if (h >= a.Hq) {
        const long page = a.table[b[m] * a.maxp + at / a.P];
        dst = a.k_pages + ((page * a.Hkv + h - a.Hq) * a.P + slot) * a.D + d;
      }
      *reinterpret_cast<short4_any*>(dst) = pack4(v * cs - u * sn);
      *reinterpret_cast<short4_any*>(dst + half) = pack4(u * cs + v * sn);
    }
  }
}

// The fold of a split product whose row m has q, k and v of token m % T of sequence m / T: a
// thread turns eight columns of both halves of a head. grid: M * N / 16 / 256; D a power
// of two of 32 to 256. us of a product of 6144 x 4096, 32, 8 and 8
// heads of 128, with a fold and rope_kv_rows_kernel, and so: 33 rows in 5 splits 18.4, 17.5;
// 97 24.6, 23.0; 250 in 2 36.3, 33.7; 10240 x 8192, 250 rows in 3 66.5, 59.1.
__global__ __launch_bounds__(256) void gemm_rows_fold_rope_kernel(RowsArgs a, StreamArgs r) {
  const long item = (long)blockIdx.x * 256 + threadIdx.x;
  const int per = a.N / 16;                  // of a row
  const int m = (int)(item / per), half = r.D / 2;
  if (m >= a.M) return;
  const int c = (int)(item - (long)m * per) * 8, h = c / half, d = c % half;
  const int b = m / r.T, at = r.start[b] + m % r.T;
  const int p = min(max(r.pos ? r.pos[m] : at, 0), r.max_pos - 1);
  const long page = h < r.Hq ? 0 : r.table[(long)b * r.maxp + at / r.P];
  f32x4 cs[2], sn[2], v[2], u[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    cs[i] = *reinterpret_cast<const f32x4_any*>(r.cos_t + (long)p * half + d + i * 4);
    sn[i] = *reinterpret_cast<const f32x4_any*>(r.sin_t + (long)p * half + d + i * 4);
    v[i] = u[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  const long n = (long)a.M * a.N;
  const float* src = a.part + (long)m * a.N + h * r.D + d;
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      v[i] += *reinterpret_cast<const f32x4*>(src + s * n + i * 4);
      u[i] += *reinterpret_cast<const f32x4*>(src + s * n + half + i * 4);
    }
  if (h >= r.Hq + r.Hkv) {
    unsigned short* vp =
        r.v_pages + ((page * r.Hkv + h - r.Hq - r.Hkv) * r.D + d) * r.P + at % r.P;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      vp[(long)e * r.P] = f2bf(v[e / 4][e % 4]);
      vp[(long)(half + e) * r.P] = f2bf(u[e / 4][e % 4]);
    }
    return;
  }
  unsigned short* dst = h < r.Hq
      ? a.C + (long)m * a.N + h * r.D + d
      : r.k_pages + ((page * r.Hkv + h - r.Hq) * r.P + at % r.P) * r.D + d;
  float x[8], y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x[e] = v[e / 4][e % 4] * cs[e / 4][e % 4] - u[e / 4][e % 4] * sn[e / 4][e % 4];
    y[e] = u[e / 4][e % 4] * cs[e / 4][e % 4] + v[e / 4][e % 4] * sn[e / 4][e % 4];
  }
  store_bf16x8(dst, x);
  store_bf16x8(dst + half, y);
}
