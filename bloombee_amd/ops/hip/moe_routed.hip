// Routed experts over (token, choice) slots: slot = token * top + choice.
//
//   act[.]  = glu(W_gate[e] h, W_up[e] h)              one fused launch
//   y[slot] = wts[slot] * (W_down[e] act)              one launch
//
// with glu(g, u) = g sigmoid(slope g) (u + shift) after g = min(g, limit) and
// u = clamp(u, -limit, limit): silu(g) * u for an infinite limit, slope 1 and
// shift 0; or act = relu(W_up[e] h)^2, and the weight may multiply h instead: by then
// it has passed through the linear map, so the first launch's epilogue applies
// it ahead of the activation.
//
// ids[slot] < 0 marks a choice without weights (an identity expert, which the
// residual fold adds by itself): it is skipped everywhere.
//
// First weights (E, planes, F, K): of two planes, row f of plane 0 is the gate of
// activation f, of plane 1 its up projection; a single plane is the up projection
// of relu^2. down (E, N, F). K, F and N are padded to 64.
//
// Kernels take UP, the planes of the first product, 0 for the second, and wts,
// the weights to apply or null.
//
//  * moe_few_kernel — up to 32 tokens: streams each chosen expert's weights
//    once; a workgroup finds its expert's slots by scanning the ids itself, so
//    a decode step needs no sort.
//  * moe_sort_kernel + moe_rows_kernel — longer batches: expert-sorted slots,
//    tiles of 64 to 256 rows (gemm_rows.hip).
//  * moe_simple_kernel — f32 arithmetic on f32 data.

#pragma once
#include "common.h"
#include "gemm_rows.hip"
#include "rows.hip"

static constexpr int MOE_MAX_E = 1024;
static constexpr int MOE_GROUP = 8;

struct GluConst {
  float limit, slope, shift;
  // gate and up are rounded to bf16 ahead of silu(gate) * up, as where the two
  // products and the activation are steps of their own: same bits as those
  bool stepwise;
};

DEVINL float gated(const GluConst& c, float g, float u) {
  if (c.stepwise) {
    g = bf2f(f2bf(g));
    return g / (1.f + fast_expf(-g)) * bf2f(f2bf(u));
  }
  g = fminf(g, c.limit);
  u = fminf(fmaxf(u, -c.limit), c.limit) + c.shift;
  return g * sigmoid_f(c.slope * g) * u;
}

// XCD-aware order: consecutive tiles, which share operand rows, on one XCD.
DEVINL int xcd_order(int id, int n) {
  const int q = n / 8, r = n % 8, x = id % 8, o = id / 8;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + o;
}

// ---------------------------------------------------------------------------
// sort: one workgroup of 1024
// ---------------------------------------------------------------------------

// sorted (S) slots, tiles (max_tiles + 1, 4): expert and MOE_MAX_E * rows (-1 = unused),
// first sorted position, group's first tile and number of tiles of every tile; then the
// number of tiles. An expert's rows are shared out evenly to as few tiles
// of up to BM as there can be (nearly), and its tiles to groups of at most MOE_GROUP.
__global__ __launch_bounds__(1024) void moe_sort_kernel(
    const int* __restrict__ ids, int* __restrict__ sorted, int* __restrict__ tiles,
    int S, int E, int BM, int max_tiles) {
  __shared__ int cnt[MOE_MAX_E], scan[MOE_MAX_E], tscan[MOE_MAX_E];
  const int tid = threadIdx.x;
  cnt[tid] = 0;
  __syncthreads();
  for (int i = tid; i < S; i += 1024) {
    const int e = ids[i];
    if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  // two tiles read an expert's weights from one L2 faster than a high one takes them
  // from memory (225 rows: 800 us for 915)
  const int c = cnt[tid], nt = BM == 256 && c > 192 && c <= 256 ? 2 : (c + BM - 1) / BM;
  scan[tid] = c;
  tscan[tid] = nt;
  __syncthreads();
  for (int d = 1; d < MOE_MAX_E; d <<= 1) {
    const int a = tid >= d ? scan[tid - d] : 0;
    const int b = tid >= d ? tscan[tid - d] : 0;
    __syncthreads();
    scan[tid] += a;
    tscan[tid] += b;
    __syncthreads();
  }
  const int first = scan[tid] - c;
  if (tid < E) {
    const int t0 = tscan[tid] - nt, groups = (nt + MOE_GROUP - 1) / MOE_GROUP;
    const int per = nt ? (nt + groups - 1) / groups : 1;
    for (int k = 0; k < nt; ++k) {
      const int at = t0 + k, g = k / per * per;
      if (at < max_tiles) {
        const int from = (long)c * k / nt, to = (long)c * (k + 1) / nt;
        tiles[4 * at] = tid + MOE_MAX_E * (to - from);
        tiles[4 * at + 1] = first + from;
        tiles[4 * at + 2] = t0 + g;
        tiles[4 * at + 3] = min(per, min(nt, max_tiles - t0) - g);
      }
    }
  }
  if (tid == 0) tiles[4 * max_tiles] = min(tscan[MOE_MAX_E - 1], max_tiles);
  for (int i = tscan[MOE_MAX_E - 1] + tid; i < max_tiles; i += 1024)
    tiles[4 * i] = -1;
  cnt[tid] = first;
  __syncthreads();
  for (int i = tid; i < S; i += 1024) {
    const int e = ids[i];
    if (e >= 0 && e < E) sorted[atomicAdd(&cnt[e], 1)] = i;
  }
}

// ---------------------------------------------------------------------------
// few rows: grid (column tiles, E), at most 32 tokens
// ---------------------------------------------------------------------------

DEVINL float relu_sq(float z) {
  const float r = fmaxf(z, 0.f);
  return r * r;
}

// UP: A row = slot / top (the token), out row = slot, activation (of two planes half of a
// tile's rows of W are gates, half ups).
// else: A row = slot, out row = slot.
//
// A tile of gemm_rows.hip with an expert's 1 to 32 rows. Its weights are read once, by whole
// lines past the caches, and bound it. us for both products by half lines of 16 rows a wave
// and here: eight experts, 4096 x 14336, two a token: 1 token 220, 126; 16 tokens 490, 381
// (6.6 TB/s); 64 experts, 2048 x 1024, eight a token: 55, 34; 141, 116. K % 64 == 0
template <typename T, int UP>
__global__ __launch_bounds__(T::THREADS, T::MINW) void moe_few_kernel(
    const unsigned short* __restrict__ A, const unsigned short* __restrict__ W,
    const int* __restrict__ ids, const float* __restrict__ wts,
    unsigned short* __restrict__ C, int S, int top, int N, int K, int lda,
    int ldc, GluConst glu) {
  static_assert(T::WK == 1 && (UP < 2 || T::NI % 2 == 0), "pairs");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  __shared__ int slots[32];
  __shared__ int n_slots;
  constexpr int HALF = T::NI * 8;                    // a wave's gates, then its ups
  const int e = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x & (WAVE - 1), li = lane & 15;
  if (wave == 0) {
    int n = 0;
    for (int b = 0; b < S; b += WAVE) {
      const bool mine = b + lane < S && ids[b + lane] == e;
      const unsigned long long m = __builtin_amdgcn_ballot_w64(mine);
      const int at = n + __popcll(m & ((1ull << lane) - 1));
      if (mine && at < 32) slots[at] = b + lane;
      n += __popcll(m);
    }
    if (lane == 0) n_slots = min(n, 32);  // choices of a token are distinct
  }
  __syncthreads();
  const int cnt = n_slots;
  if (cnt == 0) return;
  const int n0 = xcd_order(blockIdx.x, gridDim.x) * (UP == 2 ? T::BN / 2 : T::BN);

  unsigned ofs[T::LPW];
#pragma unroll
  for (int j = 0; j < T::LPW; ++j) {
    const int r = T::load_row(j, wave, lane);
    unsigned row;
    if (j < T::AJ) {
      const int sl = slots[min(r, cnt - 1)];
      row = (unsigned)(UP ? sl / top : sl) * (unsigned)lda;
    } else {
      row = (unsigned)min(UP == 2 ? r / (2 * HALF) * HALF + r % HALF : r, N - 1 - n0) *
            (unsigned)K;
    }
    ofs[j] = row * 2 + T::load_byte(j, wave, lane);
  }
  typename T::Acc acc;
  T::template run<false, true>(
      ofs, A, W + ((long)e * (UP ? UP : 1) * N + n0) * K, K / T::BK, lds, acc,
      [&](int j) {
        // the eight rows of a load are of one plane
        return UP == 2 ? (long)(T::load_row(j, wave, 0) / HALF % 2) * N * K : 0L;
      }, T::BK, 0.f, rows_begin(K / T::BK));

  const int r0 = T::row0(), c0 = n0 + (UP == 2 ? T::col0() / 2 : T::col0());
  constexpr int STRIPS = UP == 2 ? T::NI / 2 : T::NI;
#pragma unroll
  for (int m = 0; m < T::MI; ++m) {
    const int r = r0 + m * 16 + li;
    const float w = wts && r < cnt ? wts[slots[r]] : 1.f;
    T::template out16<STRIPS>(lds, [&](int n) {
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = acc[m][n][j] * w;
        if constexpr (UP == 2) v[j] = gated(glu, v[j], acc[m][n + STRIPS][j] * w);
        if constexpr (UP == 1) v[j] = relu_sq(v[j]);
      }
      return pack4(v);
    }, [&](int i, int c, auto v) {
      const int at = r0 + m * 16 + i;
      if (at < cnt && c0 + c < N)
        *reinterpret_cast<decltype(v)*>(C + (long)slots[at] * ldc + c0 + c) = v;
    });
  }
}

// ---------------------------------------------------------------------------
// tile: grid of column tiles * row tiles; K % 64 == 0, N % 8 == 0
// ---------------------------------------------------------------------------

// UP: A row = sorted slot / top, out row = sorted position, N = activations
//     (two planes: half of a tile's rows of W are gates, half ups).
// else: A row = sorted position, out row = slot.
//
// A tile of gemm_rows.hip a workgroup: T::BM rows of one expert.
//
// Every expert's weights come from memory once at best; what bounds it is how often
// they come again. Hence the order of the tiles below: an expert's row tiles take one
// column after the other together and find W in their XCD's L2. Tiles of several
// experts in a group of eight took 1430 us for both products at 1400 tokens, two of
// eight experts, 4096 x 14336, in this order 1254 on tiles of 128 x 256 with 32 of K a
// step, all rows a wave, and 1105 on these (160 tokens 637, 495; 700: 934, 684; 4000:
// 3255, 2696).
struct MoeArgs {
  const unsigned short* A;   // rows of lda
  const unsigned short* W;   // (E, UP or 1, N, K)
  const int* sorted;
  const int* tiles;
  const float* wts;          // or null
  unsigned short* C;         // rows of ldc
  int max_tiles, top, N, K, lda, ldc;
  GluConst glu;
  bool large;                // weights that no cache holds until the next step
};

struct MoeTile {
  int e, p0, cnt, nt;        // expert, first sorted position, rows, column tile
  bool alone;                // read its weights once: no other tile does
};

// The workgroup's tile; false: none.
DEVINL bool moe_tile(const MoeArgs& a, int ntn, MoeTile& t) {
  const int total = a.tiles[4 * a.max_tiles] * ntn;
  if ((int)blockIdx.x >= total) return false;
  const int id = xcd_order(blockIdx.x, total);
  const int* group = a.tiles + 4 * (id / ntn);
  const int first = group[2], gsz = group[3];
  const int rt = first + (id - first * ntn) % gsz;
  t.nt = (id - first * ntn) / gsz;
  t.alone = a.large && gsz == 1;
  t.e = a.tiles[4 * rt] % MOE_MAX_E;
  t.cnt = a.tiles[4 * rt] / MOE_MAX_E;
  t.p0 = a.tiles[4 * rt + 1];
  return true;
}

// Column tiles of BN.
template <int UP>
__host__ DEVINL int moe_columns(int N, int BN) {
  const int per = UP == 2 ? BN / 2 : BN;
  return (N + per - 1) / per;
}

template <typename T, int UP, bool ONCE = false>
DEVINL void moe_rows(const MoeArgs& a, const MoeTile& t, unsigned char* lds) {
  static_assert(T::WK == 1 && (UP < 2 || T::NI % 2 == 0), "pairs");
  const int p0 = t.p0, cnt = t.cnt, N = a.N, K = a.K;
  constexpr int HALF = T::NI * 8;                    // a wave's gates, then its ups
  const int n0 = t.nt * (UP == 2 ? T::BN / 2 : T::BN);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x & (WAVE - 1), li = lane & 15;

  unsigned ofs[T::LPW];
#pragma unroll
  for (int j = 0; j < T::LPW; ++j) {
    const int r = T::load_row(j, wave, lane);
    unsigned row;
    if (j < T::AJ) {
      const int i = min(r, cnt - 1);
      row = (unsigned)(UP ? a.sorted[p0 + i] / a.top : i) * (unsigned)a.lda;
    } else {
      row = (unsigned)min(UP == 2 ? r / (2 * HALF) * HALF + r % HALF : r, N - 1 - n0) *
            (unsigned)K;
    }
    ofs[j] = row * 2 + T::load_byte(j, wave, lane);
  }
  typename T::Acc acc;
  T::template run<false, ONCE>(
      ofs, UP ? a.A : a.A + (long)p0 * a.lda,
      a.W + ((long)t.e * (UP ? UP : 1) * N + n0) * K, K / T::BK, lds, acc,
      [&](int j) {
        // the eight rows of a load are of one plane
        return UP == 2 ? (long)(T::load_row(j, wave, 0) / HALF % 2) * N * K : 0L;
      }, T::BK, 0.f, ONCE ? rows_begin(K / T::BK) : 0);

  const int r0 = T::row0(), c0 = n0 + (UP == 2 ? T::col0() / 2 : T::col0());
  constexpr int S = UP == 2 ? T::NI / 2 : T::NI;
#pragma unroll
  for (int m = 0; m < T::MI; ++m) {
    const int r = r0 + m * 16 + li;
    const float w = a.wts && r < cnt ? a.wts[a.sorted[p0 + r]] : 1.f;
    T::template out16<S>(lds, [&](int n) {
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = acc[m][n][j] * w;
        if constexpr (UP == 2) v[j] = gated(a.glu, v[j], acc[m][n + S][j] * w);
        if constexpr (UP == 1) v[j] = relu_sq(v[j]);
      }
      return pack4(v);
    }, [&](int i, int c, auto v) {
      const int at = r0 + m * 16 + i;
      if (at >= cnt || c0 + c >= N) return;
      const long row = UP ? p0 + at : a.sorted[p0 + at];
      *reinterpret_cast<decltype(v)*>(a.C + row * a.ldc + c0 + c) = v;
    });
  }
}

// Where an expert has one tile, as most have, its weights pass the caches and each XCD
// begins K elsewhere: eight experts, 4096 x 14336, 64 tokens of two, both products 498 us
// without, 445; 64 experts, 2048 x 1024, 128 tokens of eight 171, 133. Where a cache holds
// all experts it is not worth its code (8 of 512 x 256, 33 tokens: 15.2, 16.8).
template <typename T, int UP>
__global__ __launch_bounds__(T::THREADS, T::MINW) void moe_rows_kernel(MoeArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  MoeTile t;
  if (!moe_tile(a, moe_columns<UP>(a.N, T::BN), t)) return;
  if (t.alone) moe_rows<T, UP, true>(a, t, lds);
  else moe_rows<T, UP>(a, t, lds);
}

// Tiles of up to 256 rows on the height that fits, since experts' counts differ. They are
// 256 columns wide, but where those leave CUs idle in their last round half as wide ones
// end sooner: a stage of 64 columns takes 1.14 us there, 0.66 here (19 tiles of 4096
// columns: two rounds for three).
template <int UP>
__global__ __launch_bounds__(512, 2) void moe_rows_any_kernel(MoeArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tiles = a.tiles[4 * a.max_tiles];
  const int wide = moe_columns<UP>(a.N, 256), half = moe_columns<UP>(a.N, 128);
  MoeTile t;
  if ((tiles * wide + 255) / 256 * 12 <= (tiles * half + 255) / 256 * 7) {
    if (!moe_tile(a, wide, t)) return;
    if (t.cnt > 192) moe_rows<RowsTile<256, 256, 2, 4, 1, 2, 2, false, 2>, UP>(a, t, lds);
    else if (t.cnt > 128) moe_rows<RowsTile<192, 256, 2, 4, 1, 2, 2, false, 2>, UP>(a, t, lds);
    else moe_rows<RowsTile<128, 256, 2, 4, 1, 3, 2>, UP>(a, t, lds);
  } else {
    if (!moe_tile(a, half, t)) return;
    if (t.cnt > 192) moe_rows<RowsTile<256, 128, 4, 2, 1, 3, 2>, UP>(a, t, lds);
    else if (t.cnt > 128) moe_rows<RowsTile<192, 128, 4, 2, 1, 3, 2>, UP>(a, t, lds);
    else moe_rows<RowsTile<128, 128, 4, 2, 1, 4, 2>, UP>(a, t, lds);
  }
}

// ---------------------------------------------------------------------------
// plain f32: 64 x 64 tiles, same row tiles (BM = 64)
// ---------------------------------------------------------------------------

template <int UP>
__global__ __launch_bounds__(256) void moe_simple_kernel(
    const float* __restrict__ A, const float* __restrict__ W,
    const int* __restrict__ sorted,
    const int* __restrict__ tiles, const float* __restrict__ wts,
    float* __restrict__ C, int top, int N, int K, int lda, int ldc,
    GluConst glu) {
  constexpr int NW = UP ? UP : 1, BK = 16;
  __shared__ float al[BK][64 + 4], wl[NW][BK][64 + 4];
  if (tiles[4 * blockIdx.y] < 0) return;
  const int e = tiles[4 * blockIdx.y] % MOE_MAX_E;
  const int cnt = tiles[4 * blockIdx.y] / MOE_MAX_E;
  const int p0 = tiles[4 * blockIdx.y + 1];
  const int n0 = blockIdx.x * 64;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  float acc[NW][4][4] = {};
  for (int k = 0; k < K; k += BK) {
    for (int i = threadIdx.x; i < 64 * BK; i += 256) {
      const int r = i / BK, c = i % BK;
      const int p = p0 + min(r, cnt - 1);
      al[c][r] = A[(long)(UP ? sorted[p] / top : p) * lda + k + c];
      for (int w = 0; w < NW; ++w)
        wl[w][c][r] = W[(((long)e * NW + w) * N + n0 + r) * K + k + c];
    }
    __syncthreads();
    for (int c = 0; c < BK; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int w = 0; w < NW; ++w)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[w][i][j] += al[c][ty * 4 + i] * wl[w][c][tx * 4 + j];
    __syncthreads();
  }
  for (int i = 0; i < 4; ++i) {
    const int r = ty * 4 + i;
    if (r >= cnt) continue;
    const int sl = sorted[p0 + r];
    const float w = wts ? wts[sl] : 1.f;
    for (int j = 0; j < 4; ++j) {
      float v = acc[0][i][j] * w;
      if constexpr (UP == 2) v = gated(glu, v, acc[NW - 1][i][j] * w);
      if constexpr (UP == 1) v = relu_sq(v);
      C[(long)(UP ? p0 + r : sl) * ldc + n0 + tx * 4 + j] = v;
    }
  }
}
