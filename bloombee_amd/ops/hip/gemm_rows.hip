// A tile of rows times a tile of W's rows, C(BM,BN) = A(BM,K) @ W(BN,K)^T, for products
// of some dozen rows to some thousand: the workgroups of moe_routed.hip.
//
// Stages of 64 columns of K (RB bytes a row, 16 B piece c of row r at c ^ (r & 7): what
// the lanes read together covers all banks) come into LDS by DMA, ST of them on their
// way or in use. Rows of 128 B, since half lines cost a whole one (27 B a clock and CU
// of L2's 50 with 64 B). A wave holds BM / WM rows of BN / WN columns, the larger the
// fewer bytes of LDS a product reads: 128 x 128 with one wave a SIMD and 256 sums a lane
// in accumulation registers. While it multiplies one half of a stage, it reads the other
// half's fragments, or the next stage's behind the one barrier a stage has, and asks for
// the stage that takes the place of the one just read.
//
// Measured, 4096 columns, cold W. Large sizes want 256 x 256, on which power and the way
// from L2 bound it together (a stage 1.4 us: products alone 1.1 at the clock that power
// leaves them, DMA alone 1.2): four waves and two buffers 1326 TF at 2800 rows of 28672
// columns, eight waves of half the columns, with a third buffer for W in what LDS is left,
// 1450 to 1510 from 4096 rows on (a third one for A: 1440; the library's 1525 to 1640).
// Where one round of workgroups streams W, three stages of smaller tiles hide more of
// memory: 333 rows 73 us with 192 x 224, 87 with 192 x 256 and two stages, 94 with
// 192 x 128 and four (W alone takes 50 in step, 37 with its K begun apart, rows_begin: no
// more than 1 us of it is left here, nor does K begun apart by column tile for the L2's
// channels gain anything, 1 to 5 us slower).
// What it writes goes through LDS by whole lines (8 B a lane straight from the sums: 78 us
// for 73, 513 for 496).
// Tried and left: 32 columns a stage with five stages, L2 touched a stage or two ahead,
// all of a stage's DMA at the phase's start (1347 us for 1320, 8192 rows), the compiler's
// own order of reads and products in a phase (1430), priorities (1340).

#pragma once
#include "common.h"

// A product whose sums stay where they are in the accumulation registers: with more
// than 256 registers a wave the compiler moves them around between products (four
// moves each). It knows nothing of the product's latency: settle() goes ahead of what
// reads the sums.
// Accumulation registers hold 64 such sums a lane; IN_VECTOR: one beyond them.
template <bool IN_VECTOR = false>
DEVINL void mfma_acc(f32x4& c, bf16x8 x, bf16x8 y) {
  if constexpr (IN_VECTOR)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(x), "v"(y));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
}

DEVINL void settle() { asm volatile("s_nop 15\n\ts_nop 7" ::: "memory"); }

DEVINL short4v pack4(f32x4 v) {
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  return __builtin_bit_cast(short4v, __builtin_convertvector(v, bf16x4));
}

DEVINL f32x4 pick(bool c, f32x4 x, f32x4 y) {
  f32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = c ? x[e] : y[e];
  return r;
}

// WM x WN waves, times WK groups that take 64 columns each of a stage; ST stages; MINW
// waves a SIMD. TURNED: sums run over rows of W instead, C(BM,BN) = A(BM,K) @ W(K,BN):
// 64 rows of it are a stage, by 128 columns, 16 B piece c of row r at c ^ turn(r), and
// fragments come by transposing reads. MORE: one more buffer for A (1) or for W (2), whose
// loads then come behind the other's.
template <int BM_, int BN_, int WM_, int WN_, int WK_, int ST_, int MINW_,
          bool TURNED_ = false, int MORE_ = 0>
struct RowsTile {
  static constexpr bool TURNED = TURNED_;
  static constexpr int MORE = MORE_;
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_, ST = ST_;
  static constexpr int MINW = MINW_;
  static constexpr int NW = WM * WN * WK, THREADS = NW * 64;
  static constexpr int MI = BM / WM / 16, NI = BN / WN / 16;
  static constexpr int BK = 64 * WK, RB = BK * 2, RPC = 1024 / RB;
  static constexpr int STAGE = (BM + BN) * RB;
  static constexpr int AJ = BM * RB / 1024 / NW, LPW = AJ + BN * RB / 1024 / NW;
  static constexpr int EXCHANGE = WK > 1 ? BM * BN * 4 : 0;
  static constexpr int OUT_RS = NI * 64 + 16;            // f32 row of the way out
  static constexpr int OUT = NW * 16 * OUT_RS;
  // buffers of A and of W; loads of the operand that has one more
  static constexpr int SA = ST + (MORE == 1), SW = ST + (MORE == 2);
  static constexpr int EX = MORE == 1 ? AJ : MORE == 2 ? LPW - AJ : 0;
  static constexpr int WBASE = SA * BM * RB, STAGES = WBASE + SW * BN * RB;
  static constexpr int LDS0 = STAGES > EXCHANGE ? STAGES : EXCHANGE;
  static constexpr int LDS = LDS0 > OUT ? LDS0 : OUT;
  static_assert(AJ * NW * 1024 == BM * RB &&
                (LPW - AJ) * NW * 1024 == BN * RB && LDS <= 160 * 1024, "chunks");

  typedef f32x4 Acc[MI][NI];

  static DEVINL int turn(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

  // Row of the tile (of A for j < AJ, else of W) that load j of the thread is for, and
  // the byte in the row.
  static DEVINL int load_row(int j, int wave, int lane) {
    const int chunk = (j < AJ ? j : j - AJ) * NW + wave;
    if (TURNED && j >= AJ) return chunk % 16 * 4 + lane / 16;
    return chunk * RPC + lane / (RB / 16);
  }
  static DEVINL unsigned load_byte(int j, int wave, int lane) {
    const int r = load_row(j, wave, lane);
    if (TURNED && j >= AJ)
      return ((j - AJ) * NW + wave) / 16 * 256 + ((lane % 16) ^ turn(r)) * 16;
    return ((lane % (RB / 16)) ^ (r & 7)) * 16;
  }

  // Sums of `steps` stages. ofs: bytes from ap (j < AJ) or wp, which move on by a
  // stage's columns (wp by w_step); beyond(j): what the rows of a load lie behind wp, the
  // wave's. NORM: rows of A are divided by their root mean square, columns of K; a row's
  // sum of squares is the diagonal of A A^T, made from the fragments at hand. ONCE: nobody
  // else reads these rows of W, and stage `begin` comes first, number 0 behind the last.
  template <bool NORM = false, bool ONCE = false, typename B>
  static DEVINL void run(const unsigned (&ofs)[LPW], const unsigned short* ap,
                         const unsigned short* wp, int steps, unsigned char* lds,
                         Acc& acc, B beyond, long w_step = BK, float eps = 0.f,
                         int begin = 0) {
    const int lane = threadIdx.x & (WAVE - 1), li = lane & 15, hi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wk = wave % WK, wn = wave / WK % WN, wm = wave / (WK * WN);
    const unsigned base = (unsigned)(unsigned long)(lptr_t)lds;
#pragma unroll
    for (int m = 0; m < MI; ++m)
#pragma unroll
      for (int n = 0; n < NI; ++n) acc[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (steps <= 0) return;

    int a_left = steps - begin, w_left = a_left;
    if constexpr (ONCE) {
      ap += (long)begin * BK;
      wp += begin * w_step;
    }
    auto next_a = [&]() {
      ap += BK;
      if (ONCE && --a_left == 0) {
        ap -= (long)steps * BK;
        a_left = steps;
      }
    };
    auto next_w = [&]() {
      wp += w_step;
      if (ONCE && --w_left == 0) {
        wp -= steps * w_step;
        w_left = steps;
      }
    };
    auto load = [&](int j, int slot_a, int slot_w) {
      if (j < AJ)
        dma16(ap, ofs[j], base + slot_a * (BM * RB) + (j * NW + wave) * 1024);
      else
        dma16<ONCE>(wp + beyond(j), ofs[j],
              base + WBASE + slot_w * (BN * RB) + ((j - AJ) * NW + wave) * 1024);
    };
    // load i of an iteration: of the operand with fewer buffers first
    auto turn_of = [](int i) { return MORE == 1 ? (i + AJ) % LPW : i; };
    // a lane's pieces of its rows
    unsigned fa[2], fw[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const unsigned piece = ((wk * 8 + s * 4 + hi) ^ (li & 7)) * 16;
      fa[s] = (wm * MI * 16 + li) * RB + piece;
      fw[s] = WBASE + (wn * NI * 16 + li) * RB + piece;
    }
    unsigned turned[NI][2];
    if constexpr (TURNED) {
      static_assert(WK == 1 && BN % 128 == 0, "stages by 128 columns");
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int c = (wn * NI + i) * 16, r = hi * 8 + q * 4 + (li >> 2);
          const int piece = c % 128 / 8 + ((li >> 1) & 1);
          turned[i][q] = WBASE + c / 128 * 16384 + r * 256 + ((piece ^ turn(r)) << 4) +
                         (li & 1) * 8;
        }
    }
    f32x4 sq[MI];
#pragma unroll
    for (int m = 0; m < MI; ++m) sq[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 af[2][MI], wf[2][NI];
    auto frag = [&](int i, int s, int slot_a, int slot_w) {
      const unsigned char* stage = lds + (i < NI ? slot_w * (BN * RB) : slot_a * (BM * RB));
      if (TURNED && i < NI) {
        // column li of rows s * 32 + hi * 8 .. +7
        typedef __attribute__((address_space(3))) short4v lds4;
        short8 v;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const short4v c = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds4*)(stage + turned[i][q] + s * 8192));
#pragma unroll
          for (int e = 0; e < 4; ++e) v[q * 4 + e] = c[e];
        }
        wf[s][i] = as_bf16x8(v);
      } else if (i < NI)
        wf[s][i] = as_bf16x8(
            *reinterpret_cast<const short8*>(stage + fw[s] + i * 16 * RB));
      else
        af[s][i - NI] = as_bf16x8(
            *reinterpret_cast<const short8*>(stage + fa[s] + (i - NI) * 16 * RB));
    };
    // products of half s of a stage, with the other set's reads from slots a, w and, with
    // loads, those to slots to_a, to_w in between
    auto phase = [&](int s, int a, int w, auto loads, int to_a, int to_w) {
      constexpr int FR = MI + NI, P = MI * NI;
      int p = 0;
#pragma unroll
      for (int i = 0; i < FR; ++i) {
        frag(i, s ^ 1, a, w);
        if constexpr (decltype(loads)::value) {
#pragma unroll
          for (int j = i * LPW / FR; j < (i + 1) * LPW / FR; ++j)
            load(turn_of(j), to_a, to_w);
        }
#pragma unroll
        for (; p < (i + 1) * P / FR; ++p) {
          if constexpr (MINW == 1) {
            if (P > 64 && p >= 58)
              mfma_acc<true>(acc[p % MI][p / MI], wf[s][p / MI], af[s][p % MI]);
            else
              mfma_acc(acc[p % MI][p / MI], wf[s][p / MI], af[s][p % MI]);
          }
          else
            acc[p % MI][p / MI] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wf[s][p / MI], af[s][p % MI], acc[p % MI][p / MI], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (NORM)
#pragma unroll
        for (int m = 0; m < MI; ++m)
          sq[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[s][m], af[s][m], sq[m], 0, 0,
                                                          0);
    };
    auto barrier = [&]() {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    // until all but n stages have landed
    auto wait = [&](int n) {
      static_assert(ST <= 6 && (ST - 1) * LPW < 64, "stages");
      if (ST > 5 && n >= 5) wait_loads<(ST > 5 ? 5 : 0) * LPW>();
      else if (ST > 4 && n >= 4) wait_loads<(ST > 4 ? 4 : 0) * LPW>();
      else if (n >= 3) wait_loads<3 * LPW>();
      else if (n == 2) wait_loads<2 * LPW>();
      else if (n == 1) wait_loads<LPW>();
      else wait_loads<0>();
    };

    // ap and wp stand behind what was asked for, the operand with one more buffer ahead
#pragma unroll
    for (int s = 0; s < ST; ++s)
      if (s < steps) {
#pragma unroll
        for (int j = 0; j < LPW; ++j) load(j, s, s);
        next_a();
        next_w();
      }
    if (MORE && ST < steps) {
#pragma unroll
      for (int j = 0; j < LPW; ++j)
        if ((j < AJ) == (MORE == 1)) load(j, ST, ST);
      if (MORE == 1) next_a();
      else next_w();
      wait_loads<(ST - 1) * LPW + EX>();
    } else {
      wait(min(ST, steps) - 1);
    }
    barrier();
#pragma unroll
    for (int i = 0; i < MI + NI; ++i) frag(i, 0, 0, 0);
    int a = 0, w = 0, t = 0;
    for (; t + ST + (MORE > 0) < steps; ++t) {
      phase(0, a, w, std::false_type{}, 0, 0);
      wait_loads<(ST - 2) * LPW + EX>();
      barrier();
      const int na = a + 1 == SA ? 0 : a + 1, nw = w + 1 == SW ? 0 : w + 1;
      phase(1, na, nw, std::true_type{}, a, w);
      next_a();
      next_w();
      a = na;
      w = nw;
      if (MINW == 1) settle();
    }
    for (; t < steps; ++t) {
      phase(0, a, w, std::false_type{}, 0, 0);
      if (MORE) wait_loads<0>();
      else wait(steps - 2 - t);
      barrier();
      if (MORE && t + ST < steps) {
        // the last stage of the operand with fewer buffers
#pragma unroll
        for (int j = 0; j < LPW; ++j)
          if ((j < AJ) != (MORE == 1)) load(j, a, w);
      }
      a = a + 1 == SA ? 0 : a + 1;
      w = w + 1 == SW ? 0 : w + 1;
      // behind the last stage these reads bring what nothing uses
      phase(1, a, w, std::false_type{}, 0, 0);
      if (MINW == 1) settle();
    }

    if constexpr (WK > 1) {
      // a k group keeps half of the columns and hands the others' sums over
      static_assert(WK == 2 && NI % 2 == 0, "halves");
      constexpr int H = NI / 2;
      __syncthreads();
      f32x4* ex = reinterpret_cast<f32x4*>(lds) + (wm * WN + wn) * (MI * NI * 64);
#pragma unroll
      for (int m = 0; m < MI; ++m)
#pragma unroll
        for (int n = 0; n < H; ++n)
          ex[((wk ^ 1) * MI * H + m * H + n) * 64 + lane] =
              pick(wk, acc[m][n], acc[m][n + H]);
      __syncthreads();
#pragma unroll
      for (int m = 0; m < MI; ++m)
#pragma unroll
        for (int n = 0; n < H; ++n)
          acc[m][n] = pick(wk, acc[m][n + H], acc[m][n]) +
                      ex[(wk * MI * H + m * H + n) * 64 + lane];
    }
    if constexpr (NORM) {
      static_assert(MINW > 1 && WK * BM * 4 + EXCHANGE <= STAGES, "squares");
      if (WK == 1) __syncthreads();
      float* squares = reinterpret_cast<float*>(lds + EXCHANGE);
#pragma unroll
      for (int m = 0; m < MI; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (hi * 4 + e == li) squares[wk * BM + (wm * MI + m) * 16 + li] = sq[m][e];
      __syncthreads();
#pragma unroll
      for (int m = 0; m < MI; ++m) {
        float all = 0.f;
#pragma unroll
        for (int g = 0; g < WK; ++g) all += squares[g * BM + (wm * MI + m) * 16 + li];
        const float r = rsqrtf(all / (float)(steps * BK) + eps);
#pragma unroll
        for (int n = 0; n < NI / WK; ++n) acc[m][n] *= r;
      }
    }
    __syncthreads();   // the way out takes the place of the stages
  }

  // The wave's columns of the tile after run(): COLS of them from col0().
  static constexpr int COLS = NI * 16 / WK;
  static DEVINL int col0() {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    return wave / WK % WN * NI * 16 + wave % WK * COLS;
  }
  static DEVINL int row0() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) / (WK * WN) * MI * 16;
  }

  // Sixteen rows at a time, of STRIPS strips of 16 columns (the first PIECES * 8 of
  // them), through LDS, so that whole lines are written: value(n) gives a lane's four of
  // strip n, as f32 or bf16; put(row, column, eight values as they were).
  template <int STRIPS, int PIECES = STRIPS * 2, typename V, typename P>
  static DEVINL void out16(unsigned char* lds, V value, P put) {
    typedef decltype(value(0)) T4;
    constexpr int E = sizeof(T4) / 4, RS = STRIPS * 16 * E + 16;
    const int lane = threadIdx.x & (WAVE - 1), li = lane & 15, hi = lane >> 4;
    unsigned char* mine = lds + threadIdx.x / WAVE * (16 * OUT_RS);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int n = 0; n < STRIPS; ++n)
      *reinterpret_cast<T4*>(mine + li * RS + (n * 16 + hi * 4) * E) = value(n);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < (PIECES + 3) / 4; ++i) {
      const int at = i * 64 + lane, r = at / PIECES, c = at % PIECES * 8;
      if (PIECES % 4 && r >= 16) break;
      struct alignas(16) T8 { T4 lo, hi; };
      put(r, c, *reinterpret_cast<const T8*>(mine + r * RS + c * E));
    }
  }
};

struct RowsArgs {
  const unsigned short* A;     // (M, K)
  const unsigned short* W;     // (N, K); turned: (K, N)
  const unsigned short* R;     // (M, N) residual or null
  const unsigned short* bias;  // (N,) or null
  unsigned short* C;           // (M, N), or null:
  float* part;                 // (splits, M, N)
  int M, N, K, splits;
};

// The chip's order of tiles: up to eight row tiles of a column tile side by side on one
// XCD, which share W there, column after column, then the next rows: 32 workgroups at a
// time read 12 tiles' operands from beyond L2 (64 row tiles side by side, 33 of them: 3338
// us for 2745, 16384 rows of 28672 columns).
template <typename T>
DEVINL void rows_place(int M, int n_tiles, int& m0, int& nt, int& split) {
  const int mt = (M + T::BM - 1) / T::BM;
  const int n = gridDim.x, q = n / 8, r = n % 8, x = blockIdx.x % 8;
  int id = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + blockIdx.x / 8;
  split = id / (mt * n_tiles);
  id -= split * (mt * n_tiles);
  const int first = id / (8 * n_tiles) * 8, rows = min(8, mt - first);
  id -= first * n_tiles;
  m0 = (first + id % rows) * T::BM;
  nt = id / rows;
}

// Where a workgroup begins with K: rows of W are often a multiple of 4 KiB apart, so that
// workgroups in step read from a part of memory's channels at a time; an eighth of K apart
// by XCD, they read from all. us, W from memory, without, with, and with ONCE: 64 rows of
// 28672 x 4096 gated 51.2, 42.1, 38.9; 97 rows 54.3, 49.4, 46.2; 8192 x 8192, W alone 63.0,
// 48.4. Rows of 10 KiB have no such difference, splits begin apart as it is (same_channels;
// 4096 x 14336 in 8, 40 rows 23.6, 27.6), and where more row tiles share W, their products
// bound it: 333 rows 83.0, 83.5; 4096 rows 715, 713.
DEVINL int rows_begin(int steps) { return (int)(blockIdx.x % 8) * steps / 8; }

// grid: row tiles * column tiles * splits; K % BK == 0, N % 8 == 0. ONCE: one row tile.
template <typename T, bool ONCE = false>
__global__ __launch_bounds__(T::THREADS, T::MINW) void gemm_rows_kernel(RowsArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  int m0, nt, split;
  rows_place<T>(a.M, (a.N + T::BN - 1) / T::BN, m0, nt, split);
  const int n0 = nt * T::BN;
  const int all = a.K / T::BK, per = (all + a.splits - 1) / a.splits;
  const int first = split * per;

  unsigned ofs[T::LPW];
#pragma unroll
  for (int j = 0; j < T::LPW; ++j) {
    const int r = T::load_row(j, wave, lane);
    const unsigned byte = T::load_byte(j, wave, lane);
    if (T::TURNED && j >= T::AJ) {
      ofs[j] = (unsigned)r * (unsigned)(a.N * 2) + min(byte, (a.N - n0) * 2 - 16u);
    } else {
      const int row = j < T::AJ ? min(r, a.M - 1 - m0) : min(r, a.N - 1 - n0);
      ofs[j] = (unsigned)row * (unsigned)(a.K * 2) + byte;
    }
  }
  typename T::Acc acc;
  const long w_step = T::TURNED ? 64L * a.N : T::BK;
  const int steps = min(all, first + per) - first;
  T::template run<false, ONCE>(
      ofs, a.A + (long)m0 * a.K + (long)first * T::BK,
      a.W + (T::TURNED ? (long)n0 : (long)n0 * a.K) + first * w_step, steps, lds, acc,
      [](int) { return 0L; }, w_step, 0.f,
      ONCE && !T::TURNED && a.splits == 1 ? rows_begin(steps) : 0);

  const int c0 = n0 + T::col0(), r0 = m0 + T::row0();
  constexpr int S = T::COLS / 16;
#pragma unroll
  for (int m = 0; m < T::MI; ++m) {
    const int row0 = r0 + m * 16;
    if (!a.C) {
      float* part = a.part + ((long)split * a.M + row0) * a.N + c0;
      T::template out16<S>(lds, [&](int n) { return acc[m][n]; },
                           [&](int r, int c, auto v) {
        if (row0 + r >= a.M || c0 + c >= a.N) return;
        *reinterpret_cast<f32x4*>(part + (long)r * a.N + c) = v.lo;
        *reinterpret_cast<f32x4*>(part + (long)r * a.N + c + 4) = v.hi;
      });
    } else if (a.R || a.bias) {
      T::template out16<S>(lds, [&](int n) { return acc[m][n]; },
                           [&](int r, int c, auto v) {
        if (row0 + r >= a.M || c0 + c >= a.N) return;
        const long at = (long)(row0 + r) * a.N + c0 + c;
        float y[8], x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = e < 4 ? v.lo[e & 3] : v.hi[e & 3];
        if (a.bias) {
          load_bf16x8(a.bias + c0 + c, x);
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] += x[e];
        }
        if (a.R) {
          load_bf16x8(a.R + at, x);
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] += x[e];
        }
        store_bf16x8(a.C + at, y);
      });
    } else {
      T::template out16<S>(lds, [&](int n) { return pack4(acc[m][n]); },
                           [&](int r, int c, auto v) {
        if (row0 + r < a.M && c0 + c < a.N)
          *reinterpret_cast<decltype(v)*>(a.C + (long)(row0 + r) * a.N + c0 + c) = v;
      });
    }
  }
}

struct RowsGlu {
  int up, F, ldc;            // rows of W from a gate to its up, activations, C's columns
  const float* gate_b;       // CLAMPED: (F,) biases or null
  const float* up_b;
  float limit, slope;
  float eps;                 // NORM
};

// The gated product of a fused [gate | up] W, C (M, ldc) with zeros behind F, unsplit:
// silu(gate) * up, or with CLAMPED g = min(gate, limit), u = clamp(up, -limit, limit), g *
// sigmoid(slope * g) * (u + 1). A strip of 16 rows of the tile is eight gates and their
// eight ups: half of a lane's sums change places with those of the lane 32 on, and every
// lane has both. grid: row tiles * tiles of BN / 2 of C's columns; F, ldc % 8 == 0
// NORM: of the rows of A, their norm's weight folded into W.
template <typename T, bool CLAMPED, bool NORM = false, bool ONCE = false>
__global__ __launch_bounds__(T::THREADS, T::MINW) void gemm_rows_glu_kernel(RowsArgs a,
                                                                            RowsGlu glu) {
  static_assert(8 % T::RPC == 0, "rows of a load are of one kind");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & (WAVE - 1), hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  int m0, nt, split;
  rows_place<T>(a.M, (glu.ldc + T::BN / 2 - 1) / (T::BN / 2), m0, nt, split);
  const int n0 = nt * (T::BN / 2), w0 = min(n0, glu.F - 1);

  unsigned ofs[T::LPW];
#pragma unroll
  for (int j = 0; j < T::LPW; ++j) {
    const int r = T::load_row(j, wave, lane);
    const int row = j < T::AJ ? min(r, a.M - 1 - m0)
                              : min(r / 16 * 8 + r % 8, glu.F - 1 - w0);
    ofs[j] = (unsigned)row * (unsigned)(a.K * 2) + T::load_byte(j, wave, lane);
  }
  typename T::Acc acc;
  T::template run<NORM, ONCE>(
      ofs, a.A + (long)m0 * a.K, a.W + (long)w0 * a.K, a.K / T::BK, lds, acc,
      [&](int j) { return (long)(T::load_row(j, wave, 0) / 8 % 2) * glu.up * a.K; }, T::BK,
      glu.eps, ONCE ? rows_begin(a.K / T::BK) : 0);

  const int c0 = n0 + T::col0() / 2, r0 = m0 + T::row0();
  constexpr int NO = T::COLS / 16, S = (NO + 1) / 2;
  f32x4 gb[S], ub[S];
  if constexpr (CLAMPED) {
#pragma unroll
    for (int n = 0; n < S; ++n)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int at = min(c0 + n * 16 + hi * 4 + e, glu.F - 1);
        gb[n][e] = glu.gate_b ? glu.gate_b[at] : 0.f;
        ub[n][e] = glu.up_b ? glu.up_b[at] : 0.f;
      }
  }
#pragma unroll
  for (int m = 0; m < T::MI; ++m) {
    const int row0 = r0 + m * 16;
    T::template out16<S, NO>(lds, [&](int n) {
      const int col = c0 + n * 16 + hi * 4;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = acc[m][2 * n][e];
        const float y = 2 * n + 1 < NO ? acc[m][2 * n + 1 < NO ? 2 * n + 1 : 0][e] : 0.f;
        const auto s = __builtin_amdgcn_permlane32_swap(
            __builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y), false, false);
        float g = __builtin_bit_cast(float, (unsigned)s[0]);
        float u = __builtin_bit_cast(float, (unsigned)s[1]);
        if constexpr (CLAMPED) {
          g = fminf(g + gb[n][e], glu.limit);
          u = fminf(fmaxf(u + ub[n][e], -glu.limit), glu.limit);
          v[e] = g / (1.f + fast_expf(-glu.slope * g)) * (u + 1.f);
        } else {
          v[e] = g / (1.f + fast_expf(-g)) * u;
        }
        if (col >= glu.F) v[e] = 0.f;
      }
      return pack4(v);
    }, [&](int r, int c, auto v) {
      if (row0 + r < a.M && c0 + c < glu.ldc)
        *reinterpret_cast<decltype(v)*>(a.C + (long)(row0 + r) * glu.ldc + c0 + c) = v;
    });
  }
}

// Folds the splits, eight columns a thread; grid M * N / 8 / 256.
__global__ __launch_bounds__(256) void gemm_rows_fold_kernel(RowsArgs a) {
  const long n = (long)a.M * a.N;
  const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (at >= n) return;
  float v[8] = {};
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(a.part + s * n + at);
    const f32x4 y = *reinterpret_cast<const f32x4*>(a.part + s * n + at + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] += x[j];
      v[j + 4] += y[j];
    }
  }
  float x[8];
  if (a.bias) {
    load_bf16x8(a.bias + at % a.N, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += x[j];
  }
  if (a.R) {
    load_bf16x8(a.R + at, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += x[j];
  }
  store_bf16x8(a.C + at, v);
}

// The fold of a row with its residual, and the row's RMS norm in y. grid: M; N <= 4096 *
// ITERS. us of a product of 4096 x 4096 with a
// fold and a norm, and so: 33 rows in 8 splits 16.3, 15.4 (17.1 by 256 threads, which have
// fewer loads on their way); 97 in 4 18.3, 16.4; 250 26.2, 23.2; 8192 x 8192, 97 rows 42.3,
// 37.8.
template <int ITERS>
__global__ __launch_bounds__(512) void gemm_rows_fold_norm_kernel(
    RowsArgs a, const unsigned short* __restrict__ w, unsigned short* __restrict__ y,
    float eps) {
  const long row = (long)blockIdx.x * a.N, n = (long)a.M * a.N;
  float v[ITERS][8], wv[ITERS][8], r[ITERS][8];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int d = (it * 512 + threadIdx.x) * 8, c = d < a.N ? d : 0;
    load_bf16x8(w + c, wv[it]);
    load_bf16x8(a.R + row + c, r[it]);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[it][j] = 0.f;
  }
#pragma unroll 8
  for (int s = 0; s < a.splits; ++s)
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int d = (it * 512 + threadIdx.x) * 8, c = d < a.N ? d : 0;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(a.part + s * n + row + c);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(a.part + s * n + row + c + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[it][j] += lo[j];
        v[it][j + 4] += hi[j];
      }
    }
  float ssq = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int d = (it * 512 + threadIdx.x) * 8;
    if (d >= a.N) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[it][j] = bf2f(f2bf(v[it][j] + r[it][j]));
    store_bf16x8(a.C + row + d, v[it]);
#pragma unroll
    for (int j = 0; j < 8; ++j) ssq += v[it][j] * v[it][j];
  }
  ssq = wave_reduce_sum(ssq);
  __shared__ float sums[8];
  if ((threadIdx.x & (WAVE - 1)) == 0) sums[threadIdx.x / WAVE] = ssq;
  __syncthreads();
  ssq = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ssq += sums[i];
  const float inv = rsqrtf(ssq / (float)a.N + eps);
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int d = (it * 512 + threadIdx.x) * 8;
    if (d >= a.N) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[it][j] *= inv * wv[it][j];
    store_bf16x8(y + row + d, v[it]);
  }
}
