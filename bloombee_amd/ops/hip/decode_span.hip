// One decoded token of each of up to four sequences through a span of decoder layers, in
// one launch: [norm, q | k | v] -> [head norms, rotation, pages, attention] -> [output
// projection, sum] -> [norm, gated product] -> [down projection, sum], layer after layer.
//
// A launch costs 3 to 5 us whatever it does, and a small model's layer has little else:
// its weights are 6 us of memory, its six launches took 28. Here what one step makes and
// all workgroups need for the next goes through memory in a few KB, past the L2s, and
// nobody waits for a launch. 28 layers of 1024 columns, one sequence of 170 tokens: 795 us
// layer by layer, 385 here, 5 of them the launch ahead that clears the exchange; four layers
// of 4096 columns, one of 1024 tokens: 404 and 328 (358 where weights took their place in
// the caches, 333 with two pieces of the down projection on their way for four).
//
// Exchange. The words of a step's result (pairs of bf16, or an f32) are stored once each to
// memory that was filled with ones in all bits, which no result has, so that a word is its
// own flag: a reader asks for it again until it is there. Stores and loads are atomics of
// the agent's scope, which the L2s of other XCDs see. What all workgroups read is there in
// four copies. 256 workgroups exchange 2 KB in 0.95 us if they first ask when most of it is
// there (FIRST_POLL), in 1.5 if they ask at once and hold up the stores, in 2.0 to 2.3
// with a single copy. A CU's loads return in order: results are stored before the next
// weights are asked for, and no more of them than come during an exchange are asked for
// ahead of one that is waited for (a step that streams 12.6 MB takes 2.6 us with its
// exchange, 4.8 TB/s).
//
// Slots. The work of every step is cut in slots of equal size, one a CU; a workgroup owns a
// slot for the whole launch. Nothing here needs all workgroups to be resident: one that has
// waited long looks for slots that nobody has begun, and stands in for one until its own
// workgroup comes, from the first step on (results stay where they are for the whole
// launch; whoever runs a step stores the same bits). A slot that waits waits for earlier
// steps of slots that someone runs, so the earliest step always goes on, with any number of
// workgroups and whatever else the device is doing. Where another launch holds a CU for all
// of the time, who stands in does the work of two slots, and everybody waits for it: the
// drafter 930 us (391 alone, 800 layer by layer), four layers of 4096 columns 655 (370,
// 400); when all who waited left their straight way for catch_up(), 1170 and 922. Beside
// copies that fill the chip for 200 us each, the drafter 740 (1490 layer by layer; 2240 when
// a workgroup that came late found its slot taken). Several such launches at once take as
// long as one after the other: three drafters 1140 us, 1090 layer by layer.
// Attention's keys and values are many times what another slot has to load: where up to
// half the slots do for it they have nothing else (MOST_SPARED), and the others wait for
// it with all other weights of the layer in registers.
//
// Products. A unit is four rows of W; a wave takes 128 columns of it at a time, one 16-byte
// load a lane, whole lines of each row. What would be 16 rows of an MFMA operand are the
// four in four parts of 32 columns, against four rows of x in the same parts: products of
// unequal parts are nobody's. The eight waves of a workgroup split K.
//
// Between exchanges a step is one chain of latencies, some 0.8 to 1.2 us of it. Measured on
// the way: waits for loads that are still on their way (flat loads, registers that a branch
// joins, loads under conditions) cost 1 to 1.5 us each; LDS reads waited for one by one 0.5;
// ds_bpermute in place of DPP 0.1 each. Registers are short all the same: SmallSizes takes
// 256 and spills 72 more where a slot has attention and products, and both sizes keep some
// 700 scalar registers' worth in lanes.

#pragma once
#include "common.h"

namespace span {

constexpr int NW = 8, NT = NW * 64, SLOTS = 256, COPIES = 4, HEAD = 128;
constexpr int MAX_ROWS = 4, MAX_LAYERS = 48;
constexpr int STEPS = 6;            // of a layer
constexpr int PITCH = 144;          // floats of a unit's partial sums, 32 x 4 and padding
// Cached tokens of an attention split: a tile a wave. Twice that where it keeps attention
// to slots of its own: 4 sequences of 2000 tokens 646 us, 834 with 256; 1 of 300 would take
// 4% longer unsplit.
constexpr int MIN_PART = 256;
constexpr int PART_FLOATS = HEAD + 2;
// Slots for attention alone, at most: 4 sequences of 500 tokens 473 us, 548 where 32 was
// the most and all slots had rows of products; short contexts the same within 2%.
constexpr int MOST_SPARED = 128;
// From a step's results to the first look at the others', in 64 cycles. 12: 398 us, 22: 392,
// 26: 396, 30: 401; 4 of them between two looks: 395.
constexpr int FIRST_POLL = 22;
// Looks, of a quarter of a microsecond, until one for idle slots; such looks until a
// workgroup steps back though there are none; times it does so, some ten seconds.
constexpr int PATIENCE = 256, TRIES = 64, GIVE_UP = 1 << 12;
// A slot's flag: not begun, run by its own workgroup, or by another one, which adds the steps
// that it has done.
constexpr int IDLE = 0, OWN = 1, STAND_IN = 2;

typedef unsigned long long u64;
typedef unsigned short u16;
typedef __attribute__((ext_vector_type(4))) unsigned uint4v;

// What comes from a table in LDS says that it points to memory: loads of unknown kind
// would be waited for like LDS.
#define IN_MEMORY __attribute__((address_space(1)))
typedef IN_MEMORY u16* mem16;
typedef const IN_MEMORY u16* cmem16;

struct Layer {
  cmem16 qkv, o, gate_up, down;          // (N, K) each
  cmem16 q_norm, k_norm;                 // (HEAD,) or null
  mem16 k_pages, v_pages;                // (np, Hkv, P, HEAD), (np, Hkv, HEAD, P)
};

// words of a layer's exchange
struct Places { int x, h2, att, mid, qkv, part, all; };

struct Args {
  const u16* hidden;      // (M, H)
  u16* out;               // (M, H)
  const float *cos_t, *sin_t;   // (max_pos, HEAD / 2)
  const int *pos;         // (M,) or null: start
  const int *start;       // (M,)
  const int *table;       // (M, maxp)
  unsigned* work;         // SLOTS words of zeros, then the layers' exchanges
  int layers, M, H, I, Hq, Hkv, maxp, max_pos;
  int plog;               // tokens of a page, 1 << plog
  int parts;              // attention splits at most
  int units;              // of a slot, in partial sums
  int lds_wide, lds_sums, lds_squares, lds_control;   // byte offsets
  float inv_h, eps, scale;
  Places at;
  Layer layer[MAX_LAYERS];
};

static inline long fill_places(Places& p, long M, long H, long I, long Hq, long Hkv,
                               long parts) {
  long at = 0;
  auto take = [&](int& place, long words) {
    place = (int)at;
    at += words;
  };
  take(p.x, COPIES * M * H / 2);
  take(p.h2, COPIES * M * H / 2);
  take(p.att, COPIES * M * Hq * HEAD / 2);
  take(p.mid, COPIES * M * I / 2);
  take(p.qkv, M * (Hq + 2 * Hkv) * HEAD);
  take(p.part, parts > 1 ? M * Hq * parts * PART_FLOATS : 0);
  p.all = (int)at;
  return at;
}

struct Control {
  int late[2];          // of this step and of the one before
  int got, count, rounds, fail;
  short slot[SLOTS];
  int next[SLOTS];
  // of the launch's arguments, which are far away and not cached for long
  __attribute__((aligned(16))) Layer layer[MAX_LAYERS];
};

// LDS of attention: rows of queries, key and value, weights, results of waves
constexpr int ROW_B = (HEAD + 8) * 2, PROW_B = 32 * 2 + 16;
__host__ DEVINL int attention_lds(int G) {
  return (G + 2) * ROW_B + NW * 16 * PROW_B + NW * G * PART_FLOATS * 4;
}

DEVINL u64 peek(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL void put(unsigned* p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL void put(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL bool there(u64 v) { return (unsigned)v != ~0u && (unsigned)(v >> 32) != ~0u; }
// all ones is NaN (twice, of bf16): another one stands for it
DEVINL unsigned settled(unsigned w) { return w == ~0u ? 0x7fff7fffu : w; }
DEVINL unsigned bits(float v) { return __builtin_bit_cast(unsigned, v); }
DEVINL float as_float(unsigned v) { return __builtin_bit_cast(float, v); }
DEVINL unsigned to_bf16(float v) { return __builtin_bit_cast(u16, (__bf16)v); }

// barriers that leave loads in flight
DEVINL void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The value of another lane of the same sixteen: xor 1, xor 2, n lanes up, n lanes around.
template <int CTRL>
DEVINL unsigned lane_of(unsigned v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
constexpr int XOR1 = 0xb1, XOR2 = 0x4e, UP = 0x100, AROUND = 0x120;
template <int CTRL>
DEVINL float lane_of(float v) { return as_float(lane_of<CTRL>(bits(v))); }
// Of a lane and the one 16 (32) lanes away: v as it is in rows 0 and 2 (halves 0), and in
// the others.
struct Two { float a, b; };
DEVINL Two rows16(float v) {
  const auto s = __builtin_amdgcn_permlane16_swap(bits(v), bits(v), false, false);
  return {as_float(s[0]), as_float(s[1])};
}
DEVINL Two halves(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(bits(v), bits(v), false, false);
  return {as_float(s[0]), as_float(s[1])};
}
DEVINL float max_over_rows(float v) {
  Two t = rows16(v);
  t = halves(fmaxf(t.a, t.b));
  return fmaxf(t.a, t.b);
}
DEVINL float sum_over_rows(float v) {
  Two t = rows16(v);
  t = halves(t.a + t.b);
  return t.a + t.b;
}
DEVINL float sum_of_wave(float v) {
  v += lane_of<AROUND + 8>(v);
  v += lane_of<AROUND + 4>(v);
  v += lane_of<AROUND + 2>(v);
  v += lane_of<AROUND + 1>(v);
  return sum_over_rows(v);
}
DEVINL float sum_of_four(float v) {
  v += lane_of<XOR1>(v);
  return v + lane_of<XOR2>(v);
}

// A slot's rows of W in one step: units [first, first + units), pairs of units where gate
// and up rows go together. Offsets of W are 32 bits of bytes.
struct Job {
  cmem16 W;
  unsigned up;          // from a gate row to its up row
  int K, steps;         // pieces of 128 columns
  int first, units, last;
};

template <bool PAIRED>
DEVINL Job job_of(cmem16 W, int rows, int K, int i, int slots) {
  Job j;
  const int all = rows / (PAIRED ? 8 : 4);
  j.W = W;
  j.up = (unsigned)(rows / 2) * K * 2;
  j.K = K;
  j.steps = K / 128;
  j.first = max(i, 0) * all / slots;
  j.units = i < 0 ? 0 : (i + 1) * all / slots - j.first;
  j.last = max(j.first + j.units - 1, 0);
  return j;
}

// U units of which DP pieces are on their way, in registers. A wave takes pieces wave,
// wave + 8, ... of K. ONE: a slot has no more than that.
template <int U, int DP, bool PAIRED, bool ONE>
struct Stream {
  static constexpr int UNITS = U, PER = PAIRED ? U / 2 : U;
  static constexpr bool WHOLE = ONE;
  short8 w[DP][U];
  int group, turn;      // of the next piece that is asked for

  template <int FROM = 0, int TO = U>
  DEVINL void load(const Job& j, int wave, unsigned lane_ofs, int d, int g, int t) {
    const int s = min(wave + t * NW, j.steps - 1);
#pragma unroll
    for (int u = FROM; u < TO; ++u) {
      if (ONE && (PAIRED ? u / 2 : u) >= j.units) break;
      const int unit = min(j.first + g * PER + (PAIRED ? u / 2 : u), j.last);
      const unsigned at = (unsigned)(unit * 4 * j.K + s * 128) * 2 +
                          (PAIRED && (u & 1) ? j.up : 0) + lane_ofs;
      w[d][u] = __builtin_nontemporal_load(reinterpret_cast<const IN_MEMORY short8*>(
          reinterpret_cast<const IN_MEMORY char*>(j.W) + at));
    }
  }
  DEVINL static unsigned place(int K, int lane) {
    return (unsigned)((lane & 3) * K + (lane >> 2 & 3) * 32 + (lane >> 4) * 8) * 2;
  }
  DEVINL void next(const Job& j, int wave, unsigned lane_ofs, int d) {
    load(j, wave, lane_ofs, d, group, turn);
    if (++turn * NW >= j.steps) {
      turn = 0;
      ++group;
    }
  }
  DEVINL void begin(const Job& j, int wave, int lane) {
    if constexpr (ONE) {
      begin_units<0, U>(j, wave, lane);
      return;
    }
    group = turn = 0;
#pragma unroll
    for (int d = 0; d < DP; ++d) next(j, wave, place(j.K, lane), d);
    __builtin_amdgcn_sched_barrier(0);
  }
  template <int FROM, int TO>
  DEVINL void begin_units(const Job& j, int wave, int lane) {
#pragma unroll
    for (int d = 0; d < DP; ++d) load<FROM, TO>(j, wave, place(j.K, lane), d, 0, d);
    __builtin_amdgcn_sched_barrier(0);
  }
  // x: (M, K) in LDS. Partial sums of the wave go to sums, [row of x][unit][32][4].
  // Waits for what is on its way, so that what is asked for next can stay so.
  DEVINL void arrive() {
#pragma unroll
    for (int d = 0; d < DP; ++d)
#pragma unroll
      for (int u = 0; u < U; ++u) asm volatile("" : "+v"(w[d][u]));
  }
  template <bool NORM>
  DEVINL void run(const Job& j, int wave, int lane, const u16* x, int M, int units,
                  float* sums, float* squares) {
    const int li = lane & 15, hi = lane >> 4, m = li & 3, part = li >> 2;
    const u16* xl = x + min(m, M - 1) * j.K + part * 32 + hi * 8;
    f32x4 acc[U], sq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int d, int t, bool squared) {
      const int s = wave + t * NW;
      short8 xf = *reinterpret_cast<const short8*>(xl + min(s, j.steps - 1) * 128);
      if (s >= j.steps) xf = short8{};
#pragma unroll
      for (int u = 0; u < U; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[d][u]),
                                                         as_bf16x8(xf), acc[u], 0, 0, 0);
      if (NORM && squared)
        sq = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(xf), as_bf16x8(xf), sq, 0,
                                                     0, 0);
    };
    // lanes of the sixteen rows that hold this part's
    auto flush = [&](int g) {
      if (hi == part && m < M) {
        float* to = sums + (m * units + g * U) * PITCH + (wave * 4 + part) * 4;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (ONE && (PAIRED ? u / 2 : u) >= j.units) break;
          *reinterpret_cast<f32x4*>(to + u * PITCH) = acc[u];
        }
      }
    };
    if constexpr (ONE) {
#pragma unroll
      for (int d = 0; d < DP; ++d) multiply(d, d, true);
      flush(0);
    } else {
      const unsigned lane_ofs = place(j.K, lane);
      const int turns = (j.steps + NW - 1) / NW;
      const int all = (j.units + PER - 1) / PER * turns;
      int g = 0, t = 0;
      auto consume = [&](int d) {
        multiply(d, t, g == 0);
        if (++t == turns) {
          flush(g);
#pragma unroll
          for (int u = 0; u < U; ++u) acc[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
          t = 0;
          ++g;
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      int i = 0;
      for (; i + 2 * DP <= all; i += DP)
#pragma unroll
        for (int d = 0; d < DP; ++d) {
          consume(d);
          next(j, wave, lane_ofs, d);
        }
      for (; i < all; i += DP)
#pragma unroll
        for (int d = 0; d < DP; ++d)
          if (i + d < all) {
            consume(d);
            if (i + d + DP < all) next(j, wave, lane_ofs, d);
          }
    }
    if (NORM) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (hi * 4 + e == li) squares[wave * 16 + li] = sq[e];
    }
  }
};

// What differs with the size of a model: units and pieces in registers of each product.
// Small: all that a slot has of a layer of 1024 columns, also where half of them are spared;
// what a slot does not have is not loaded. Large: pieces follow each other. Any: whatever
// slot, a step at a time; its units divide the others', whose partial sums have room.
struct SmallSizes {
  static constexpr bool EARLY = true, SPARES = true;
  typedef Stream<8, 1, false, true> Qkv;
  typedef Stream<2, 2, false, true> O;
  typedef Stream<12, 1, true, true> Glu;
  typedef Stream<2, 3, false, true> Down;
  typedef Stream<2, 2, false, false> AnyRows;
  typedef Stream<2, 2, true, false> AnyPairs;
};
struct LargeSizes {
  static constexpr bool EARLY = false, SPARES = false;
  typedef Stream<6, 2, false, false> Qkv;
  typedef Stream<4, 2, false, false> O;
  typedef Stream<4, 2, true, false> Glu;
  typedef Stream<4, 4, false, false> Down;
  typedef Stream<2, 4, false, false> AnyRows;
  typedef Stream<4, 2, true, false> AnyPairs;
};

template <class Sizes>
struct Worker {
  const Args& a;
  unsigned char* lds;
  Control* ctl;
  int tid, lane, wave;
  int flag;             // which of the two late ones is this step's
  int parts, grain;     // attention splits of the longest sequence, tokens of one
  int spared;           // slots that have attention only, no rows of the products
  int patience;         // the other slots' is longer: who has attention only stands in first

  DEVINL Worker(const Args& args, unsigned char* l) : a(args), lds(l) {
    ctl = reinterpret_cast<Control*>(lds + a.lds_control);
    tid = threadIdx.x;
    lane = tid & 63;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    flag = 0;
    int longest = 0;
    for (int b = 0; b < a.M; ++b) longest = max(longest, a.start[b] + 1);
    grain = MIN_PART;
    spared = 0;
    if constexpr (Sizes::SPARES) {
      const int units = a.M * a.Hkv;
      if (units * parts_of(longest) > MOST_SPARED) grain = 2 * MIN_PART;
      spared = units * parts_of(longest);
      if (spared > MOST_SPARED) {
        spared = 0;
        grain = MIN_PART;
      }
    }
    parts = parts_of(longest);
    patience = (int)blockIdx.x < spared || !spared ? PATIENCE : 8 * PATIENCE;
  }
  DEVINL int parts_of(int ctx) { return min(a.parts, (ctx + grain - 1) / grain); }
  DEVINL Layer layer_of(int l) {
    constexpr int N = sizeof(Layer) / 4;
    struct Words { int w[N]; } t = __builtin_bit_cast(Words, ctl->layer[l]);
#pragma unroll
    for (int i = 0; i < N; ++i) t.w[i] = __builtin_amdgcn_readfirstlane(t.w[i]);
    return __builtin_bit_cast(Layer, t);
  }
  DEVINL u16* hid() { return reinterpret_cast<u16*>(lds); }
  DEVINL unsigned char* wide() { return lds + a.lds_wide; }
  DEVINL u16* wide16() { return reinterpret_cast<u16*>(wide()); }
  DEVINL float* sums() { return reinterpret_cast<float*>(lds + a.lds_sums); }
  DEVINL float* squares() { return reinterpret_cast<float*>(lds + a.lds_squares); }
  DEVINL unsigned* exchange(int l) { return a.work + SLOTS + (long)l * a.at.all; }
  DEVINL int qkv_rows() { return (a.Hq + 2 * a.Hkv) * HEAD; }
  // Addresses are made anew: kept for all layers they would fill the registers.
  DEVINL void fresh() {
    asm volatile("" : "+v"(tid));
    lane = tid & 63;
    flag ^= 1;
  }

  // ---- jobs
  template <bool PAIRED>
  DEVINL Job job(cmem16 W, int rows, int K, int slot) {
    return job_of<PAIRED>(W, rows, K, slot - spared, SLOTS - spared);
  }
  DEVINL Job qkv_job(const Layer& w, int slot) {
    return job<false>(w.qkv, qkv_rows(), a.H, slot);
  }
  DEVINL Job o_job(const Layer& w, int slot) {
    return job<false>(w.o, a.H, a.Hq * HEAD, slot);
  }
  DEVINL Job glu_job(const Layer& w, int slot) {
    return job<true>(w.gate_up, 2 * a.I, a.H, slot);
  }
  DEVINL Job down_job(const Layer& w, int slot) {
    return job<false>(w.down, a.H, a.I, slot);
  }

  // ---- waiting. Who waited in vain says so; after the next barrier all know, and take up
  // a slot that nobody has begun, if there is one.
  DEVINL bool late() { return __builtin_amdgcn_readfirstlane(ctl->late[flag]); }
  DEVINL int* flags() { return reinterpret_cast<int*>(a.work); }
  DEVINL bool idle(int slot) {
    return __hip_atomic_load(flags() + slot, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT) == IDLE;
  }
  // Whether to look again after a look in vain. Only who could take up a slot leaves the
  // straight way for it: results are late where others load long contexts, too.
  DEVINL bool patient(int& looks) {
    if (++looks % PATIENCE || looks % patience) return true;
    bool any = looks == PATIENCE * TRIES;
#pragma unroll
    for (int k = 0; k < SLOTS; k += WAVE) any |= idle(k + lane);
    return !__builtin_amdgcn_ballot_w64(any);
  }
  // Everybody begins to look at another place, so that they find different ones.
  DEVINL void claim_idle() {
    if (tid == 0) ctl->got = SLOTS;
    meet();
    const int own = __builtin_amdgcn_readfirstlane(ctl->slot[0]);
    if (tid < SLOTS && idle(tid)) atomicMin(&ctl->got, (tid - own) & (SLOTS - 1));
    meet();
    if (tid == 0) {
      const int s = (own + ctl->got) & (SLOTS - 1);
      int nobody = IDLE;
      ctl->late[0] = ctl->late[1] = 0;
      ctl->fail = ++ctl->rounds > GIVE_UP;
      if (ctl->got < SLOTS &&
          __hip_atomic_compare_exchange_strong(flags() + s, &nobody, STAND_IN,
                                               __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)) {
        ctl->slot[ctl->count] = (short)s;
        ctl->next[ctl->count++] = 0;
      }
    }
    meet();
  }
  // Whether a slot's own workgroup has come, so that nobody need stand in any more; it is told
  // how far that has got.
  DEVINL bool relieved(int slot, int done) {
    int seen = __hip_atomic_load(flags() + slot, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
    return seen == OWN || !__hip_atomic_compare_exchange_strong(
                              flags() + slot, &seen, STAND_IN + done, __ATOMIC_RELAXED,
                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // Whether this workgroup runs its own slot: not if another one has done half of it.
  DEVINL bool begins(int slot) {
    int seen = __hip_atomic_load(flags() + slot, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
    while (seen < STAND_IN + a.layers * STEPS / 2)
      if (__hip_atomic_compare_exchange_strong(flags() + slot, &seen, OWN,
                                               __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        return true;
    return false;
  }
  // Rows of 64 words of 8 bytes to LDS; false if some were not there for long. Waves take
  // rows in turns, without masks.
  template <int DELAY>
  DEVINL bool gather(const u64* src, unsigned char* dst, int rows) {
    constexpr int J = 4;
    const u64* from = src + lane;
    u64* to = reinterpret_cast<u64*>(dst) + lane;
    int looks = 0;
    if (DELAY && wave < rows) __builtin_amdgcn_s_sleep(DELAY);
    for (int r = wave; r < rows; r += NW * J) {
      u64 v[J];
      while (true) {
        bool missing = false;
#pragma unroll
        for (int j = 0; j < J; ++j)
          if (r + j * NW < rows) v[j] = peek(from + (r + j * NW) * 64);
#pragma unroll
        for (int j = 0; j < J; ++j)
          if (r + j * NW < rows) missing |= !there(v[j]);
        if (!__builtin_amdgcn_ballot_w64(missing)) break;
        if (!patient(looks)) return false;
      }
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (r + j * NW < rows) to[(r + j * NW) * 64] = v[j];
    }
    return true;
  }
  template <int DELAY = 0>
  DEVINL void fetch(const unsigned* src, unsigned char* dst, int words) {
    if (!gather<DELAY>(reinterpret_cast<const u64*>(src), dst, words / 128))
      ctl->late[flag] = 1;
  }
  // a slot's copy of what all read
  DEVINL void fetch_copy(const unsigned* src, unsigned char* dst, int columns, int slot) {
    const int words = a.M * columns / 2;
    fetch<FIRST_POLL>(src + (slot & (COPIES - 1)) * words, dst, words);
  }
  DEVINL void fetch_hidden(int l, int slot) {
    if (l > 0) {
      fetch_copy(exchange(l - 1) + a.at.x, lds, a.H, slot);
      return;
    }
    for (int i = tid; i < a.M * a.H / 4; i += NT)
      reinterpret_cast<u64*>(lds)[i] = reinterpret_cast<const u64*>(a.hidden)[i];
  }
  DEVINL void fetch_attention(int l, int slot) {
    fetch_copy(exchange(l) + a.at.att, wide(), a.Hq * HEAD, slot);
  }
  DEVINL void fetch_h2(int l, int slot) {
    fetch_copy(exchange(l) + a.at.h2, lds, a.H, slot);
  }
  DEVINL void fetch_mid(int l, int slot) {
    fetch_copy(exchange(l) + a.at.mid, wide(), a.I, slot);
  }

  // ---- products of what was fetched; false: it was late, nothing has been handed on
  template <bool NORM, class S>
  DEVINL bool multiply(const Job& j, S& s, const u16* x) {
    meet();
    const int in_vain = ctl->late[flag];
    if (S::WHOLE) s.arrive();
    s.template run<NORM>(j, wave, lane, x, a.M, a.units, sums(), squares());
    meet();
    return !__builtin_amdgcn_readfirstlane(in_vain);
  }
  // f(unit, row of x, row of the unit, quarter): four lanes an output, sixteen a unit; the
  // rows of x are shared out among the waves
  template <class F>
  DEVINL void outputs(int units, F f) {
    const int log = a.M > 2 ? 2 : a.M - 1, m = wave & ((1 << log) - 1);
    if (m >= a.M) return;
    for (int u = (wave >> log) * 4; u < units; u += NT / 16 >> log)
      if (u + (lane >> 4) < units) f(u + (lane >> 4), m, lane >> 2 & 3, lane & 3);
  }
  // Terms are read all at once: one after the other they would be waited for so.
  struct Terms { float v[NW]; };
  DEVINL Terms terms(int unit, int m, int row, int q) {
    return read(sums() + (m * a.units + unit) * PITCH + q * 4 + row);
  }
  DEVINL Terms squares_of(int m, int q) { return read(squares() + q * 4 + m); }
  DEVINL Terms read(const float* p) {
    Terms t;
#pragma unroll
    for (int w = 0; w < NW; ++w) t.v[w] = p[w * 16];
    return t;
  }
  DEVINL float total(const Terms& t) {
    float v = t.v[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += t.v[w];
    return sum_of_four(v);
  }
  DEVINL float inverse_rms(const Terms& t) {
    return rsqrtf(total(t) * a.inv_h + a.eps);
  }
  // A unit's four rows, for the lanes of the first
  DEVINL u64 pack_rows(float v) {
    const unsigned b = to_bf16(v);
    const unsigned lo = b | lane_of<UP + 4>(b) << 16;
    const unsigned hi = lane_of<UP + 8>(b) | lane_of<UP + 12>(b) << 16;
    return settled(lo) | (u64)settled(hi) << 32;
  }
  template <class S>
  DEVINL bool run_qkv(int l, const Job& j, S& s) {
    if (!multiply<true>(j, s, hid())) return false;
    unsigned* dst = exchange(l) + a.at.qkv + j.first * 4;
    const int N = qkv_rows();
    outputs(j.units, [&](int u, int m, int row, int q) {
      const Terms t = terms(u, m, row, q), sq = squares_of(m, q);
      __builtin_amdgcn_sched_barrier(0);
      const float v = total(t) * inverse_rms(sq);
      if (q == 0) put(dst + m * N + u * 4 + row, settled(bits(v)));
    });
    return true;
  }
  // a product's sum with the residual in hid
  template <class S>
  DEVINL bool run_sum(const Job& j, S& s, unsigned* dst) {
    if (!multiply<false>(j, s, wide16())) return false;
    outputs(j.units, [&](int u, int m, int row, int q) {
      const int n = m * a.H + (j.first + u) * 4;
      const Terms t = terms(u, m, row, q);
      const u16 residual = hid()[n + row];
      __builtin_amdgcn_sched_barrier(0);
      const u64 w = pack_rows(total(t) + bf2f(residual));
      if (row) return;
      if (dst)
        put(reinterpret_cast<u64*>(dst) + (q * a.M * a.H + n) / 4, w);
      else if (q == 0)
        reinterpret_cast<u64*>(a.out)[n / 4] = w;
    });
    return true;
  }
  template <class S>
  DEVINL bool run_o(int l, const Job& j, S& s) {
    return run_sum(j, s, exchange(l) + a.at.h2);
  }
  template <class S>
  DEVINL bool run_glu(int l, const Job& j, S& s) {
    if (!multiply<true>(j, s, hid())) return false;
    u64* dst = reinterpret_cast<u64*>(exchange(l) + a.at.mid);
    outputs(j.units, [&](int u, int m, int row, int q) {
      const Terms tg = terms(2 * u, m, row, q), tv = terms(2 * u + 1, m, row, q);
      const Terms sq = squares_of(m, q);
      __builtin_amdgcn_sched_barrier(0);
      const float r = inverse_rms(sq), g = total(tg) * r, v = total(tv) * r;
      const u64 w = pack_rows(g / (1.f + fast_expf(-g)) * v);
      if (row == 0) put(dst + ((q * a.M + m) * a.I) / 4 + j.first + u, w);
    });
    return true;
  }
  template <class S>
  DEVINL bool run_down(int l, const Job& j, S& s) {
    return run_sum(j, s, l + 1 < a.layers ? exchange(l) + a.at.x : nullptr);
  }

  // ---- attention: a slot is a split of a sequence's keys for a key head. Scores are
  // transposed (rows: positions, columns: heads of the group), as in attn_decode_mfma.hip;
  // a wave takes tiles of 32 positions in turns, the first one's keys and values are asked
  // for before the queries are there. What does not change from layer to layer:
  struct Split {
    bool any, tile;             // the split has tokens, this wave a tile
    int b, head, split, parts, ctx, c0, c1;
    int page, vpage, kpage[2];  // of the new token; of the wave's first tile
    float cs[2], sn[2];         // of dimensions 2 (lane % 32) and the next
  };
  DEVINL Split split_of(int slot) {
    Split s = {};
    const int BH = a.M * a.Hkv;
    if (slot >= BH * parts) return s;
    const int bh = slot % BH;
    s.split = slot / BH;
    s.b = bh / a.Hkv;
    s.head = bh % a.Hkv;
    s.ctx = a.start[s.b] + 1;
    const int tiles = (s.ctx + 31) / 32;
    const int want = parts_of(s.ctx);
    const int per = (tiles + want - 1) / want;
    s.parts = (tiles + per - 1) / per;
    s.c0 = s.split * per * 32;
    s.c1 = min(s.ctx, s.c0 + per * 32);
    s.any = s.split < s.parts;
    if (!s.any) return s;
    const int last = s.ctx - 1;
    const int p = min(max(a.pos ? a.pos[s.b] : last, 0), a.max_pos - 1);
    const long d = (long)p * (HEAD / 2) + (lane & 31) * 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s.cs[i] = a.cos_t[d + i];
      s.sn[i] = a.sin_t[d + i];
    }
    s.page = a.table[(long)s.b * a.maxp + (last >> a.plog)];
    s.tile = s.c0 + wave * 32 < s.c1;
    if (s.tile) look_up(s, s.c0 + wave * 32, s.vpage, s.kpage);
    return s;
  }
  DEVINL void look_up(const Split& s, int tb, int& v, int (&k)[2]) {
    const int* t = a.table + (long)s.b * a.maxp;
    v = t[min(tb + (lane >> 4) * 8, (s.c1 - 1) & ~7) >> a.plog];
#pragma unroll
    for (int n = 0; n < 2; ++n) k[n] = t[min(tb + (lane & 15) + 16 * n, s.c1 - 1) >> a.plog];
  }
  DEVINL void load_k(short8 (&k)[2][4], const Layer& w, const Split& s, int tb,
                     const int (&page)[2]) {
    const int P = 1 << a.plog;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int pos = min(tb + (lane & 15) + 16 * n, s.c1 - 1);
      cmem16 row = w.k_pages +
                       (((long)page[n] * a.Hkv + s.head) * P + (pos & (P - 1))) * HEAD +
                       (lane >> 4) * 8;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        k[n][kk] = __builtin_nontemporal_load(
            reinterpret_cast<const IN_MEMORY short8*>(row + 32 * kk));
    }
  }
  DEVINL void load_v(short8 (&v)[8], const Layer& w, const Split& s, int tb, int page) {
    const int P = 1 << a.plog;
    const int pos = min(tb + (lane >> 4) * 8, (s.c1 - 1) & ~7);
    cmem16 row = w.v_pages +
                     (((long)page * a.Hkv + s.head) * HEAD + (lane & 15)) * P +
                     (pos & (P - 1));
#pragma unroll
    for (int n = 0; n < 8; ++n)
      v[n] = __builtin_nontemporal_load(
          reinterpret_cast<const IN_MEMORY short8*>(row + 16 * n * P));
  }
  struct Tile {
    short8 k[2][4], v[8];
    unsigned norm;        // weights of this wave's head, two dimensions
  };
  DEVINL void load_tile(Tile& t, const Layer& w, const Split& s) {
    if (s.tile) {
      load_k(t.k, w, s, s.c0 + wave * 32, s.kpage);
      load_v(t.v, w, s, s.c0 + wave * 32, s.vpage);
    }
    if (w.q_norm) t.norm = norm_of(w, wave);
    __builtin_amdgcn_sched_barrier(0);
  }
  DEVINL unsigned norm_of(const Layer& w, int h) {
    return reinterpret_cast<const IN_MEMORY unsigned*>(
        h < a.Hq / a.Hkv ? w.q_norm : w.k_norm)[lane];
  }

  // The group's queries, the new key and value, a wave a head: from the exchange through
  // norm and rotation to LDS. A lane has dimensions 2 lane and the next.
  DEVINL bool fetch_heads(int l, const Layer& w, const Split& s, unsigned norm) {
    const int G = a.Hq / a.Hkv, P = 1 << a.plog, last = s.ctx - 1;
    const bool newest = s.c1 == s.ctx;
    unsigned kept[2] = {0, 0};
    for (int h = wave; h < G + 2; h += NW) {
      const int from = h < G ? s.head * G + h : a.Hq + (h == G ? 0 : a.Hkv) + s.head;
      const u64* src = reinterpret_cast<const u64*>(
                           exchange(l) + a.at.qkv + s.b * qkv_rows() + from * HEAD) + lane;
      u64 got;
      int looks = 0;
      do got = peek(src);
      while (__builtin_amdgcn_ballot_w64(!there(got)) && patient(looks));
      if (!there(got)) ctl->late[flag] = 1;
      float x = as_float((unsigned)got), y = as_float((unsigned)(got >> 32));
      if (h <= G) {
        if (w.q_norm) {
          const unsigned n = h == wave ? norm : norm_of(w, h);
          const float r = rsqrtf(sum_of_wave(x * x + y * y) / HEAD + a.eps);
          x *= r * as_float(n << 16);
          y *= r * as_float(n & 0xffff0000u);
        }
        // dimension d turns with d + HEAD / 2, which is 32 lanes away
        const Two tx = halves(x), ty = halves(y);
        const bool up = lane >= 32;
        x = up ? tx.b * s.cs[0] + tx.a * s.sn[0] : tx.a * s.cs[0] - tx.b * s.sn[0];
        y = up ? ty.b * s.cs[1] + ty.a * s.sn[1] : ty.a * s.cs[1] - ty.b * s.sn[1];
      }
      const unsigned b = to_bf16(x) | to_bf16(y) << 16;
      reinterpret_cast<unsigned*>(wide() + h * ROW_B)[lane] = b;
      kept[h / NW] = b;
    }
    meet();
    if (late()) return false;
    for (int h = wave; newest && h < G + 2; h += NW) {
      const unsigned b = kept[h / NW];
      const long row = (long)s.page * a.Hkv + s.head;
      if (h == G) {
        reinterpret_cast<IN_MEMORY unsigned*>(
            w.k_pages + (row * P + (last & (P - 1))) * HEAD)[lane] = b;
      } else if (h == G + 1) {
        mem16 dst = w.v_pages + (row * HEAD + 2 * lane) * P + (last & (P - 1));
        dst[0] = (u16)b;
        dst[P] = (u16)(b >> 16);
      }
    }
    return true;
  }

  // Attention of the split; t: the wave's first tile.
  DEVINL void attend(int l, const Layer& w, const Split& s, Tile& t) {
    const int G = a.Hq / a.Hkv, li = lane & 15, hi = lane >> 4, last = s.ctx - 1;
    unsigned char* rows = wide();      // bf16: queries, key, value
    unsigned char* p_lds = rows + (G + 2) * ROW_B + wave * 16 * PROW_B;
    float* merge = reinterpret_cast<float*>(rows + (G + 2) * ROW_B + NW * 16 * PROW_B);
    const float sc2 = a.scale * LOG2E;
    float m2 = NEG_BIG, sum = 0.f;
    f32x4 acc[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) acc[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 q[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      q[kk] = as_bf16x8(*reinterpret_cast<const short8*>(
          rows + min(li, G - 1) * ROW_B + (hi * 8 + 32 * kk) * 2));
    for (int tb = s.c0 + wave * 32; tb < s.c1; tb += NW * 32) {
      const bool more = tb + NW * 32 < s.c1;
      int vnext = 0, knext[2] = {0, 0};
      if (more) look_up(s, tb + NW * 32, vnext, knext);
      if (tb + 32 >= s.ctx) {      // the new token; positions behind it are zero
#pragma unroll
        for (int n = 0; n < 2; ++n)
          if (tb + li + 16 * n == last) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
              t.k[n][kk] = *reinterpret_cast<const short8*>(
                  rows + G * ROW_B + (hi * 8 + 32 * kk) * 2);
          }
        const u16* nv = reinterpret_cast<const u16*>(rows + (G + 1) * ROW_B);
        const int e = last - (tb + hi * 8);
        unsigned old[4], mine[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          old[i] = e > 2 * i + 1 ? ~0u : e > 2 * i ? 0xffffu : 0u;
          mine[i] = e == 2 * i ? 0xffffu : e == 2 * i + 1 ? 0xffff0000u : 0u;
        }
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const unsigned x = nv[li + 16 * n] * 0x10001u;
          uint4v v = __builtin_bit_cast(uint4v, t.v[n]);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = (v[i] & old[i]) | (x & mine[i]);
          t.v[n] = __builtin_bit_cast(short8, v);
        }
      }
      f32x4 st[2];
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        st[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          st[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(t.k[n][kk]), q[kk],
                                                          st[n], 0, 0, 0);
      }
      if (more) load_k(t.k, w, s, tb + NW * 32, knext);
      float p[2][4], rm = NEG_BIG;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int pos = tb + 16 * n + hi * 4 + e;
          p[n][e] = pos < s.c1 ? st[n][e] * sc2 : NEG_BIG;
          rm = fmaxf(rm, p[n][e]);
        }
      const float mn = fmaxf(m2, max_over_rows(rm)), corr = fast_exp2(m2 - mn);
      float ps = 0.f;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        u64 packed = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[n][e] = fast_exp2(p[n][e] - mn);
          ps += p[n][e];
          packed |= (u64)to_bf16(p[n][e]) << (16 * e);
        }
        *reinterpret_cast<u64*>(p_lds + li * PROW_B + (16 * n + hi * 4) * 2) = packed;
      }
      sum = sum * corr + sum_over_rows(ps);
      m2 = mn;
#pragma unroll
      for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[n][e] *= corr;
      const bf16x8 pf = as_bf16x8(
          *reinterpret_cast<const short8*>(p_lds + li * PROW_B + hi * 16));
#pragma unroll
      for (int n = 0; n < 8; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(t.v[n]), pf, acc[n], 0,
                                                         0, 0);
      if (more) load_v(t.v, w, s, tb + NW * 32, vnext);
    }
    if (li < G) {
      float* dst = merge + (wave * G + li) * PART_FLOATS;
#pragma unroll
      for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int e = 0; e < 4; e += 2)
          *reinterpret_cast<f32x2*>(dst + 16 * n + hi * 4 + e) =
              (f32x2){acc[n][e], acc[n][e + 1]};
      if (hi == 0) *reinterpret_cast<f32x2*>(dst + HEAD) = (f32x2){m2, sum};
    }
    meet();
    for (int i = tid; i < G * HEAD; i += NT) {
      const int g = i / HEAD, d = i % HEAD;
      const float* src = merge + g * PART_FLOATS;
      f32x2 ml[NW];
      float x[NW], mx = NEG_BIG, lt = 0.f, o = 0.f;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        ml[v] = *reinterpret_cast<const f32x2*>(src + v * G * PART_FLOATS + HEAD);
        x[v] = src[v * G * PART_FLOATS + d];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int v = 0; v < NW; ++v) mx = fmaxf(mx, ml[v][0]);
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        const float c = fast_exp2(ml[v][0] - mx);
        lt += ml[v][1] * c;
        o += x[v] * c;
      }
      if (s.parts == 1) {
        put_head(l, s.b, s.head * G + g, d, lt > 0.f ? o * (1.f / lt) : 0.f);
        continue;
      }
      unsigned* dst = part_of(l, s, g);
      put(dst + s.split * HEAD + d, settled(bits(o)));
      if (d == 0)
        put(reinterpret_cast<u64*>(dst + a.parts * HEAD) + s.split,
            settled(bits(mx)) | (u64)settled(bits(lt)) << 32);
    }
  }
  DEVINL unsigned* part_of(int l, const Split& s, int g) {
    return exchange(l) + a.at.part +
           (s.b * a.Hq + s.head * (a.Hq / a.Hkv) + g) * a.parts * PART_FLOATS;
  }
  // dimension d of a head's result; four lanes have the same four
  DEVINL void put_head(int l, int b, int h, int d, float v) {
    const unsigned x = to_bf16(v), o = lane_of<XOR1>(x);
    const unsigned w = settled(lane & 1 ? o | x << 16 : x | o << 16);
    const unsigned p = lane_of<XOR2>(w);
    const u64 all = lane & 2 ? p | (u64)w << 32 : w | (u64)p << 32;
    const int n = a.Hq * HEAD;
    put(reinterpret_cast<u64*>(exchange(l) + a.at.att) +
            (((d & 3) * a.M + b) * n + h * HEAD + d) / 4,
        all);
  }
  // Splits of heads, which the slots of a key head share out. [split][HEAD] and [split] of
  // (maximum, sum).
  DEVINL bool merge_parts(int l, const Split& s) {
    const int G = a.Hq / a.Hkv;
    for (int g = s.split; g < G; g += s.parts) {
      meet();      // the LDS of what came before is free
      const unsigned* src = part_of(l, s, g);
      float* to = reinterpret_cast<float*>(wide());
      fetch(src, wide(), s.parts * HEAD);
      // up to three key heads may have more splits than a wave has lanes
      for (int i0 = 0; wave == NW - 1 && i0 < s.parts; i0 += WAVE) {
        const int i = i0 + lane;
        const u64* ml =
            reinterpret_cast<const u64*>(src + a.parts * HEAD) + min(i, s.parts - 1);
        u64 got;
        int looks = 0;
        do got = peek(ml);
        while (__builtin_amdgcn_ballot_w64(!there(got)) && patient(looks));
        if (!there(got)) ctl->late[flag] = 1;
        if (i < s.parts) reinterpret_cast<u64*>(to + s.parts * HEAD)[i] = got;
      }
      meet();
      if (late()) return false;
      if (tid < HEAD) {
        const float* ml = to + s.parts * HEAD;
        float mx = NEG_BIG, lt = 0.f, o = 0.f;
        for (int i = 0; i < s.parts; ++i) mx = fmaxf(mx, ml[2 * i]);
        for (int i = 0; i < s.parts; ++i) {
          const float c = fast_exp2(ml[2 * i] - mx);
          lt += ml[2 * i + 1] * c;
          o += to[i * HEAD + tid] * c;
        }
        put_head(l, s.b, s.head * G + g, tid, lt > 0.f ? o * (1.f / lt) : 0.f);
      }
      flag ^= 1;
    }
    return true;
  }

  // ---- all slots of the list, step by step; those behind come first
  DEVINL void catch_up() {
    typedef typename Sizes::AnyRows Rows;
    typedef typename Sizes::AnyPairs Pairs;
    static_assert(Sizes::Qkv::UNITS % Rows::UNITS == 0 && Sizes::O::UNITS % Rows::UNITS == 0 &&
                      Sizes::Down::UNITS % Rows::UNITS == 0 &&
                      Sizes::Glu::UNITS % Pairs::UNITS == 0,
                  "partial sums");
    const int end = a.layers * STEPS;
    while (!__builtin_amdgcn_readfirstlane(ctl->fail)) {
      const int n = __builtin_amdgcn_readfirstlane(ctl->count);
      int p = end;
      for (int i = 0; i < n; ++i)
        p = min(p, __builtin_amdgcn_readfirstlane(ctl->next[i]));
      if (p == end) return;
      const int l = p / STEPS, step = p % STEPS;
      const Layer w = layer_of(l);
      bool ok = true, fetched = false;
      for (int i = 0; i < n && ok; ++i) {
        if (__builtin_amdgcn_readfirstlane(ctl->next[i]) != p) continue;
        const int slot = __builtin_amdgcn_readfirstlane(ctl->slot[i]);
        // without work in this step: what would be looked up for it takes microseconds
        if (step == 1 || step == 2
                ? slot >= a.M * a.Hkv * parts || (step == 2 && parts == 1)
                : slot < spared)
          continue;
        meet();      // the LDS of the slot before is free
        fresh();
        Rows rows;
        Pairs pairs;
        // what one slot has fetched of a product's rows is there for the others
        if (step == 0) {
          rows.begin(qkv_job(w, slot), wave, lane);
          if (!fetched) fetch_hidden(l, slot);
          ok = run_qkv(l, qkv_job(w, slot), rows);
        } else if (step == 1 || step == 2) {
          const Split s = split_of(slot);
          if (!s.any) continue;
          if (step == 2) {
            ok = s.parts == 1 || merge_parts(l, s);
          } else {
            Tile t = {};
            load_tile(t, w, s);
            ok = fetch_heads(l, w, s, t.norm);
            if (ok) attend(l, w, s, t);
          }
        } else if (step == 3) {
          rows.begin(o_job(w, slot), wave, lane);
          if (!fetched) {
            fetch_hidden(l, slot);      // the residual
            fetch_attention(l, slot);
          }
          ok = run_o(l, o_job(w, slot), rows);
        } else if (step == 4) {
          pairs.begin(glu_job(w, slot), wave, lane);
          if (!fetched) fetch_h2(l, slot);
          ok = run_glu(l, glu_job(w, slot), pairs);
        } else {
          rows.begin(down_job(w, slot), wave, lane);
          if (!fetched) {
            fetch_h2(l, slot);
            fetch_mid(l, slot);
          }
          ok = run_down(l, down_job(w, slot), rows);
        }
        fetched = true;
      }
      if (!ok) {
        claim_idle();
        continue;
      }
      meet();
      if (tid < n && ctl->next[tid] == p)
        ctl->next[tid] =
            tid && step == STEPS - 1 && relieved(ctl->slot[tid], p + 1) ? end : p + 1;
      meet();
    }
  }

  // ---- one slot, to the end. False: something was late (or the launch has failed), after
  // that many steps; what has to be done from there on is done by catch_up(). To do a step
  // again here would cost every step: loads in flight are counted only on straight ways. To
  // come back here for the next layer takes registers (drafter 407 us for 390).
  // EARLY: the weights of a layer's other products are asked for behind the first one's
  // results, to come while attention is waited for, those of the next layer's first one
  // behind the others' results, no more at a time than an exchange takes. Otherwise those
  // of the next step behind a step's results.
  template <bool ATTENDS>
  DEVINL bool go(int slot, int& done) {
    constexpr bool EARLY = Sizes::EARLY;
    Layer w = layer_of(0);
    typename Sizes::Qkv qkv;
    typename Sizes::O o;
    typename Sizes::Glu glu;
    typename Sizes::Down down;
    Split s;
    Tile tile;
    if constexpr (ATTENDS) s = split_of(slot);
    qkv.begin(qkv_job(w, slot), wave, lane);
    for (int l = 0; l < a.layers; ++l) {
      done = l * STEPS;
      const Job jo = o_job(w, slot), jg = glu_job(w, slot), jd = down_job(w, slot);
      const Layer following = layer_of(min(l + 1, a.layers - 1));
      const Job jq = qkv_job(following, slot);
      fresh();
      fetch_hidden(l, slot);
      if (!run_qkv(l, qkv_job(w, slot), qkv)) return false;
      if constexpr (ATTENDS) load_tile(tile, w, s);
      o.begin(jo, wave, lane);
      if constexpr (EARLY && !ATTENDS) {
        glu.begin(jg, wave, lane);
        down.begin(jd, wave, lane);
      }
      if constexpr (ATTENDS) {
        done = l * STEPS + 1;
        fresh();
        if (!fetch_heads(l, w, s, tile.norm)) return false;
        attend(l, w, s, tile);
        done = l * STEPS + 2;
        fresh();
        if (s.parts > 1 && !merge_parts(l, s)) return false;
        meet();      // the LDS of attention is free
        if constexpr (EARLY) glu.begin(jg, wave, lane);
      }
      done = l * STEPS + 3;
      fresh();
      fetch_attention(l, slot);
      if (!run_o(l, jo, o)) return false;
      if constexpr (EARLY && ATTENDS) down.begin(jd, wave, lane);
      if constexpr (EARLY && !ATTENDS) qkv.template begin_units<0, 3>(jq, wave, lane);
      if constexpr (!EARLY) glu.begin(jg, wave, lane);
      done = l * STEPS + 4;
      fresh();
      fetch_h2(l, slot);
      if (!run_glu(l, jg, glu)) return false;
      if constexpr (EARLY && ATTENDS) qkv.begin(jq, wave, lane);
      if constexpr (EARLY && !ATTENDS) qkv.template begin_units<3, 6>(jq, wave, lane);
      if constexpr (!EARLY) down.begin(jd, wave, lane);
      done = l * STEPS + 5;
      fresh();
      fetch_mid(l, slot);
      if (!run_down(l, jd, down)) return false;
      if constexpr (EARLY && !ATTENDS) qkv.template begin_units<6, 8>(jq, wave, lane);
      if constexpr (!EARLY) qkv.begin(jq, wave, lane);
      w = following;
    }
    return true;
  }
  // of a slot that has nothing but attention
  DEVINL bool go_attention(int slot, int& done) {
    Layer w = layer_of(0);
    const Split s = split_of(slot);
    Tile tile;
    load_tile(tile, w, s);
    for (int l = 0; l < a.layers; ++l) {
      done = l * STEPS + 1;
      const Layer following = layer_of(min(l + 1, a.layers - 1));
      fresh();
      if (!fetch_heads(l, w, s, tile.norm)) return false;
      attend(l, w, s, tile);
      done = l * STEPS + 2;
      fresh();
      if (s.parts > 1 && !merge_parts(l, s)) return false;
      load_tile(tile, following, s);
      meet();      // the LDS of attention is free
      w = following;
    }
    done = a.layers * STEPS;
    return true;
  }
};

template <class Sizes>
__global__ __launch_bounds__(NT, 2) void decode_span_kernel(const Args a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  Worker<Sizes> w(a, lds);
  if (w.tid == 0) {
    w.ctl->got = w.begins(blockIdx.x);
    w.ctl->late[0] = w.ctl->late[1] = w.ctl->rounds = w.ctl->fail = 0;
    w.ctl->count = 1;
    w.ctl->slot[0] = (short)blockIdx.x;
  }
  for (int i = w.tid; i < a.layers * (int)sizeof(Layer) / 16; i += NT)
    reinterpret_cast<uint4v*>(w.ctl->layer)[i] =
        reinterpret_cast<const uint4v*>(a.layer)[i];
  meet();
  if (!__builtin_amdgcn_readfirstlane(w.ctl->got)) return;
  int done = 0;
  const int slot = blockIdx.x;
  const bool attends = w.split_of(slot).any;
  if (attends && slot < w.spared) {
    if (w.go_attention(slot, done)) return;
  } else if (slot < w.spared) {
    return;      // its sequence is shorter than others
  } else if (attends) {
    if (w.template go<true>(slot, done)) return;
  } else {
    if (w.template go<false>(slot, done)) return;
  }
  w.claim_idle();
  if (w.tid == 0) w.ctl->next[0] = done;
  meet();
  w.catch_up();
  // nothing of this is known to happen: what is not there is not a number
  if (w.ctl->fail)
    for (int i = w.tid; i < a.M * a.H; i += NT) a.out[i] = 0x7fff;
}

// words of ones behind SLOTS of zeros
__global__ __launch_bounds__(256) void decode_span_fill_kernel(uint4* work, long n) {
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    const unsigned v = i < SLOTS / 4 ? 0u : ~0u;
    work[i] = make_uint4(v, v, v, v);
  }
}

}  // namespace span
