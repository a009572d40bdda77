// Prefill (multi-token) paged attention for gfx950 — flash-style on MFMA.
//
// Replaces the reference's mha_llama prefill path
// (flexgen_utils/pytorch_backend.py:665-731), reading K/V directly from the
// paged cache (new tokens are kv_write'n first, then attended — one code path
// for first-prefill, multi-turn continuation, chunked prefill and the tree
// steps of speculative decoding).
//
// Rows are (token, head of the group) pairs, so that a K/V tile serves all heads
// that share it; a wave owns 32 rows, a workgroup 128. Tiles of 64 keys go to LDS
// without passing through registers, double-buffered.
//
// Both products run transposed on v_mfma_f32_32x32x16_bf16: S^T = K Q^T, then
// O^T = V^T P^T. The keys of a tile lie in LDS in an order (bits 2 and 3 of a key's
// number swapped) in which the 16 scores a lane gets are the eight consecutive keys
// it must hand to each of two value products: the weights never leave registers, a
// row's maximum takes one exchange between the halves of a wave, and its sum none
// until the end.
//
// The matrix cores bound long prompts (a tile is 32 products of 32 clocks a wave,
// and its softmax about as many clocks on the vector units, which two waves a SIMD
// overlap); the chain of tiles bounds short ones, so there the keys are shared out to two
// groups of waves of a workgroup, whose sums meet in LDS, and split over workgroups, whose
// parts a second kernel folds.
//
// Measured, 32 heads on 8 of 128, a call of several in a graph: four prompts of 4096 592 us
// (930 TF/s of the visible half; 642 with an address a lane, 3808 with 16-row tiles of one
// head each, staged through registers, weights through LDS; 674 in a step, whose products
// leave less power), 2000 tokens behind 6000 250 us (277 with an address a lane), one of 333
// behind 1201 33 us (36 with an address a lane and one group a workgroup), a tree of 25
// behind 1500 18.2 us. Of 625 us for the first in another session the loads alone took 293:
// what is left overlaps by half. Scores a tile ahead of the weights within a wave took 686
// there, 256 rows a workgroup 641 (loads 172).
//
// Numerics: fp32 softmax/accum; bf16 operands — matches reference tolerance
// class (test_block_exact_match.py atol 1e-4 forward on fp32 inputs).

#include "common.h"

struct PrefillArgs {
  const unsigned short* q;        // (b, token, head) at the strides below
  const unsigned short* k_pages;  // (np, Hkv, P, D)
  const unsigned short* v_pages;  // (np, Hkv, D, P)
  const int* page_table;          // (B, maxp)
  const int* q_start;             // (B,)
  const float* alibi;             // (Hq,) slopes or null
  const unsigned char* tree_mask; // (B, Tq, Tq) bool or null: spec-verify ancestor
                                  // mask over the NEW tokens (ref
                                  // backend.py:944-1047); committed positions
                                  // < q_start stay fully visible
  unsigned short* out;
  float* pml;                     // splits: (n_split, B * Hkv, Tq * G, 2)
  float* pacc;                    // (n_split, B * Hkv, Tq * G, D)
  int B, Hkv, G, Tq, P, maxp, window, n_split;
  int p_log2;                     // of P where it is a power of two
  float scale;
  long q_sb, q_st, q_sh, o_sb, o_st, o_sh;
};

template <int D>
struct PrefillTile {
  static constexpr int KT = 64, RC = D / 8;       // 16 B pieces of a key row
  static constexpr int KB = KT * D * 2;           // bytes of K, and of V
  static constexpr int BYTES = 2 * KB;
  static constexpr int NI = KB / 1024 / 4;        // loads of a wave, K or V
  // piece c of LDS row r lies at c ^ swizzle(r): 16 rows read at one piece cover
  // all banks
  DEVINL static int swizzle(int r) {
    return RC >= 16 ? r & 15 : RC == 8 ? (r >> 1) & 7 : (r >> 2) & 3;
  }
};

// Where values beyond the last key come from: weights of zero meet them, which a value
// that is not finite would turn into NaN.
__device__ const unsigned short prefill_zeros[8] __attribute__((aligned(16))) = {};

// GENERAL: slopes, scales that are not positive; TREE: these and tree masks, whose code
// in between took slopes as long as it did trees (two tokens, 16 heads of 64: 7.4 us, 5.6
// apart).
enum PrefillForm { PREFILL_PLAIN, PREFILL_GENERAL, PREFILL_TREE };

// A load brings keys (values) of one group of sixteen. GROUPS: pages hold a power of two of
// keys, 16 or more, so that a load's page is the wave's. EIGHTS: of 8, which a lane looks up
// for itself; MIXED: not a power of two. Forms of their own, since even the choice costs
// where a lane finds pages by shifts (0.75 us of a tree's 18).
enum PrefillPages { PREFILL_GROUPS, PREFILL_EIGHTS, PREFILL_MIXED };

// KG groups of four waves share out the keys of a workgroup; what each of two has found
// meets in LDS.
template <int D, int FORM, int PAGES, int KG>
__global__ __launch_bounds__(256 * KG, D > 128 ? 1 : 2) void attn_prefill_kernel(
    PrefillArgs a) {
  using Tile = PrefillTile<D>;
  constexpr int KT = Tile::KT, RC = Tile::RC, NI = Tile::NI;
  constexpr int NKK = D / 16, ND = D / 32;
  constexpr bool GENERAL = FORM != PREFILL_PLAIN, DIVIDE = PAGES == PREFILL_MIXED;
  constexpr bool LANES = PAGES != PREFILL_GROUPS;
  static_assert(NI >= 1, "tile smaller than the workgroup");
  extern __shared__ __attribute__((aligned(16))) unsigned char prefill_lds[];

  // consecutive workgroups take different (sequence, head group, split) units, so
  // that the row tiles of one unit meet in one XCD's L2 (units are a multiple of 8
  // where the heads are); late rows see the most keys and go first
  const int units = a.B * a.Hkv;
  const int unit = blockIdx.x % units, split = blockIdx.x / units;
  const int b = unit / a.Hkv, g = unit % a.Hkv;
  const int G = a.G, R = a.Tq * G;
  const int base = (int)(gridDim.y - 1 - blockIdx.y) * 128;
  const int tid = threadIdx.x;
  const int any = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wave = KG > 1 ? any % 4 : any, group = KG > 1 ? any / 4 : 0;
  unsigned char* const lds = prefill_lds + group * (2 * Tile::BYTES);
  const int lane = tid & (WAVE - 1);
  const int li = lane & 31, hi = lane >> 5;
  const int qs = a.q_start[b];
  const bool tree = FORM == PREFILL_TREE && a.tree_mask != nullptr;
  const int plog = PAGES == PREFILL_EIGHTS ? 3 : a.p_log2, pmask = (1 << plog) - 1;
  auto page_of = [&](int pos) { return DIVIDE ? pos / a.P : pos >> plog; };
  auto slot_of = [&](int pos) { return DIVIDE ? pos % a.P : pos & pmask; };
  auto first_of = [&](long page) { return DIVIDE ? page * a.P : page << plog; };
  const int* table = a.page_table + (long)b * a.maxp;

  // this lane's row (column of S^T)
  const int row = base + wave * 32 + li;
  const int r = min(row, R - 1);
  const int tok = r / G, head = g * G + r % G, qpos = qs + tok;
  const unsigned short* qp =
      a.q + (long)b * a.q_sb + (long)tok * a.q_st + (long)head * a.q_sh + hi * 8;
  bf16x8 qf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)
    qf[kk] = as_bf16x8(*reinterpret_cast<const short8*>(qp + kk * 16));
  const float sc2 = a.scale * LOG2E;
  const float slope2 = GENERAL && a.alibi ? a.alibi[head] * LOG2E : 0.f;
  const unsigned char* mask =
      tree ? a.tree_mask + ((long)b * a.Tq + tok) * a.Tq : nullptr;

  // keys the workgroup and this wave see; tree nodes may see any new token
  const int last = min(base + 128, R) - 1;
  const int kend = tree ? qs + a.Tq : qs + last / G + 1;
  const int kbeg =
      a.window > 0 ? max(0, qs + base / G - a.window + 1) & ~(KT - 1) : 0;
  const int w0 = base + wave * 32, w1 = min(w0 + 31, R - 1);
  const int wlast = w0 >= R ? -1 : tree ? kend - 1 : qs + w1 / G;
  const int wfirst = a.window > 0 ? qs + w0 / G - a.window + 1 : 0;
  // tiles in [ilo, ihi] need no mask
  const int ihi = tree ? qs - 1 : qs + w0 / G;
  const int ilo = a.window > 0 ? qs + w1 / G - a.window + 1 : 0;
  const int sees = a.window > 0 ? a.window : 0x7fffffff;

  const int tiles = (kend - kbeg + KT - 1) / KT;
  const int per = (tiles + a.n_split - 1) / a.n_split;
  const int turns = (per + KG - 1) / KG;         // tiles of a group
  const int u0 = kbeg + split * per * KT, u1 = min(kend, u0 + per * KT);
  const int t0 = u0 + group * turns * KT;
  const int t1 = KG == 1 ? u1 : min(u1, t0 + turns * KT);

  // Where this lane's pieces come from. Load i of a wave brings pieces of keys (values) of
  // group group_of(i) of sixteen: of the wave's page, at offsets that are the same in every
  // tile. (An address a lane took 139 vector instructions a tile, some of them four times
  // as long as others; the softmax takes 105.)
  int kkey[NI], kcol[NI], vkey[NI], vrow[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int at = (wave + i * 4) * 64 + lane;
    const int lr = at / RC;
    kcol[i] = ((at % RC) ^ Tile::swizzle(lr)) * 8;
    kkey[i] = (lr & ~12) | ((lr & 4) << 1) | ((lr & 8) >> 1);
    vkey[i] = at / (2 * D) * 16 + (at & 1) * 8;   // groups of 16 keys, (d, octet)
    vrow[i] = at % (2 * D) / 2;
  }
  static_assert(64 / RC <= 16 && 2 * D >= 64, "a load is of one group");
  auto group_of = [&](int i) { return (wave + i * 4) * 32 / D * 16; };
  constexpr int OFS = 256 / RC % 16 ? 2 : 1;      // loads of different offsets
  static_assert(OFS == (256 % (2 * D) ? 2 : 1), "values as keys");
  unsigned kofs[OFS], vofs[OFS];
#pragma unroll
  for (int i = 0; i < OFS; ++i) {
    kofs[i] = (unsigned)((kkey[i] & 15) * D + kcol[i]) * 2;
    vofs[i] = (unsigned)(vrow[i] * a.P + (lane & 1) * 8) * 2;
  }
  // nothing writes the table meanwhile: scalar loads
  const auto* pages = (const __attribute__((address_space(4))) int*)table;
  int kpage[NI], vpage[NI];      // of the tile that is asked for next
  auto look_up = [&](int kb) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (LANES) {
        kpage[i] = table[page_of(min(kb + kkey[i], kend - 1))];
        vpage[i] = table[page_of(min(kb + vkey[i], kend - 1))];
      } else {
        kpage[i] = vpage[i] = pages[page_of(min(kb + group_of(i), kend - 1))];
      }
    }
  };
  auto issue = [&](int kb, unsigned char* buf) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      unsigned char* to = buf + (wave + i * 4) * 1024;
      if constexpr (LANES) {
        const int pos = slot_of(min(kb + kkey[i], kend - 1));
        copy16_to_lds(a.k_pages + (first_of((long)kpage[i] * a.Hkv + g) + pos) * D +
                          kcol[i],
                      to);
      } else {
        // keys behind the last one are masked
        const int at = (kb + group_of(i)) & pmask;
        dma16(a.k_pages + (first_of((long)kpage[i] * a.Hkv + g) + at) * D, kofs[i % OFS],
              (unsigned)(unsigned long)(lptr_t)to);
      }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      unsigned char* to = buf + Tile::KB + (wave + i * 4) * 1024;
      const unsigned short* head = a.v_pages + first_of(((long)vpage[i] * a.Hkv + g) * D);
      if constexpr (LANES) {
        const unsigned short* src = head + first_of(vrow[i]) + slot_of(kb + vkey[i]);
        if (kb + vkey[i] >= kend) src = prefill_zeros;
        copy16_to_lds(src, to);
      } else {
        head += (kb + group_of(i)) & pmask;
        if (kb + KT > kend) {
          const unsigned short* src = head + vofs[i % OFS] / 2;
          if (kb + group_of(i) + (lane & 1) * 8 >= kend) src = prefill_zeros;
          dma16_to_lds(src, to);
        } else {
          dma16(head, vofs[i % OFS], (unsigned)(unsigned long)(lptr_t)to);
        }
      }
    }
  };

  float m = NEG_BIG, l = 0.f;   // maximum of the unscaled scores, this half's sum
  f32x16 acc[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) acc[n] = f32x16{};
  const int sw = Tile::swizzle(li);
  const int krow = li * (D * 2);

  auto compute = [&](int kb, const unsigned char* kt) {
    // keys a tree's row does not see, element n * 16 + j of s below; ahead of the scores,
    // whose registers the entries take meanwhile, and eight at a time, so that their loads
    // overlap (25 tokens behind 1500: 1.3 us longer one by one)
    unsigned dead = 0;
    if (tree && kb + KT - 1 > ihi) {
      const int k0 = kb + hi * 8 - qs;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        unsigned char seen[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          seen[e] = mask[min(max(k0 + q * 16 + e, 0), a.Tq - 1)];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = k0 + q * 16 + e;
          if (k >= a.Tq || (k >= 0 && !seen[e])) dead |= 1u << (q * 8 + e);
        }
      }
    }
    f32x16 s[2];
    s[0] = s[1] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const bf16x8 kf = as_bf16x8(*reinterpret_cast<const short8*>(
            kt + n * (32 * D * 2) + krow + (((kk * 2 + hi) ^ sw) << 4)));
        s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kk], s[n], 0, 0, 0);
      }
    // s[n][j] is key kb + n * 32 + (j & 8) * 2 + hi * 8 + (j & 7)
    if (GENERAL) {
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          s[n][j] = s[n][j] * sc2 +
                    slope2 * (float)(kb + n * 32 + (j & 8) * 2 + hi * 8 + (j & 7));
    }
    if (kb < ilo || kb + KT - 1 > ihi) {
      if (tree) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (dead >> (n * 16 + j) & 1) s[n][j] = NEG_BIG;
      } else {
        const int d0 = qpos - kb - hi * 8;
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int dist = d0 - (n * 32 + (j & 8) * 2 + (j & 7));
            if (dist < 0 || dist >= sees) s[n][j] = NEG_BIG;
          }
      }
    }
    float mx = m;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s[n][j]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float f = GENERAL ? 1.f : sc2;
    if (__builtin_amdgcn_ballot_w64(mx > m)) {
      const float corr = fast_exp2((m - mx) * f);
      l *= corr;
#pragma unroll
      for (int n = 0; n < ND; ++n)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[n][j] *= corr;
      m = mx;
    }
    // a row that has seen nothing yet keeps weights of zero
    const float ref = m > 0.5f * NEG_BIG ? m * f : 0.f;
    bf16x8 pf[4];
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float p = fast_exp2(fmaf(s[n][j], f, -ref));
        ps[n] += p;
        pf[n * 2 + (j >> 3)][j & 7] = (__bf16)p;
      }
    l += ps[0] + ps[1];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const bf16x8 vf = as_bf16x8(*reinterpret_cast<const short8*>(
            kt + Tile::KB + j * (D * 32) + (n * 32 + li) * 32 + hi * 16));
        acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[j], acc[n], 0, 0, 0);
      }
  };

  // every group takes as many turns as the first one, which has most tiles
  const int stop = KG == 1 ? t1 : t0 + min(u1 - u0, turns * KT);
  if (u0 < u1) {
    // page numbers are looked up a tile ahead of the loads that need them
    if (KG == 1 || t0 < t1) {
      look_up(t0);
      issue(t0, lds);
      look_up(t0 + KT);
    }
    if (!LANES) wait_loads<0>();
    __syncthreads();
    int buf = 0;
    for (int kb = t0; kb < stop; kb += KT) {
      if (kb + KT < t1) {
        issue(kb + KT, lds + (buf ^ 1) * Tile::BYTES);
        look_up(kb + 2 * KT);
      }
      if ((KG == 1 || kb < t1) && kb <= wlast && kb + KT > wfirst)
        compute(kb, lds + buf * Tile::BYTES);
      if (!LANES) wait_loads<0>();
      __syncthreads();
      buf ^= 1;
    }
  }
  if (KG == 2 && u0 + turns * KT >= u1) {
    if (group) return;      // it had no keys
  } else if constexpr (KG == 2) {
    // what the second group has found goes to the first
    static_assert(4 * (ND * 16 + 2) * 256 <= 4 * Tile::BYTES, "place");
    float* at = reinterpret_cast<float*>(prefill_lds) + wave * (ND * 16 + 2) * 64 + lane;
    if (group) {
#pragma unroll
      for (int n = 0; n < ND; ++n)
#pragma unroll
        for (int j = 0; j < 16; ++j) at[(n * 16 + j) * 64] = acc[n][j];
      at[ND * 16 * 64] = m;
      at[(ND * 16 + 1) * 64] = l;
    }
    __syncthreads();
    if (group) return;
    const float m2 = at[ND * 16 * 64], l2 = at[(ND * 16 + 1) * 64];
    const float f = GENERAL ? 1.f : sc2, mx = fmaxf(m, m2);
    const float c = fast_exp2((m - mx) * f), c2 = fast_exp2((m2 - mx) * f);
    l = l * c + l2 * c2;
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int j = 0; j < 16; ++j)
        acc[n][j] = acc[n][j] * c + at[(n * 16 + j) * 64] * c2;
    m = mx;
  }

  // a row's values are spread over the two lanes of its column
  l += __shfl_xor(l, 32);
  if (row >= R) return;
  if (a.n_split > 1) {
    const long at = ((long)split * units + unit) * R + r;
    if (hi == 0) {
      a.pml[at * 2] = GENERAL ? m : m * sc2;
      a.pml[at * 2 + 1] = l;
    }
    if (l != 0.f) {   // NaN sums, too: the fold is to see them
#pragma unroll
      for (int n = 0; n < ND; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *reinterpret_cast<f32x4*>(a.pacc + at * D + n * 32 + j * 8 + hi * 4) =
              f32x4{acc[n][j * 4], acc[n][j * 4 + 1], acc[n][j * 4 + 2],
                    acc[n][j * 4 + 3]};
    }
    return;
  }
  const float inv = l != 0.f ? 1.f / l : 0.f;
  unsigned short* op =
      a.out + (long)b * a.o_sb + (long)tok * a.o_st + (long)head * a.o_sh + hi * 4;
#pragma unroll
  for (int n = 0; n < ND; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      short4v o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (short)f2bf(acc[n][j * 4 + e] * inv);
      *reinterpret_cast<short4v*>(op + n * 32 + j * 8) = o;
    }
}

// Folds the splits of a row, four columns a thread, which asks for all of C splits at once:
// their maxima and sums with their values, that none waits for another. A split that saw
// nothing has a sum of zero and left its values unwritten; a NaN in a split makes the row
// NaN. grid: rows of all units * D / 4 / 256. us of attention in a graph, 32 heads
// of 128 on 8, with a wave a row that shares out the weights first, and so: 333 tokens
// behind 1201 33.9, 31.6; 17 behind 8000 26.1, 20.4; 2 behind 8000 23.4, 16.4; a tree of 25
// behind 1500 18.0, 15.9; 4 x 8 behind 2000 17.3, 15.2. (Decode's folds, of up to 32 parts
// of fewer rows, are faster with a wave a row: one context of 4000 12.3, 14.3.)
template <int D, int C>
__global__ __launch_bounds__(256) void attn_prefill_fold_kernel(PrefillArgs a) {
  constexpr int L = D / 4;                   // threads of a row
  const int units = a.B * a.Hkv, R = a.Tq * a.G;
  const long rows = (long)units * R;
  const long item = (long)blockIdx.x * 256 + threadIdx.x, at = item / L;
  const int col = (int)(item % L) * 4;
  if (at >= rows) return;
  float m = NEG_BIG, l = 0.f;
  f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < a.n_split; s0 += C) {
    f32x4 v[C];
    float ms[C], ls[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const long row = min(s0 + i, a.n_split - 1) * rows + at;
      ms[i] = a.pml[row * 2];
      ls[i] = a.pml[row * 2 + 1];
      v[i] = *reinterpret_cast<const f32x4*>(a.pacc + row * D + col);
    }
    float top = m;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      if (s0 + i >= a.n_split) ls[i] = 0.f;
      if (ls[i] != 0.f) top = fmaxf(top, ms[i]);
    }
    const float keep = fast_exp2(m - top);
    l *= keep;
    o *= keep;
    m = top;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      if (ls[i] == 0.f) continue;
      const float w = fast_exp2(ms[i] - top);
      l += w * ls[i];
      o += w * v[i];
    }
  }
  const float inv = l != 0.f ? 1.f / l : 0.f;
  const int unit = (int)(at / R), r = (int)(at % R);
  unsigned short* op = a.out + (long)(unit / a.Hkv) * a.o_sb +
                       (long)(r / a.G) * a.o_st +
                       (long)(unit % a.Hkv * a.G + r % a.G) * a.o_sh + col;
  short4v y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = (short)f2bf(o[e] * inv);
  *reinterpret_cast<short4v*>(op) = y;
}
