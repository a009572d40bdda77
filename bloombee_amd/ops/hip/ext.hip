// Torch extension bindings for the bloombee_amd gfx950 kernel library.
// Host-side shape checks, template dispatch, and stream plumbing only —
// all compute lives in the .hip translation units.

#include <torch/extension.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <cstdlib>

#include "common.h"

// Single translation unit: the template kernels must be visible at their
// launch sites for instantiation.
#include "elementwise.hip"
#include "kvcache.hip"
#include "attn_decode.hip"
#include "attn_decode_mfma.hip"
#include "attn_prefill.hip"
#include "gemm_skinny.hip"
#include "gemm_stream.hip"
#include "gemm_rows_host.h"
#include "gemm_rows_rope.hip"
#include "moe_gemm.hip"
#include "moe_route.hip"
#include "w4_gemm.hip"
#include "mfma_selftest.hip"
#include "quant4.hip"
#include "wire.h"

typedef __attribute__((ext_vector_type(8))) short short8_h;

#define CHECK_DEV(x) TORCH_CHECK(x.is_cuda(), #x " must be on device")
// a CPU tensor pointer reaching a kernel is a GPU memory fault at a random
// later point — check EVERY tensor argument, not just the big ones
#define CHECK_DEV_ALL1(a) CHECK_DEV(a)
#define CHECK_DEV_ALL2(a, b) { CHECK_DEV(a); CHECK_DEV(b); }
#define CHECK_DEV_ALL3(a, b, c) { CHECK_DEV(a); CHECK_DEV(b); CHECK_DEV(c); }
#define CHECK_BF16(x) TORCH_CHECK(x.scalar_type() == at::kBFloat16, #x " must be bf16")
#define CHECK_CONTIG(x) TORCH_CHECK(x.is_contiguous(), #x " must be contiguous")

static inline const unsigned short* bf_ptr(const torch::Tensor& t) {
  return reinterpret_cast<const unsigned short*>(t.data_ptr());
}
static inline unsigned short* bf_ptr_mut(torch::Tensor& t) {
  return reinterpret_cast<unsigned short*>(t.data_ptr());
}
static inline hipStream_t cur_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

// ---------------------------------------------------------------------------
// norms
// ---------------------------------------------------------------------------

template <typename F>
static void dispatch_iters(int H, F f) {
  constexpr int BLOCK = 256;
  const int per_iter = BLOCK * 8;
  if (H <= per_iter) f(std::integral_constant<int, 1>{});
  else if (H <= 2 * per_iter) f(std::integral_constant<int, 2>{});
  else if (H <= 4 * per_iter) f(std::integral_constant<int, 4>{});
  else if (H <= 8 * per_iter) f(std::integral_constant<int, 8>{});
  else TORCH_CHECK(false, "hidden size too large for norm kernel: ", H);
}

torch::Tensor rms_norm(torch::Tensor x, torch::Tensor w, double eps) {
  CHECK_DEV(x); CHECK_BF16(x); CHECK_CONTIG(x);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H must be a multiple of 8");
  const long N = x.numel() / H;
  auto y = torch::empty_like(x);
  dispatch_iters(H, [&](auto iters) {
    rmsnorm_kernel<256, decltype(iters)::value><<<N, 256, 0, cur_stream()>>>(
        bf_ptr(x), nullptr, bf_ptr(w), nullptr, bf_ptr_mut(y), H, (float)eps);
  });
  return y;
}

std::vector<torch::Tensor> rms_norm_residual(torch::Tensor x, torch::Tensor res,
                                             torch::Tensor w, double eps) {
  CHECK_DEV(x); CHECK_BF16(x); CHECK_CONTIG(x); CHECK_CONTIG(res);
  const int H = x.size(-1);
  const long N = x.numel() / H;
  auto h = torch::empty_like(x);
  auto y = torch::empty_like(x);
  dispatch_iters(H, [&](auto iters) {
    rmsnorm_kernel<256, decltype(iters)::value><<<N, 256, 0, cur_stream()>>>(
        bf_ptr(x), bf_ptr(res), bf_ptr(w), bf_ptr_mut(h), bf_ptr_mut(y), H,
        (float)eps);
  });
  return {h, y};
}

torch::Tensor layer_norm(torch::Tensor x, torch::Tensor w,
                         c10::optional<torch::Tensor> bias, double eps) {
  CHECK_DEV(x); CHECK_BF16(x); CHECK_CONTIG(x);
  const int H = x.size(-1);
  const long N = x.numel() / H;
  auto y = torch::empty_like(x);
  const unsigned short* bp = bias.has_value() ? bf_ptr(*bias) : nullptr;
  dispatch_iters(H, [&](auto iters) {
    layernorm_kernel<256, decltype(iters)::value><<<N, 256, 0, cur_stream()>>>(
        bf_ptr(x), nullptr, bf_ptr(w), bp, nullptr, bf_ptr_mut(y), H, (float)eps);
  });
  return y;
}

// ---------------------------------------------------------------------------
// rope / activations
// ---------------------------------------------------------------------------

void rope_apply_(torch::Tensor q, torch::Tensor k, torch::Tensor cos_t,
                 torch::Tensor sin_t, torch::Tensor pos) {
  CHECK_DEV(q); CHECK_BF16(q); CHECK_CONTIG(q); CHECK_CONTIG(k);
  CHECK_DEV_ALL3(cos_t, sin_t, pos);
  TORCH_CHECK(pos.scalar_type() == at::kInt, "pos must be int32");
  const int B = q.size(0), Hq = q.size(1), T = q.size(2), D = q.size(3);
  const int Hkv = k.size(1);
  TORCH_CHECK(cos_t.scalar_type() == at::kFloat && cos_t.size(1) == D / 2);
  dim3 grid(B * T, Hq + Hkv);
  rope_kernel<<<grid, 64, 0, cur_stream()>>>(
      bf_ptr_mut(q), bf_ptr_mut(k), cos_t.data_ptr<float>(),
      sin_t.data_ptr<float>(), pos.data_ptr<int>(), B, Hq, Hkv, T, D,
      (int)cos_t.size(0));
}

torch::Tensor swiglu(torch::Tensor gu) {
  CHECK_DEV(gu); CHECK_BF16(gu); CHECK_CONTIG(gu);
  const long I = gu.size(-1) / 2;
  const long N = gu.numel() / (2 * I);
  TORCH_CHECK(I % 8 == 0);
  auto sizes = gu.sizes().vec();
  sizes.back() = I;
  auto out = torch::empty(sizes, gu.options());
  const long nvec = N * (I / 8);
  const int grid = (int)std::min<long>((nvec + 255) / 256, 2048);
  swiglu_kernel<<<grid, 256, 0, cur_stream()>>>(bf_ptr(gu), bf_ptr_mut(out), N, I);
  return out;
}

torch::Tensor gelu_tanh(torch::Tensor x) {
  CHECK_DEV(x); CHECK_BF16(x); CHECK_CONTIG(x);
  auto out = torch::empty_like(x);
  const long nvec = x.numel() / 8;
  const int grid = (int)std::min<long>((nvec + 255) / 256, 2048);
  gelu_kernel<<<grid, 256, 0, cur_stream()>>>(bf_ptr(x), bf_ptr_mut(out), x.numel());
  return out;
}

torch::Tensor add_bf16(torch::Tensor a, torch::Tensor b) {
  CHECK_DEV(a); CHECK_BF16(a); CHECK_CONTIG(a); CHECK_CONTIG(b);
  auto out = torch::empty_like(a);
  const long nvec = a.numel() / 8;
  const int grid = (int)std::min<long>((nvec + 255) / 256, 2048);
  add_kernel<<<grid, 256, 0, cur_stream()>>>(bf_ptr(a), bf_ptr(b), bf_ptr_mut(out),
                                             a.numel());
  return out;
}

// ---------------------------------------------------------------------------
// paged KV
// ---------------------------------------------------------------------------

void kv_write(torch::Tensor k_new, torch::Tensor v_new, torch::Tensor k_pages,
              torch::Tensor v_pages, torch::Tensor page_table,
              torch::Tensor start_pos) {
  CHECK_DEV(k_new); CHECK_BF16(k_new); CHECK_CONTIG(k_new); CHECK_CONTIG(v_new);
  CHECK_CONTIG(k_pages); CHECK_CONTIG(v_pages);
  TORCH_CHECK(page_table.scalar_type() == at::kInt && start_pos.scalar_type() == at::kInt);
  CHECK_DEV_ALL2(page_table, start_pos);
  const int B = k_new.size(0), Hkv = k_new.size(1), T = k_new.size(2), D = k_new.size(3);
  const int P = k_pages.size(2), maxp = page_table.size(1);
  TORCH_CHECK(k_pages.size(1) == Hkv && k_pages.size(3) == D);
  TORCH_CHECK(v_pages.size(2) == D && v_pages.size(3) == P,
              "v_pages must be d-major (np, Hkv, D, P)");
  const int threads = std::min(256, Hkv * D / 8);
  kv_write_kernel<<<B * T, threads, 0, cur_stream()>>>(
      bf_ptr(k_new), bf_ptr(v_new), bf_ptr_mut(k_pages), bf_ptr_mut(v_pages),
      page_table.data_ptr<int>(), start_pos.data_ptr<int>(), B, Hkv, T, D, P, maxp);
}

std::vector<torch::Tensor> kv_gather(torch::Tensor k_pages, torch::Tensor v_pages,
                                     torch::Tensor page_table, long batch_index,
                                     long ctx) {
  CHECK_DEV(k_pages); CHECK_DEV(page_table);
  const int Hkv = k_pages.size(1), P = k_pages.size(2), D = k_pages.size(3);
  auto k = torch::empty({Hkv, ctx, D}, k_pages.options());
  auto v = torch::empty({Hkv, ctx, D}, v_pages.options());
  const long nvec = ctx * Hkv * (D / 8);
  const int grid = (int)std::min<long>((nvec + 255) / 256, 2048);
  kv_gather_kernel<<<grid, 256, 0, cur_stream()>>>(
      bf_ptr(k_pages), bf_ptr(v_pages), bf_ptr_mut(k), bf_ptr_mut(v),
      page_table.data_ptr<int>(), (int)batch_index, (int)ctx, Hkv, D, P,
      page_table.size(1));
  return {k, v};
}

// ---------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------

template <int D>
static void attn_decode_launch(const torch::Tensor& q, const torch::Tensor& kp,
                               const torch::Tensor& vp, const torch::Tensor& pt,
                               const torch::Tensor& ctx,
                               const float* alibi_ptr, torch::Tensor& out,
                               torch::Tensor& pml, torch::Tensor& pacc, int B,
                               int Hkv, int G, int nch, int P, int maxp,
                               int n_split, int window, float scale, long q_off,
                               long q_sb, long q_sh, long out_sb, long out_sh,
                               int ctx_add, int share, bool wide) {
  dim3 grid(B * Hkv * nch, n_split);
  const int maxg = (G <= 4 && nch == 1) ? 4 : 16;
  // paired-tile variant (NT=2): 2x KV bytes in flight per wave — the
  // latency-bound fix (profiles/r01_st_attention.md SQ_WAIT diagnosis).
  // BBAMD_ATTN_NT=1 reverts; D>=256 keeps NT=1 (VGPR budget).
  static const int nt_env = [] {
    const char* e = std::getenv("BBAMD_ATTN_NT");
    return e ? std::atoi(e) : 2;
  }();
  // Software-pipelined variant (next tile's K+V double-buffered in
  // registers, its loads in flight behind this tile's): DEFAULT — 50 us /
  // 5.4 TB/s at B32 ctx2048 and 6.1 TB/s at ctx 8000 vs 59-62 us
  // for the NT variants at ctx2048. BBAMD_ATTN_PF=0 reverts to the NT path.
  static const bool pf_env = [] {
    const char* e = std::getenv("BBAMD_ATTN_PF");
    return !e || std::atoi(e) != 0;
  }();
  const bool pf = pf_env && (D <= 128);
  const bool nt2 = (nt_env >= 2) && (D <= 128) && !pf;
  auto launch_mfma = [&](auto mg) {
    if constexpr (D == 512) {
      // wide-head path: d split across the 4 waves (gemma-4 global layers)
      attn_decode_wide_kernel<decltype(mg)::value>
          <<<grid, 256, 0, cur_stream()>>>(
              bf_ptr(q) + q_off, bf_ptr(kp), bf_ptr(vp), pt.data_ptr<int>(),
              ctx.data_ptr<int>(), alibi_ptr, bf_ptr_mut(out),
              pml.data_ptr<float>(), pacc.data_ptr<float>(), B, Hkv, G, nch, P,
              maxp, n_split, window, scale, q_sb, q_sh, out_sb, out_sh, ctx_add,
              share);
    } else if (D <= 128 && pf) {
      auto go = [&](auto waves) {
        constexpr int NW = decltype(waves)::value;
        attn_decode_mfma_kernel<D, decltype(mg)::value, 1, 1, NW>
            <<<grid, NW * 64, 0, cur_stream()>>>(
                bf_ptr(q) + q_off, bf_ptr(kp), bf_ptr(vp), pt.data_ptr<int>(),
                ctx.data_ptr<int>(), alibi_ptr, bf_ptr_mut(out),
                pml.data_ptr<float>(), pacc.data_ptr<float>(), B, Hkv, G, nch, P,
                maxp, n_split, window, scale, q_sb, q_sh, out_sb, out_sh, ctx_add,
                share);
      };
      if constexpr (decltype(mg)::value == 4) {
        if (wide) return go(std::integral_constant<int, 8>{});
      }
      go(std::integral_constant<int, 4>{});
    } else if (D <= 128 && nt2) {
      attn_decode_mfma_kernel<D, decltype(mg)::value, 2>
          <<<grid, 256, 0, cur_stream()>>>(
              bf_ptr(q) + q_off, bf_ptr(kp), bf_ptr(vp), pt.data_ptr<int>(),
              ctx.data_ptr<int>(), alibi_ptr, bf_ptr_mut(out),
              pml.data_ptr<float>(), pacc.data_ptr<float>(), B, Hkv, G, nch, P,
              maxp, n_split, window, scale, q_sb, q_sh, out_sb, out_sh, ctx_add,
              share);
    } else {
      attn_decode_mfma_kernel<D, decltype(mg)::value, 1>
          <<<grid, 256, 0, cur_stream()>>>(
              bf_ptr(q) + q_off, bf_ptr(kp), bf_ptr(vp), pt.data_ptr<int>(),
              ctx.data_ptr<int>(), alibi_ptr, bf_ptr_mut(out),
              pml.data_ptr<float>(), pacc.data_ptr<float>(), B, Hkv, G, nch, P,
              maxp, n_split, window, scale, q_sb, q_sh, out_sb, out_sh, ctx_add,
              share);
    }
  };
  if (maxg == 4) launch_mfma(std::integral_constant<int, 4>{});
  else launch_mfma(std::integral_constant<int, 16>{});
  if (n_split > 1) {
    const int units = B * Hkv * nch;
    attn_decode_combine_kernel<D>
        <<<(units * maxg + 3) / 4, 256, 0, cur_stream()>>>(
            pml.data_ptr<float>(), pacc.data_ptr<float>(), bf_ptr_mut(out),
            units, Hkv, G, nch, maxg, n_split, nullptr, out_sb, out_sh);
  }
}

// The same in equal shares of the batch's tiles, then the parts of the cut contexts.
template <int D, int MAXG>
static void attn_decode_even_launch(
    const torch::Tensor& q, const torch::Tensor& kp, const torch::Tensor& vp,
    const torch::Tensor& pt, const torch::Tensor& ctx, const float* alibi_ptr,
    torch::Tensor& out, int B, int Hkv, int G, int nch, int P, int maxp, int window,
    float scale, long q_off, long q_sb, long q_sh, long out_sb, long out_sh, int ctx_add) {
  // two workgroups a CU: 222 registers
  const int heads = Hkv * nch, shares = std::max(1, 512 / heads);
  const long rows = (long)(B + shares) * heads;
  auto fopt = torch::TensorOptions().device(q.device()).dtype(at::kFloat);
  auto cuts = torch::empty({B, 2}, fopt.dtype(at::kInt));
  auto pml = torch::empty({rows, MAXG, 2}, fopt);
  auto pacc = torch::empty({rows, MAXG, D}, fopt);
  int2* cp = reinterpret_cast<int2*>(cuts.data_ptr<int>());
  attn_decode_even_kernel<D, MAXG, 4><<<shares * heads, 256, 0, cur_stream()>>>(
      bf_ptr(q) + q_off, bf_ptr(kp), bf_ptr(vp), pt.data_ptr<int>(), ctx.data_ptr<int>(),
      alibi_ptr, bf_ptr_mut(out), pml.data_ptr<float>(), pacc.data_ptr<float>(), cp, B, Hkv, G,
      nch, P, maxp, window, scale, q_sb, q_sh, out_sb, out_sh, ctx_add, shares);
  attn_decode_combine_kernel<D><<<(B * heads * MAXG + 3) / 4, 256, 0, cur_stream()>>>(
      pml.data_ptr<float>(), pacc.data_ptr<float>(), bf_ptr_mut(out), B * heads, Hkv, G, nch,
      MAXG, 0, cp, out_sb, out_sh);
}

// Whether a batch goes in equal shares, by the room of its contexts; their lengths are on
// the device. Where contexts and heads don't split evenly over the chip, a workgroup has all
// of one or an equal part of each, and the longest outlast the rest; what the shares cost is
// their folds, a launch, and finding them. us in a graph, without and with, 8 heads of keys,
// tokens of a context: 16 of 500 to 4000 42.6, 36.0; 24 of 100 to 2000 35.7, 26.8; 33 of 64
// to 4000 63.2, 55; 40 115, 61; 64 127, 92; 64 of 64 to 8000 245, 171; 70 223, 189; 97 of 64
// to 4000 159, 142; 200 of 64 to 2000 178, 157; 256 of 100 to 1000 119, 108; all of one
// length: 16 of 2000 29.1, 30.3; 24 41.2, 40.1; 28 43.0, 44.9; 40 of 1000 39.8, 37; 97 of
// 2000 142, 130; 300 of 2048 428, 394; 64 of 2000 87.4, 89.0. Shorter ones lose (16 of 1000
// 18.3, 19.1; 64 of 100 to 1000 34.8, 36; 100 of 150 18.3, 22.8), as do fewer (8 of 2000
// 19.1, 20.6) and those of which each CU has one (32 of 2048 46.7, 50.7; of 100 to 2000
// 37.7, 33.8).
static bool decode_even(long B, long heads, long room) {
  const long units = B * heads;
  return units >= 128 && (units <= 240 || units > 256) && room >= (units > 512 ? 1024 : 1536) &&
         heads <= 64 && B <= 1024 && B * room < 1L << 34;
}

static torch::Tensor attn_decode_core(
    const torch::Tensor& q, const torch::Tensor& k_pages,
    const torch::Tensor& v_pages, const torch::Tensor& page_table,
    const torch::Tensor& ctx_lens, const c10::optional<torch::Tensor>& alibi,
    double scale, long window, long n_split_req,
    int B, int Hq, int D, long q_off, long q_sb, long q_sh,
    torch::Tensor out, long out_sb, long out_sh, int ctx_add = 0) {
  const int Hkv = k_pages.size(1), P = k_pages.size(2), maxp = page_table.size(1);
  const int G = Hq / Hkv;
  TORCH_CHECK(Hq % Hkv == 0);
  TORCH_CHECK(D != 256 || G <= 4, "D=256 decode supports GQA group size <= 4");
  const int nch = (G + 15) / 16;  // MQA chunks (falcon G=71 -> 5)
  const float* alibi_ptr = nullptr;
  if (alibi.has_value()) {
    TORCH_CHECK(alibi->scalar_type() == at::kFloat && alibi->numel() == Hq);
    alibi_ptr = alibi->data_ptr<float>();
  }
  int n_split = (int)n_split_req;
  // Least tokens of a split: the four waves of a workgroup take 32 tokens each, and
  // shorter splits idle most of them. They share 32 where D = 512 (8 sequences of 300, 16
  // heads on 8: 31.6 us with splits of 128, 18.7 so).
  int share = n_split > 0 ? 1 : D == 512 ? 32 : 128;
  bool wide = false;
  if (n_split <= 0) {
    // measured optimum (benchmarks/bench_kernels.py attn_decode): size the
    // grid for full residency — NT=1 runs 118 VGPRs -> 4 WGs/CU (1024 WGs),
    // the paired-tile NT=2 variant 158 VGPRs -> 3 WGs/CU (768 WGs); more
    // splits only add merge traffic
    static const int nt_env0 = [] {
      const char* e = std::getenv("BBAMD_ATTN_NT");
      return e ? std::atoi(e) : 2;
    }();
    static const bool pf_env0 = [] {
      const char* e = std::getenv("BBAMD_ATTN_PF");
      return !e || std::atoi(e) != 0;
    }();
    // pipelined variant: 244 VGPRs -> 2 waves/SIMD -> 512 WGs fill the chip
    const long target = (pf_env0 && D <= 128) ? 512
                        : (nt_env0 >= 2 && D <= 128) ? 768 : 1024;
    const long units = std::max(1, B * Hkv * nch), room = (long)maxp * P;
    // Workgroups of eight waves with twice the tokens halve the splits to fold. They pay
    // where those still fill the chip as well, or where one does without any fold. us in
    // a graph, four waves and eight, heads of 128, 8 of keys: 1 sequence of 300 tokens 9.3,
    // 7.9; 500 8.6, 10.7; 4 of 1000 12.1, 13.1; 2000 16.7, 14.4; 2 of 2000 12.8, 13.2; 4000
    // 17.2, 15.0; 8 of 1000 14.9, 14.0; 8000 52.1, 48.5; 16 of 300 11.0, 9.0; 500 13.3, 12.9;
    // 2000 28.8, 28.3; 32 of 300 14.1, 10.5; 2000 48.2, 45.1. Heads of 32, 64 and 128, 1 to 32
    // of keys, 1 to 64 sequences of 100 to 8000 tokens, 4572 steps: none is slower by more than
    // 5% (0.5 us) than with one wave's fold and four waves throughout.
    if (pf_env0 && D <= 128 && decode_even(B, Hkv * nch, room)) {
      auto even = [&](auto d, auto g) {
        attn_decode_even_launch<decltype(d)::value, decltype(g)::value>(
            q, k_pages, v_pages, page_table, ctx_lens, alibi_ptr, out, B, Hkv, G, nch, P, maxp,
            (int)window, (float)scale, q_off, q_sb, q_sh, out_sb, out_sh, ctx_add);
      };
      auto of = [&](auto d) {
        if (G <= 4 && nch == 1) even(d, std::integral_constant<int, 4>{});
        else even(d, std::integral_constant<int, 16>{});
      };
      if (D == 128) of(std::integral_constant<int, 128>{});
      else if (D == 64) of(std::integral_constant<int, 64>{});
      else if (D == 32) of(std::integral_constant<int, 32>{});
      else TORCH_CHECK(false, "unsupported head_dim ", D);
      return out;
    }
    wide = pf_env0 && D <= 128 && G <= 4 && units <= 256 &&
           ((room >= 256 && room <= 352) ||
            (units * room >= 60000 && 256 / units * 2 >= target / units));
    if (wide) {
      share = 256;
      n_split = (int)std::max(1L, std::min({32L, 256 / units, room / share}));
    } else if (units > target) {
      // More units than fit at once: contexts of a large batch differ, and a
      // workgroup with a long one outlasts the rest. Pieces of 1024 tokens even it
      // out, where equal shares don't (heads wider than 128, or more than 64).
      share = 1024;
      n_split = (int)std::min(32L, (room + share - 1) / share);
    } else {
      n_split = (int)std::max(1L, std::min({32L, target / units, room / share}));
    }
  }
  const int maxg = (G <= 4 && nch == 1) ? 4 : 16;
  auto fopt = torch::TensorOptions().device(q.device()).dtype(at::kFloat);
  torch::Tensor pml, pacc;
  if (n_split > 1) {
    pml = torch::empty({(long)B * Hkv * nch * n_split, maxg, 2}, fopt);
    pacc = torch::empty({(long)B * Hkv * nch * n_split, maxg, D}, fopt);
  } else {
    pml = torch::empty({1}, fopt);
    pacc = torch::empty({1}, fopt);
  }
  auto go = [&](auto d) {
    attn_decode_launch<decltype(d)::value>(
        q, k_pages, v_pages, page_table, ctx_lens, alibi_ptr, out, pml, pacc,
        B, Hkv, G, nch, P, maxp, n_split, (int)window, (float)scale, q_off,
        q_sb, q_sh, out_sb, out_sh, ctx_add, share, wide);
  };
  if (D == 128) go(std::integral_constant<int, 128>{});
  else if (D == 64) go(std::integral_constant<int, 64>{});
  else if (D == 256) go(std::integral_constant<int, 256>{});
  else if (D == 512) go(std::integral_constant<int, 512>{});
  else if (D == 32) go(std::integral_constant<int, 32>{});
  else TORCH_CHECK(false, "unsupported head_dim ", D);
  return out;
}

torch::Tensor attn_decode(torch::Tensor q, torch::Tensor k_pages,
                          torch::Tensor v_pages, torch::Tensor page_table,
                          torch::Tensor ctx_lens, double scale, long window,
                          long n_split_req,
                          c10::optional<torch::Tensor> alibi) {
  CHECK_DEV(q); CHECK_BF16(q); CHECK_CONTIG(q);
  CHECK_DEV_ALL3(k_pages, page_table, ctx_lens);
  if (alibi.has_value()) CHECK_DEV((*alibi));
  TORCH_CHECK(q.dim() == 4 && q.size(2) == 1, "attn_decode expects (B, Hq, 1, D)");
  const int B = q.size(0), Hq = q.size(1), D = q.size(3);
  auto out = torch::empty({B, Hq, 1, D}, q.options());
  return attn_decode_core(q, k_pages, v_pages, page_table, ctx_lens, alibi,
                          scale, window, n_split_req, B, Hq, D,
                          /*q_off*/ 0, (long)Hq * D, (long)D,
                          out, (long)Hq * D, (long)D);
}

// Fused-QKV decode: q section of qkv (B, 1, (Hq+2Hkv)*D) read in place,
// out (B, 1, Hq*D) ready for the O-projection GEMM — zero transposes. A context is
// ctx_lens + ctx_add tokens.
torch::Tensor attn_decode_qkv(torch::Tensor qkv, long Hq, torch::Tensor k_pages,
                              torch::Tensor v_pages, torch::Tensor page_table,
                              torch::Tensor ctx_lens, double scale, long window,
                              long n_split_req, long ctx_add) {
  CHECK_DEV(qkv); CHECK_BF16(qkv); CHECK_CONTIG(qkv);
  CHECK_DEV_ALL3(k_pages, page_table, ctx_lens);
  const int Hkv = k_pages.size(1);
  const int D = k_pages.size(3);
  const int B = qkv.size(0);
  TORCH_CHECK(qkv.dim() == 3 && qkv.size(1) == 1 &&
              qkv.size(2) == (Hq + 2 * Hkv) * D, "bad fused qkv shape");
  auto out = torch::empty({B, 1, Hq * D}, qkv.options());
  return attn_decode_core(qkv, k_pages, v_pages, page_table, ctx_lens,
                          c10::nullopt, scale, window, n_split_req, B, (int)Hq,
                          D, /*q_off*/ 0, (long)(Hq + 2 * Hkv) * D, (long)D,
                          out, (long)Hq * D, (long)D, (int)ctx_add)
      .view({B, 1, Hq * D});
}

// beyond 2^20 keys a page's offsets would leave 32 bits
static PrefillPages prefill_pages(int P) {
  if ((P & (P - 1)) != 0 || P > 1 << 20) return PREFILL_MIXED;
  return P >= 16 ? PREFILL_GROUPS : PREFILL_EIGHTS;
}

struct PrefillPlan { int splits; bool two; };

// How the keys of attn_prefill are shared out: splits, and whether two groups of waves
// share those of a workgroup. keys: that a row may see, at most (333 tokens behind 3000
// with windows of 512 take 19.9 us by their windows, 29.8 by the context).
static PrefillPlan prefill_plan(long units, int G, int Tq, int D, int P, long keys,
                                bool tree, int window) {
  const long base = ((long)Tq * G + 127) / 128 * units;   // workgroups without splits
  // a workgroup's rows are 128 / G tokens, whose windows begin within a tile
  if (window > 0) keys = std::min(keys, (long)window + 128 / G + 64);
  // A workgroup walks its keys in a chain of tiles, about 1.7 us each at D = 128
  // when it has the CU to itself. Where row tiles alone leave CUs idle the keys are
  // split until every CU has a workgroup, and until it has two where the chains
  // stay long; no split is shorter than two tiles of the longest context. Measured with 32
  // heads on 8 and one group of waves (an address a lane, alone in a graph: some 4 us more
  // than in a row), splits as written against none / against twice as many: 25 tokens behind
  // 1500 20 / 41 / 20 us, 64 behind 8000 38 / 195 / 51, 333 behind 1201 37 / 42 / 39, 500
  // behind 7000 (four splits) 95 / 184 / 106, 1000 behind 4000 (two) 114 / 127 / 125.
  long splits = std::max<long>(1, 256 / base);
  if (keys > splits * 24 * 64) splits = std::max<long>(1, 512 / base);
  PrefillPlan plan{(int)std::max<long>(1, std::min({splits, keys / 128, 32L})), false};
  // Two groups of waves that share out a workgroup's keys halve its chain for 4.5 us, where
  // another split takes 4 and its sums' way through memory and back, 45 ns a workgroup; a
  // tile takes 2.4 us. Measured, a call of several in a graph, us with the splits above and
  // one group, an address a lane / as chosen here: 333 behind none 21 / 14, behind 300
  // 25 / 19, behind 1201 36 / 33, behind 8000 (one group) 78 / 72; 2 x 333 behind 1201
  // 43 / 35; 480 behind 100 28.5 / 19.5; 1000 behind 4000 111 / 97; 64 behind 2000
  // 22.5 / 21; 1024 behind 1024 57 / 45.5. Chains of a tile or two keep one group, and large
  // trees as many workgroups as they can have, for the bytes of their masks (600 tokens of
  // 16 heads of 64: 31; two groups take a sixth more).
  if (prefill_pages(P) == PREFILL_GROUPS && D <= 128 && base <= 256 &&
      (!tree || Tq <= 128)) {
    const long tiles = (keys + 63) / 64;
    auto cost = [&](long s, long groups) {
      return 2.4 * ((tiles + groups * s - 1) / (groups * s)) +
             (s > 1 ? 4 + 0.045 * base * s : 0.) + (groups > 1 ? 4.5 : 0);
    };
    // these costs are no closer than 8% (two trees of 40 nodes behind 2000 gain 5% by them
    // and lost 4)
    double least = cost(plan.splits, 1) / 1.08;
    const long most = std::max<long>(1, std::min({256 / base, keys / 128, 32L}));
    for (long s = 1; s <= most; ++s)
      if (cost(s, 2) < least) {
        least = cost(s, 2);
        plan = {(int)s, true};
      }
  }
  return plan;
}

// Whether the launches to come are replayed later, with contexts of any length; also where
// the stream does not tell.
static bool captured() {
  hipStreamCaptureStatus status;
  if (hipStreamIsCapturing(cur_stream(), &status) == hipSuccess)
    return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

// Launches attention of a.Tq tokens a sequence; a's tensors and strides are set. longest:
// no sequence has more tokens, these among them, as far as the caller knows; 0: unknown.
static void launch_attn_prefill(PrefillArgs a, int D, int P,
                                const torch::TensorOptions& f32, long longest) {
  // eight values of a page's row are read at once
  TORCH_CHECK(P > 0 && P % 8 == 0, "page size must be a multiple of eight");
  a.P = P;
  a.p_log2 = __builtin_ctz(P);
  const long rows = (long)a.Tq * a.G, units = (long)a.B * a.Hkv;
  if (rows == 0 || units == 0) return;
  const long row_tiles = (rows + 127) / 128;
  // A table is as wide as a session may become. By its width, 64 tokens that begin one of
  // 8192 took 16 splits of two groups for their single tile: 13.5 us, 6.8 by their number.
  long keys = (long)a.maxp * P;
  if (longest > 0 && !captured())
    keys = std::min(keys, ldiv_up(std::max<long>(longest, a.Tq), P) * P);
  const PrefillPlan plan =
      prefill_plan(units, a.G, a.Tq, D, P, keys, a.tree_mask != nullptr, a.window);
  a.n_split = plan.splits;
  torch::Tensor part;
  if (a.n_split > 1) {
    part = torch::empty({(long)a.n_split * units * rows * (D + 2)}, f32);
    a.pacc = part.data_ptr<float>();
    a.pml = a.pacc + (long)a.n_split * units * rows * D;
  }
  const dim3 grid(units * a.n_split, row_tiles);
  auto start = [&](auto d, auto form, auto pages, auto groups) {
    constexpr int DD = decltype(d)::value, KG = decltype(groups)::value;
    auto kernel =
        attn_prefill_kernel<DD, decltype(form)::value, decltype(pages)::value, KG>;
    constexpr int lds = KG * 2 * PrefillTile<DD>::BYTES;
    if (lds > 64 * 1024)
      TORCH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      lds) == hipSuccess,
                  "cannot reserve ", lds, " bytes of LDS");
    kernel<<<grid, 256 * KG, lds, cur_stream()>>>(a);
    auto fold = [&](auto c) {
      attn_prefill_fold_kernel<DD, decltype(c)::value>
          <<<ldiv_up((long)units * rows * (DD / 4), 256), 256, 0, cur_stream()>>>(a);
    };
    if (a.n_split > 4) fold(std::integral_constant<int, 8>{});
    else if (a.n_split > 2) fold(std::integral_constant<int, 4>{});
    else if (a.n_split > 1) fold(std::integral_constant<int, 2>{});
  };
  auto launch = [&](auto d, auto form, auto pages) {
    if constexpr (decltype(pages)::value == PREFILL_GROUPS && decltype(d)::value <= 128)
      if (plan.two) return start(d, form, pages, std::integral_constant<int, 2>{});
    start(d, form, pages, std::integral_constant<int, 1>{});
  };
  auto by_dim = [&](auto form, auto pages) {
    if (D == 128) launch(std::integral_constant<int, 128>{}, form, pages);
    else if (D == 64) launch(std::integral_constant<int, 64>{}, form, pages);
    else if (D == 256) launch(std::integral_constant<int, 256>{}, form, pages);
    else if (D == 32) launch(std::integral_constant<int, 32>{}, form, pages);
    else TORCH_CHECK(false, "unsupported head_dim ", D);
  };
  constexpr std::integral_constant<int, PREFILL_TREE> tree;
  auto by_form = [&](auto pages) {
    if (a.tree_mask) by_dim(tree, pages);
    else if (a.alibi || !(a.scale > 0.f))
      by_dim(std::integral_constant<int, PREFILL_GENERAL>{}, pages);
    else by_dim(std::integral_constant<int, PREFILL_PLAIN>{}, pages);
  };
  const PrefillPages kind = prefill_pages(P);
  if (kind == PREFILL_MIXED) by_dim(tree, std::integral_constant<int, PREFILL_MIXED>{});
  else if (kind == PREFILL_EIGHTS)
    by_form(std::integral_constant<int, PREFILL_EIGHTS>{});
  else by_form(std::integral_constant<int, PREFILL_GROUPS>{});
}

// Pages go to LDS by 16-byte copies: a view that does not begin at 16 bytes is copied.
static void set_pages(PrefillArgs& a, torch::Tensor& k, torch::Tensor& v) {
  for (torch::Tensor* t : {&k, &v})
    if ((size_t)t->data_ptr() % 16 != 0) *t = t->clone();
  a.k_pages = bf_ptr(k);
  a.v_pages = bf_ptr(v);
}

static void set_tree_mask(PrefillArgs& a, const c10::optional<torch::Tensor>& mask,
                          int B, int Tq, long window) {
  if (!mask.has_value()) return;
  TORCH_CHECK(mask->scalar_type() == at::kBool && mask->is_contiguous() &&
                  mask->sizes() == (at::IntArrayRef{B, Tq, Tq}),
              "tree_mask must be contiguous bool (B, Tq, Tq)");
  TORCH_CHECK(window == 0, "tree_mask + sliding window: use the torch path");
  CHECK_DEV((*mask));
  // kBool tensors dispatch data_ptr<bool>, not <unsigned char> (Byte)
  a.tree_mask = reinterpret_cast<const unsigned char*>(mask->data_ptr<bool>());
}

torch::Tensor attn_prefill(torch::Tensor q, torch::Tensor k_pages,
                           torch::Tensor v_pages, torch::Tensor page_table,
                           torch::Tensor q_start, double scale, long window,
                           c10::optional<torch::Tensor> alibi,
                           c10::optional<torch::Tensor> tree_mask, long longest) {
  CHECK_DEV(q); CHECK_BF16(q); CHECK_CONTIG(q);
  CHECK_DEV_ALL3(k_pages, page_table, q_start);
  if (alibi.has_value()) CHECK_DEV((*alibi));
  TORCH_CHECK(q.dim() == 4, "attn_prefill expects (B, Hq, Tq, D)");
  const int B = q.size(0), Hq = q.size(1), Tq = q.size(2), D = q.size(3);
  const int Hkv = k_pages.size(1), P = k_pages.size(2), maxp = page_table.size(1);
  PrefillArgs a{};
  if (alibi.has_value()) {
    TORCH_CHECK(alibi->scalar_type() == at::kFloat && alibi->numel() == Hq);
    a.alibi = alibi->data_ptr<float>();
  }
  set_tree_mask(a, tree_mask, B, Tq, window);
  auto out = torch::empty_like(q);
  a.q = bf_ptr(q);
  set_pages(a, k_pages, v_pages);
  a.page_table = page_table.data_ptr<int>();
  a.q_start = q_start.data_ptr<int>();
  a.out = bf_ptr_mut(out);
  a.B = B; a.Hkv = Hkv; a.G = Hq / Hkv; a.Tq = Tq; a.maxp = maxp;
  a.window = (int)window;
  a.scale = (float)scale;
  a.q_sb = a.o_sb = (long)Hq * Tq * D;
  a.q_st = a.o_st = D;
  a.q_sh = a.o_sh = (long)Tq * D;
  launch_attn_prefill(a, D, P, q.options().dtype(at::kFloat), longest);
  return out;
}

// Fused-QKV prefill: q read from qkv (B, Tq, (Hq+2Hkv)*D) in place,
// out (B, Tq, Hq*D) ready for the O-projection GEMM.
torch::Tensor attn_prefill_qkv(torch::Tensor qkv, long Hq_,
                               torch::Tensor k_pages, torch::Tensor v_pages,
                               torch::Tensor page_table, torch::Tensor q_start,
                               double scale, long window,
                               c10::optional<torch::Tensor> tree_mask, long longest) {
  CHECK_DEV(qkv); CHECK_BF16(qkv); CHECK_CONTIG(qkv);
  CHECK_DEV_ALL3(k_pages, page_table, q_start);
  const int Hkv = k_pages.size(1), P = k_pages.size(2), D = k_pages.size(3);
  const int maxp = page_table.size(1);
  const int Hq = (int)Hq_;
  const int B = qkv.size(0), Tq = qkv.size(1);
  const int X = Hq + 2 * Hkv;
  TORCH_CHECK(qkv.dim() == 3 && qkv.size(2) == (long)X * D, "bad fused qkv shape");
  auto out = torch::empty({B, Tq, (long)Hq * D}, qkv.options());
  PrefillArgs a{};
  set_tree_mask(a, tree_mask, B, Tq, window);
  a.q = bf_ptr(qkv);
  set_pages(a, k_pages, v_pages);
  a.page_table = page_table.data_ptr<int>();
  a.q_start = q_start.data_ptr<int>();
  a.out = bf_ptr_mut(out);
  a.B = B; a.Hkv = Hkv; a.G = Hq / Hkv; a.Tq = Tq; a.maxp = maxp;
  a.window = (int)window;
  a.scale = (float)scale;
  a.q_sb = (long)Tq * X * D;
  a.q_st = (long)X * D;
  a.q_sh = a.o_sh = D;
  a.o_sb = (long)Tq * Hq * D;
  a.o_st = (long)Hq * D;
  launch_attn_prefill(a, D, P, qkv.options().dtype(at::kFloat), longest);
  return out;
}

// Fused RoPE + paged-KV write on the raw QKV GEMM output.
void rope_kv_write_(torch::Tensor qkv, long Hq_, long Hkv_, torch::Tensor cos_t,
                    torch::Tensor sin_t, c10::optional<torch::Tensor> pos,
                    torch::Tensor k_pages, torch::Tensor v_pages,
                    torch::Tensor page_table, torch::Tensor start_pos,
                    c10::optional<torch::Tensor> q_norm,
                    c10::optional<torch::Tensor> k_norm, double eps) {
  CHECK_DEV(qkv); CHECK_BF16(qkv); CHECK_CONTIG(qkv);
  CHECK_DEV_ALL3(k_pages, page_table, start_pos);
  CHECK_DEV_ALL2(cos_t, sin_t);
  if (pos.has_value()) CHECK_DEV((*pos));
  const int Hq = (int)Hq_, Hkv = (int)Hkv_;
  const int P = k_pages.size(2), D = k_pages.size(3);
  const int maxp = page_table.size(1);
  const int B = qkv.size(0), T = qkv.size(1);
  TORCH_CHECK(qkv.size(2) == (long)(Hq + 2 * Hkv) * D, "bad fused qkv shape");
  const int* pos_ptr = nullptr;
  if (pos.has_value()) {
    TORCH_CHECK(pos->scalar_type() == at::kInt);
    pos_ptr = pos->data_ptr<int>();
  }
  const unsigned short* norms[2] = {nullptr, nullptr};
  const c10::optional<torch::Tensor>* given[2] = {&q_norm, &k_norm};
  for (int i = 0; i < 2; ++i)
    if (given[i]->has_value()) {
      const torch::Tensor& w = **given[i];
      TORCH_CHECK(w.is_cuda() && w.scalar_type() == at::kBFloat16 &&
                      w.is_contiguous() && w.numel() == D,
                  "head norm weights must be contiguous bf16 of length D");
      norms[i] = bf_ptr(w);
    }
  if (B == 0 || T == 0) return;
  // From 64 tokens on, in octets where pages and rows allow it; few tokens end sooner
  // one head a wave (32, 8 and 8 heads of 128, us): 16 tokens 2.7 (octets 3.4), 64 3.3
  // (3.3), 97 of as many sequences 4.1 (3.8), 333 7.6 (3.9), 4 x 4096 233 (70).
  auto aligned = [](const void* q) { return q == nullptr || (size_t)q % 16 == 0; };
  if ((long)B * T >= 64 && P % 8 == 0 && (D == 32 || D == 64 || D == 128 || D == 256) &&
      aligned(qkv.data_ptr()) && aligned(k_pages.data_ptr()) &&
      aligned(v_pages.data_ptr()) && aligned(norms[0]) && aligned(norms[1])) {
    const int octs = (T + 7) / 8 + 1;
    const long qk = ((long)B * T * (Hq + Hkv) * (D / 16) + 255) / 256;
    const long v = ((long)B * Hkv * octs * (D / 2) + 255) / 256;
    auto go = [&](auto l) {
      rope_kv_rows_kernel<decltype(l)::value><<<qk + v, 256, 0, cur_stream()>>>(
          bf_ptr_mut(qkv), cos_t.data_ptr<float>(), sin_t.data_ptr<float>(), pos_ptr,
          bf_ptr_mut(k_pages), bf_ptr_mut(v_pages), page_table.data_ptr<int>(),
          start_pos.data_ptr<int>(), B, Hq, Hkv, T, P, maxp, (int)cos_t.size(0),
          norms[0], norms[1], (float)eps, (int)qk, octs);
    };
    if (D == 32) go(std::integral_constant<int, 2>{});
    else if (D == 64) go(std::integral_constant<int, 4>{});
    else if (D == 128) go(std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, 16>{});
    return;
  }
  dim3 grid(B * T, Hq + 2 * Hkv);
  auto launch = [&](auto norm) {
    rope_kv_write_kernel<decltype(norm)::value><<<grid, 64, 0, cur_stream()>>>(
        bf_ptr_mut(qkv), cos_t.data_ptr<float>(), sin_t.data_ptr<float>(), pos_ptr,
        bf_ptr_mut(k_pages), bf_ptr_mut(v_pages), page_table.data_ptr<int>(),
        start_pos.data_ptr<int>(), B, Hq, Hkv, T, D, P, maxp, (int)cos_t.size(0),
        norms[0], norms[1], (float)eps);
  };
  if (norms[0] || norms[1]) launch(std::true_type{});
  else launch(std::false_type{});
}


// (a + res, its RMS norm, chosen experts (N, top) int32, their weights f32) of rows
// a, res (N, H); without res and norm_w the first two are a itself.
std::vector<torch::Tensor> norm_route(torch::Tensor a,
                                      c10::optional<torch::Tensor> res,
                                      c10::optional<torch::Tensor> norm_w,
                                      torch::Tensor router, long top, double eps) {
  CHECK_DEV_ALL2(a, router); CHECK_BF16(a); CHECK_BF16(router);
  CHECK_CONTIG(a); CHECK_CONTIG(router);
  TORCH_CHECK(a.dim() == 2 && router.dim() == 2, "(N, H) rows, (E, H) router");
  const long N = a.size(0), H = a.size(1), E = router.size(0);
  TORCH_CHECK(router.size(1) == H && H % 8 == 0 && E <= ROUTE_MAX_E && top >= 1 &&
                  top <= E && res.has_value() == norm_w.has_value(),
              "bad router shapes");
  const bool norm = norm_w.has_value();
  // rows that are handed on as they are go to LDS by 16-byte copies in the experts
  if (!norm && (size_t)a.data_ptr() % 16 != 0) a = a.clone();
  if (norm) {
    CHECK_DEV_ALL2((*res), (*norm_w)); CHECK_BF16((*res)); CHECK_BF16((*norm_w));
    CHECK_CONTIG((*res)); CHECK_CONTIG((*norm_w));
    TORCH_CHECK(res->numel() == a.numel() && norm_w->numel() == H, "bad norm shapes");
  }
  auto h = norm ? torch::empty_like(a) : a, y = norm ? torch::empty_like(a) : a;
  auto ids = torch::empty({N, top}, a.options().dtype(at::kInt));
  auto wts = torch::empty({N, top}, a.options().dtype(at::kFloat));
  if (N == 0) return {h, y, ids, wts};
  dispatch_iters(H, [&](auto iters) {
    norm_route_kernel<decltype(iters)::value><<<N, 256, 0, cur_stream()>>>(
        bf_ptr(a), norm ? bf_ptr(*res) : nullptr, norm ? bf_ptr(*norm_w) : nullptr,
        bf_ptr(router), bf_ptr_mut(h), bf_ptr_mut(y), ids.data_ptr<int>(),
        wts.data_ptr<float>(), H, E, top, (float)eps);
  });
  return {h, y, ids, wts};
}

// h (N, W), if any, + the sum over the experts of y (N, top, W).
torch::Tensor add_experts(c10::optional<torch::Tensor> h, torch::Tensor y) {
  CHECK_DEV(y); CHECK_BF16(y); CHECK_CONTIG(y);
  TORCH_CHECK(y.dim() == 3 && y.size(2) % 8 == 0, "bad expert rows");
  if (h.has_value()) {
    CHECK_DEV((*h)); CHECK_BF16((*h)); CHECK_CONTIG((*h));
    TORCH_CHECK(h->dim() == 2 && y.size(0) == h->size(0) && y.size(2) == h->size(1),
                "bad expert rows");
  }
  auto out = torch::empty({y.size(0), y.size(2)}, y.options());
  const long n = out.numel();
  if (n == 0) return out;
  add_experts_kernel<<<std::min<long>((n / 8 + 255) / 256, 4096), 256, 0,
                       cur_stream()>>>(h.has_value() ? bf_ptr(*h) : nullptr,
                                       bf_ptr(y), bf_ptr_mut(out), n, y.size(2),
                                       y.size(1));
  return out;
}

// C(S,N) = A[row(s)] @ W[expert(s)]^T — grouped decode MoE (moe_gemm.hip).
// off: (E+1,) int32 exclusive prefix sums of per-expert slot counts;
// rowmap: optional (S,) int32 slot->A-row gather; scale: optional (S,) f32
// per-slot epilogue scale (routing weights). S and mchunks are host-side
// upper-bound shapes so no device sync is needed.
torch::Tensor moe_gemm(torch::Tensor A, torch::Tensor W, torch::Tensor off,
                       c10::optional<torch::Tensor> rowmap,
                       c10::optional<torch::Tensor> scale,
                       long S, long mchunks) {
  CHECK_DEV(A); CHECK_BF16(A); CHECK_CONTIG(A);
  CHECK_DEV(W); CHECK_BF16(W); CHECK_CONTIG(W);
  CHECK_DEV(off);
  TORCH_CHECK(W.dim() == 3, "W must be (E, N, K)");
  const int E = W.size(0), N = W.size(1), K = W.size(2);
  TORCH_CHECK(A.size(-1) == K, "A/W K mismatch");
  TORCH_CHECK(K % 32 == 0 && N % 64 == 0, "K%32, N%64 required");
  TORCH_CHECK(off.scalar_type() == at::kInt && off.numel() == E + 1);
  const int* rmp = nullptr;
  if (rowmap.has_value()) {
    TORCH_CHECK(rowmap->scalar_type() == at::kInt &&
                rowmap->is_contiguous() && rowmap->numel() == S);
    CHECK_DEV((*rowmap));
    rmp = rowmap->data_ptr<int>();
  }
  const float* sp = nullptr;
  if (scale.has_value()) {
    TORCH_CHECK(scale->scalar_type() == at::kFloat &&
                scale->is_contiguous() && scale->numel() == S);
    CHECK_DEV((*scale));
    sp = scale->data_ptr<float>();
  }
  auto C = torch::empty({S, (long)N}, A.options());
  TORCH_CHECK(mchunks >= 1);
  dim3 grid(N / 64, (unsigned)(E * mchunks));
  if (K % 256 == 0)
    moe_gemm_v2_kernel<2><<<grid, 256, 0, cur_stream()>>>(
        bf_ptr(A), bf_ptr(W), off.data_ptr<int>(), rmp, sp, bf_ptr_mut(C),
        N, K, (int)mchunks);
  else
    moe_gemm_kernel<2><<<grid, 256, 0, cur_stream()>>>(
        bf_ptr(A), bf_ptr(W), off.data_ptr<int>(), rmp, sp, bf_ptr_mut(C),
        N, K, (int)mchunks);
  return C;
}


// C(M,N) = A @ dequant4(Wq)^T [+R] [+bias], M <= 32 (w4_gemm.hip). Wq/scale/
// zero in quant4_pack layout (2 codes/byte along K, f16 scale+zero per group
// of 64). ~3.5x less weight-stream bytes than the bf16 kernel.
torch::Tensor gemm_w4(torch::Tensor A, torch::Tensor Wq, torch::Tensor scale,
                      torch::Tensor zero,
                      c10::optional<torch::Tensor> residual,
                      c10::optional<torch::Tensor> bias, long N_, long ksplit_req) {
  CHECK_DEV(A); CHECK_CONTIG(A);
  TORCH_CHECK(A.scalar_type() == at::kHalf,
              "gemm_w4 takes fp16 activations (wrapper converts)");
  CHECK_DEV_ALL3(Wq, scale, zero);
  CHECK_CONTIG(Wq);
  TORCH_CHECK(Wq.scalar_type() == at::kByte && scale.scalar_type() == at::kHalf
              && zero.scalar_type() == at::kHalf);
  const int K = A.size(-1);
  const int M = A.numel() / K;
  const int N = (int)N_;
  TORCH_CHECK(M <= 32, "gemm_w4 is for M <= 32, got ", M);
  TORCH_CHECK(Wq.numel() == (long)N * K / 2, "Wq shape mismatch");
  TORCH_CHECK(scale.numel() == (long)N * K / 64, "scale shape mismatch");
  TORCH_CHECK(K % 128 == 0 && N % 64 == 0, "K%128, N%64 required");
  auto sizes = A.sizes().vec();
  sizes.back() = N;
  auto C = torch::empty(sizes, A.options().dtype(at::kBFloat16));
  const unsigned short* rp = nullptr;
  if (residual.has_value()) {
    TORCH_CHECK(residual->is_contiguous() && residual->numel() == (long)M * N);
    rp = bf_ptr(*residual);
  }
  const unsigned short* bp = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_contiguous() && bias->numel() == N);
    bp = bf_ptr(*bias);
  }
  // M==1 (the speculative-draft GEMV shape): contiguous 1 KB code loads +
  // v_dot2 — measured 2x the bf16 kernel (w4_probe.hip). The MROWS<=4
  // extension was measured and REJECTED for dispatch: amortizing the
  // dequant over rows loses to the split-K MFMA form (M4 down-proj 131 us
  // vs ~13 — the per-lane 4 B A loads scale with M and dominate); the
  // kernel keeps MROWS for completeness (parity-tested).
  if (M == 1 && K % 2048 == 0 && K / 2048 <= 7) {
    const int rpw = 4;
    dim3 gv((N / rpw + 3) / 4);
    auto lv2 = [&](auto nl, auto mr) {
      gemm_w4_gemv_kernel<decltype(nl)::value, decltype(mr)::value>
          <<<gv, 256, 0, cur_stream()>>>(
              reinterpret_cast<const _Float16*>(A.data_ptr()),
              Wq.data_ptr<unsigned char>(),
              reinterpret_cast<const __half*>(scale.data_ptr()),
              reinterpret_cast<const __half*>(zero.data_ptr()),
              rp, bp, bf_ptr_mut(C), N, K, rpw);
    };
    auto lv = [&](auto nl) {
      switch (M) {
        case 1: lv2(nl, std::integral_constant<int, 1>{}); break;
        case 2: lv2(nl, std::integral_constant<int, 2>{}); break;
        case 3: lv2(nl, std::integral_constant<int, 3>{}); break;
        default: lv2(nl, std::integral_constant<int, 4>{}); break;
      }
    };
    switch (K / 2048) {
      case 1: lv(std::integral_constant<int, 1>{}); break;
      case 2: lv(std::integral_constant<int, 2>{}); break;
      case 3: lv(std::integral_constant<int, 3>{}); break;
      case 4: lv(std::integral_constant<int, 4>{}); break;
      case 5: lv(std::integral_constant<int, 5>{}); break;
      case 6: lv(std::integral_constant<int, 6>{}); break;
      default: lv(std::integral_constant<int, 7>{}); break;
    }
    return C;
  }
  int ksplit = (int)ksplit_req;
  if (ksplit <= 0) {
    // the w4 stream is LATENCY-bound at the bf16 kernel's grid size (1.2
    // TB/s at 448 blocks); split K until the grid reaches ~1800 blocks
    // (w4_probe.hip: ksplit=4 on N=28672 -> 2.25 TB/s, plateau beyond)
    ksplit = (int)std::max<long>(1, std::min<long>(K / 512,
                                                   1792 / std::max(1, (N + 63) / 64)));
  }
  // groups of 64 must not straddle splits; slices of 128 keep the k-loop
  // tail-free
  const int nch = K / 128;
  const int per = (nch + ksplit - 1) / ksplit;
  ksplit = (nch + per - 1) / per;
  const int kchunk = per * 128;
  torch::Tensor part;
  float* pp = nullptr;
  if (ksplit > 1) {
    part = torch::empty({(long)ksplit, (long)M, (long)N},
                        torch::TensorOptions().device(A.device()).dtype(at::kFloat));
    pp = part.data_ptr<float>();
  }
  dim3 grid((N + 63) / 64, ksplit);
  auto launch = [&](auto mt) {
    gemm_skinny_w4_kernel<decltype(mt)::value><<<grid, 256, 0, cur_stream()>>>(
        reinterpret_cast<const _Float16*>(A.data_ptr()),
        Wq.data_ptr<unsigned char>(),
        reinterpret_cast<const __half*>(scale.data_ptr()),
        reinterpret_cast<const __half*>(zero.data_ptr()),
        ksplit == 1 ? rp : nullptr, ksplit == 1 ? bp : nullptr,
        bf_ptr_mut(C), pp, M, N, K, kchunk, ksplit);
  };
  if (M <= 16) launch(std::integral_constant<int, 1>{});
  else launch(std::integral_constant<int, 2>{});
  if (ksplit > 1) {
    const long total = (long)M * N;
    const int cgrid = (int)std::min<long>((total + 255) / 256, 2048);
    gemm_skinny_combine_kernel<<<cgrid, 256, 0, cur_stream()>>>(
        pp, rp, bp, bf_ptr_mut(C), M, N, ksplit);
  }
  return C;
}

// ---------------------------------------------------------------------------
// skinny-M GEMM (decode projections)
// ---------------------------------------------------------------------------

// Where the one-launch kernel (gemm_stream.hip) is the faster one. It takes 16 columns a
// workgroup over all of K and sums up by itself; the split GEMM (gemm_skinny.hip) takes 64
// and shares K out, which a second launch folds, below 16384 columns, and all of K above.
// So the first saves a launch, but it fills the chip in rounds of 256 workgroups that cost
// 1.7 us each beside their loads, and every workgroup reads all of A: twice the bytes of
// its W at 32 rows. us below: one launch, split.

// A product with the norm of its rows, which the other form takes in a pass of its own
// (4 to 5 us).
static bool stream_rows(long M, long N, long K) {
  return M <= 16 || (M <= 32 && N * K <= (32L << 20));
}

// The unsplit form of the other one leaves CUs idle in its last round.
static bool skinny_idles(long N) {
  const long wgs = N / 64, rounds = (wgs + 255) / 256;
  return N > 16384 && wgs * 10 < rounds * 256 * 7;
}

// A product alone, up to 32 rows.
static bool stream_sums(long M, long N, long K) {
  const long rounds = (N / 16 + 255) / 256;
  const bool full = N * 5 >= rounds * 4096 * 4;
  // One round: few columns leave it too little to hide a long chain over K, the more so the
  // more rows (up to 8 of few columns have another form, stream_parts, not in these figures).
  // 1024 x 3072: 1 row 5.6, 7.3; 32 rows 7.3, 8.6. 4096 x 14336: 23.8, 28.7; 16
  // rows 27.6, 28.8. 2048 x 8192: 1 row 11.2, 12.5; 16 rows 14.4, 13.3. 512 x 14336: 16.1,
  // 15.4; 22.5, 16.2.
  if (rounds == 1) return K * (192 * (M + 16) - N) <= 192L << 17;
  // Beyond 16 rows two workgroups share a CU, and each reads twice as much of A. 8192 x 1024:
  // 17 rows 6.5, 8.6. 8192 x 4096: 32 rows 20.5, 21.9. 5120 x 4096: 18.4, 17.3.
  if (M > 16)
    return (K <= 2048 && (rounds == 2 || (rounds == 3 && K >= 1024))) ||
           (rounds == 2 && K <= 4096 && N >= 6144) || (skinny_idles(N) && K >= 2048);
  // Two and three rounds, where K outweighs their start and few CUs sit the last one out.
  // 5120 x 512: 1 row 4.8, 4.4. 8192 x 8192: 29.3, 31.4; 16 rows 33.1, 33.1. 4608 x 4096:
  // 13.3, 14.6; 16.1, 16.0. 4608 x 14336: 37.0, 36.1; 46.7, 37.9.
  if (rounds <= 3) {
    if (K <= 2048) return K >= 1024;
    if (full) return M <= (rounds == 3 || K > 8192 ? 12 : 16);
    return K <= 6144 && K * M <= (rounds == 2 ? 1 << 16 : 1 << 15);
  }
  // Many columns: vocabularies and [gate | up], where the other form is one launch, too.
  // 151936 x 1024: 1 row 96, 56; 16 rows 116, 64. 128256 x 4096: 190, 191; 243, 195. 18176 x
  // 4096: 33.7, 40.1; 39.2, 42.4. 57344 x 8192: 161, 186; 192, 185.
  return (skinny_idles(N) && K >= 2048) || (K >= 8192 && M <= 8);
}

// A gated product, which the other form does in one launch, too. This one's workgroups
// take 8192 columns a round, the other's 16384: an odd number of rounds is less than the
// other takes. 8192 x 4096: 1 row 15.7, 24.6; 32 rows 17.5, 25.6. 22016 x 4096: 36.1, 40.5;
// 43.2, 45.7. 57344 x 8192: 158, 175; 186, 181. Even ones: 28672 x 4096 47.6, 48.6; 16 rows
// 49.8, 47.4; 32 rows 56.5, 51.0. Short chains do not pay their start: 28672 x 512 10.0, 8.6.
static bool stream_swiglu(long M, long N, long K) {
  const long rounds = (N / 32 + 255) / 256;
  return N <= 8192 || (K >= 1024 && (rounds % 2 == 1 || M <= 4));
}

// Queries, keys and values with their turns, 8192 columns a round: short chains, or one
// round that is more than half full, or nearly two. 4096 x 1024: 1 row 5.3, 7.5; 32 rows
// 7.4, 8.5. 6144 x 4096: 13.5, 15.4; 18.7, 18.1, where a step of 32 rows is 3 us a layer
// faster with one launch less all the same. 10240 x 8192: 44.0, 41.7; 55.1, 46.4. 2048 x
// 4096: 11.6, 8.9.
static bool stream_rope(long M, long N, long K) {
  if (M > 16) return K <= 1024 || (N >= 5120 && N <= 8192 && (K <= 4096 || N > 6144));
  return K <= 2048 || (N <= 8192 && N >= (K <= 3072 ? 3072 : 5120)) || N >= 14336;
}

// A's rows go to LDS by 16-byte copies: a view that does not begin at 16 bytes is copied
// first. W is read by loads to registers, which any address of an element suits.
static StreamArgs stream_args(torch::Tensor& A, const torch::Tensor& W) {
  CHECK_DEV(A); CHECK_BF16(A); CHECK_CONTIG(A);
  CHECK_DEV(W); CHECK_BF16(W); CHECK_CONTIG(W);
  if ((size_t)A.data_ptr() % 16 != 0) A = A.clone();
  StreamArgs a{};
  a.K = A.size(-1);
  TORCH_CHECK(W.dim() == 2 && W.size(1) == a.K && a.K > 0, "A/W K mismatch");
  a.M = A.numel() / a.K;
  a.N = W.size(0);
  TORCH_CHECK(a.M <= 32, "at most 32 rows, got ", a.M);
  a.A = bf_ptr(A);
  a.W = bf_ptr(W);
  return a;
}

// f(rows of A / 16, loads of four of its rows)
template <typename F>
static void by_rows(int M, F f) {
  if (M <= 4) f(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
  else if (M <= 16) f(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
  else f(std::integral_constant<int, 2>{}, std::integral_constant<int, 8>{});
}

// How many parts of K a product of few rows and columns is taken in at once
// (gemm_stream_parts_kernel), 0: none, workgroups of 16 rows of W. Parts pay where these
// leave half of the chip or more idle and theirs fit one round, the more of them the
// longer K. us in a graph, with 0, 2, 4 parts: 1024 x 1024: 1 row 3.6, 3.7, 3.9; x 2048:
// 4.6, 3.7, 4.0; 8 rows 5.1, 4.4; x 3072: 1 row 5.6, 4.8, 4.0; 4 rows 5.7, 5.6, 4.7; 8 rows
// 6.4, 6.2; x 8192: 1 row 10.7, 7.1, 5.3. 2048 x 1024: 3.7, 3.9, 5.0; x 2048: 4.7, 4.0,
// 5.1; x 4096: 6.7, 5.3, 5.3; 4 rows 6.8, 5.8, 6.5; 8 rows 7.5, 6.4. Two rounds: 2560 x
// 2048: 4.8, 5.0, 6.2; 4096 x 4096: 7.9, 7.8, 7.6; 4 rows 7.9, 8.8, 10.1.
static int stream_parts(long M, long N, long K) {
  if (M > 8 || N > 2048 || K <= 1024) return 0;
  return M <= 4 && N <= 1024 && K > 2048 ? 4 : 2;
}

// C(M,N) = A @ W^T [* 1/rms of A's rows] [+ bias] [+ residual], M <= 32; eps < 0: no
// norm.
torch::Tensor gemm_stream(torch::Tensor A, torch::Tensor W,
                          c10::optional<torch::Tensor> residual,
                          c10::optional<torch::Tensor> bias, double eps) {
  StreamArgs a = stream_args(A, W);
  TORCH_CHECK(a.N % 16 == 0 && a.K % 128 == 0, "N%16, K%128 required");
  auto sizes = A.sizes().vec();
  sizes.back() = a.N;
  auto C = torch::empty(sizes, A.options());
  a.C = bf_ptr_mut(C);
  a.eps = eps;
  if (residual.has_value()) {
    TORCH_CHECK(residual->is_cuda() && residual->scalar_type() == at::kBFloat16 &&
                residual->is_contiguous() &&
                residual->numel() == (long)a.M * a.N, "bad residual");
    a.R = bf_ptr(*residual);
  }
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_cuda() && bias->scalar_type() == at::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == a.N, "bad bias");
    a.bias = bf_ptr(*bias);
  }
  if (a.M == 0 || a.N == 0) return C;
  const int parts = eps < 0 ? stream_parts(a.M, a.N, a.K) : 0;
  if (parts) {
    if (parts == 4)
      gemm_stream_parts_kernel<4, 8><<<a.N / 4, 512, 0, cur_stream()>>>(a);
    else
      gemm_stream_parts_kernel<2, 8><<<a.N / 8, 512, 0, cur_stream()>>>(a);
    HIP_OK(hipGetLastError());
    return C;
  }
  by_rows(a.M, [&](auto mt, auto xn) {
    constexpr int MT = decltype(mt)::value, XN = decltype(xn)::value;
    constexpr int DP = MT == 1 ? 4 : 1;
    if (eps >= 0)
      gemm_stream_kernel<EPI_SUM, 1, MT, XN, true, 8, DP>
          <<<a.N / 16, 512, 0, cur_stream()>>>(a);
    else
      gemm_stream_kernel<EPI_SUM, 1, MT, XN, false, 8, DP>
          <<<a.N / 16, 512, 0, cur_stream()>>>(a);
  });
  return C;
}

// Split or unsplit v2 GEMM of the fused forms below; squares of the rows on the way.
template <bool SWIGLU>
static void launch_skinny_fused(const StreamArgs& a, int kchunk, int ksplit,
                                float* part, float* squares) {
  const dim3 grid(a.N / 64, ksplit);
  auto launch = [&](auto mt) {
    gemm_skinny_v2_kernel<decltype(mt)::value, false, SWIGLU, true>
        <<<grid, 256, 0, cur_stream()>>>(a.A, a.W, nullptr, nullptr, a.C, part, a.M,
                                         a.N, a.K, kchunk, ksplit, nullptr, a.eps, 0,
                                         nullptr, 0, squares);
  };
  if (a.M <= 16) launch(std::integral_constant<int, 1>{});
  else launch(std::integral_constant<int, 2>{});
}

// ---------------------------------------------------------------------------
// decode products on a tile of gemm_rows.hip
// ---------------------------------------------------------------------------

// 32 rows by 64 columns, two groups of waves over K, two workgroups a CU: W comes by whole
// lines and by DMA, up to 48 KB ahead a workgroup, and its rows of A once for 64 columns.
typedef RowsTile<32, 64, 2, 1, 2, 3, 2> FewRows;

// Splits of K that let all CUs take part, one or two workgroups each, and do not meet in
// the channels of memory (two splits of up to 8192 do no harm: 8192 x 8192, 32 rows 32.8
// with 2, 34.4 with 3).
static int few_splits(long N, long K) {
  const long wgs = ldiv_up(N, 64);
  int best = 1;
  float most = 0.f;
  for (int s = 1; s <= 16 && (s == 1 || (wgs * s <= 512 && K / s >= 512)); ++s) {
    if (s > 1 && (K > 8192 || s > 2) && same_channels(K, ldiv_up(K / 128, s) * 128))
      continue;
    const float fill = wgs * s / (256.f * ldiv_up(wgs * s, 256));
    if (fill > most + .02f) {
      most = fill;
      best = s;
    }
    if (fill >= .9f) break;
  }
  return best;
}

// The same 32 to 160 columns wide, unsplit. What a CU reads bounds them where memory does
// not: W's columns, A again for every workgroup, 45 B a ns. So the width is the one that
// leaves a CU the fewest columns, and of those the widest, whose workgroups read A the
// least. 32 rows, gated, us for 32, 64, 96, 128 and 160: 28672 x 4096 45.7, 41.6, 50.4, 36.4,
// 38.4; 24576 x 4096 35.0, 36.6, 32.4, 33.7, 36.8; 36864 x 4096 57.0, 57.4, 56.5, 63.5, 46.6;
// 16384 x 4096 24.2, 22.1, 25.3, 28.5, 33.6; 8192 x 4096 14.0, 18.7, 22.8, 26.9, 31.4; 8 rows
// of 28672 x 4096 41.1, 38.6, 47.0, 36.3, 36.8.
static int few_width(long N) {
  int best = 0;
  long least = 0;
  for (int bn : {160, 128, 96, 64, 32}) {
    const long columns = ldiv_up(ldiv_up(N, bn), 256) * bn;
    if (!best || columns < least) {
      best = bn;
      least = columns;
    }
  }
  return best;
}

template <typename F>
static void few_tile(int width, F f) {
  switch (width) {
    case 32: f(RowsTile<32, 32, 2, 1, 2, 4, 2>{}); break;
    case 64: f(FewRows{}); break;
    case 96: f(RowsTile<32, 96, 2, 2, 1, 4, 2>{}); break;
    case 128: f(RowsTile<32, 128, 2, 2, 1, 4, 2>{}); break;
    default: f(RowsTile<32, 160, 2, 2, 1, 4, 2>{}); break;
  }
}

// A sum's width and splits of K: what a CU reads at 45 B a ns, memory at 6.6 TB/s, 2 us of a
// launch, 4 of the fold. 32 rows, us for 32 columns unsplit and 64 in few_splits: 6144 x 4096
// 13.3, 15.5; 8192 x 8192 23.0, 30.8; 8192 x 1024 5.9, 7.0; 4096 x 14336 36, 23.9.
static RowsPlan few_plan(long M, long N, long K) {
  RowsPlan best;
  auto look = [&](int width, int splits) {
    const float cu = ldiv_up(ldiv_up(N, width) * splits, 256) * (width + 32.f) * 2.f *
                     ldiv_up(K / 128, splits) * 128 / 45000.f;
    const float us = std::max(cu, N * K * 2 / 6.6e6f) +
                     (splits > 1 ? 6.f + splits * M * N * 1.6e-6f : 2.f);
    if (us < best.us) best = {width, splits, us};
  };
  look(few_width(N), 1);
  look(64, few_splits(N, K));
  return best;
}

// Whether it beats the gated products of gemm_stream.hip and gemm_skinny.hip, which the
// smallest are left to and those whose W does not begin at 16 bytes. us in a graph, W from
// memory, the faster of those and this: 28672 x 4096: 1 row 45.9, 36.8; 32 rows 46.9, 36.8.
// 57344 x 8192: 161, 146; 183, 162. 36864 x 4096 60.3, 49.5; 72.7, 47.6. 20480 x 5120 46.7,
// 35.4; 57.9, 40.7. 12288 x 1536 11.5, 9.1; 10.8, 9.8. 8192 x 4096 14.5, 12.5; 17.0, 13.9.
// 6144 x 1024 5.6, 5.7; 6.8, 5.7. 22528 x 768 10.6, 8.8; 13.2, 9.4. 1536 x 512 3.8, 3.8; 4.5,
// 4.2. 512 x 256 3.0, 3.3; 8 rows 3.2, 3.4; 32 rows 3.7, 3.5.
static bool few_swiglu(long M, long N, long K) {
  return M > 0 && M <= 32 && K % 128 == 0 && (M > 8 || K > 256 || N > 2048);
}

// Whether it beats the turned projections of gemm_stream.hip and gemm_skinny.hip (a second
// launch folds its splits): few columns leave it too few workgroups for a long K, and the
// smallest are left to the former. us in a graph, W from memory, the faster of those and
// this: 6144 x 4096: 1 row 13.8, 13.5; 8 rows 15.2, 13.5; 32 rows 20.2, 16.2. 4096 x 1024:
// 5.6, 5.5; 6.0, 5.9; 8.2, 7.1. 24576 x 8192 78.6, 70.7; 85.9, 71.8; 106, 74.0. 12288 x 4096
// 25.3, 20.9; 26.4, 21.2; 29.7, 24.9. 2048 x 2048 7.5, 7.0; 7.9, 7.2; 10.1, 8.6. 2048 x 4096
// 8.9, 11.0; 9.4, 11.2; 10.5, 13.0. 1024 x 512 3.8, 4.2; 4.0, 4.3; 5.3, 4.8.
static bool few_rope(long M, long N, long K) {
  return M > 0 && M <= 32 && (K <= 2048 || N >= 4096) && (M > 16 || K >= 1024);
}

// Whether it beats their sums: wherever those want the split form (whose waves take W by
// 64 B of a row), and from some rows on where the one-launch form reads all of A for every
// 16 columns. us in a graph, W from memory, those and this: 4096 x 14336: 9 rows 25.4, 25.7;
// 16 28.4, 25.8; 32 30.9, 26.1. 5120 x 13824: 1 row 36.0, 29.9; 32 40.1, 31.1. 28672 x 4096:
// 44.2, 43.6; 16 48.4, 44.5. 512 x 14336: 15.1, 9.3. 8192 x 28672: 17 rows 99.7, 84.8; 32
// 104.6, 86.4. 151936 x 1024: 16 rows 64.3, 60.6. One launch: 6144 x 4096: 4 rows 14.4, 14.4;
// 16 16.5, 15.0; 32 19.4, 15.9. 20480 x 5120: 4 44.1, 47.0; 16 58.1, 49.2. 4096 x 4096: 16
// 10.3, 11.4; 18176 x 4096, 284 workgroups: 17 rows 36.3, 39.6. 1024 x 3072: any 5.6 to 7.2,
// 6.8 to 7.6. Up to 12 rows of few columns or long K that form keeps up: 9 rows, 4096 x 8192
// 15.5, 17.2; x 16384 30.2, 32.4; 12288 x 16384 76.4, 89.3; but 10240 x 8192 40.4, 37.9.
static bool few_sums(long M, long N, long K) {
  if (M <= 0 || M > 32 || K % 128 || K < 1024 || N <= 0 || N % 8) return false;
  if (K >= 1 << 20 || N >= 1 << 24) return false;   // rows_args
  if (!stream_sums(M, N, K)) return true;
  const long wgs = ldiv_up(N, 64) * few_splits(N, K);
  return M > 8 && (M > 12 || (N > 4096 && K <= 8192)) && N * K >= 24L << 20 && K >= 3072 &&
         wgs * 10 >= ldiv_up(wgs, 256) * 256 * 6;
}

// Whether a sum goes to few_plan's tiles. Beside few_sums, where 64 columns did with W kept
// in the caches: more than one round of 16-row workgroups, and long K, the earlier the more
// rows. us in a graph, W from memory, the faster of gemm_stream.hip and gemm_skinny.hip, and
// this: 8192 x 8192: 1 row 31.1, 25.1; 8 rows 34.1, 25.0. 6144 x 4096 14.6, 13.2; 15.7, 13.2.
// 8192 x 2048 10.4, 8.5; 32 rows 13.2, 9.0. 8192 x 28672 86.8, 78.3; 12 rows 101, 79. 4352 x
// 1024 6.2, 5.3. 4160 x 512 4.2, 4.1; 16384 x 512 5.7, 6.0. One round: 4096 x 11008, 8 rows
// 23.7, 21.0; 3584 x 18944, 1 row 28.2, 29.3, 8 rows 32.4, 30.0; 4096 x 5120, 13 rows 13.2,
// 12.3; 4096 x 4096, 16 rows 10.3, 10.9, 32 rows 12.6, 11.4; 4096 x 3072, 32 rows 9.5, 9.9.
static bool few_wins(long M, long N, long K) {
  if (few_sums(M, N, K)) return true;
  if (M <= 0 || M > 32 || K % 128 || K < 512 || N <= 0 || N % 8) return false;
  if (K >= 1 << 20 || N >= 1 << 24) return false;   // rows_args
  return (N > 4096 && (K >= 1024 || N <= 8192)) || (M >= 8 && K > 8192) ||
         (M >= 13 && K >= 4864) || (M > 16 && K >= 4096);
}

// silu(gate) * up of [gate | up] = rms(A) @ W^T, norm weight folded into W.
torch::Tensor gemm_swiglu(torch::Tensor A, torch::Tensor W, double eps) {
  StreamArgs a = stream_args(A, W);
  TORCH_CHECK(a.K % 256 == 0 && a.N % 64 == 0, "K%256, N%64 required");
  auto sizes = A.sizes().vec();
  sizes.back() = a.N / 2;
  auto C = torch::empty(sizes, A.options());
  a.C = bf_ptr_mut(C);
  a.eps = eps;
  if (a.M == 0) return C;
  if ((size_t)W.data_ptr() % 16 == 0 && few_swiglu(a.M, a.N, a.K)) {
    RowsArgs r{};
    r.A = a.A;
    r.W = a.W;
    r.C = a.C;
    r.M = a.M;
    r.N = a.N;
    r.K = a.K;
    r.splits = 1;
    RowsGlu glu{a.N / 2, a.N / 2, a.N / 2};
    glu.eps = a.eps;
    few_tile(few_width(a.N), [&](auto tile) {
      typedef decltype(tile) T;
      rows_launch(gemm_rows_glu_kernel<T, false, true, true>, ldiv_up(a.N, T::BN),
                  T::THREADS, T::LDS, cur_stream(), r, glu);
    });
    return C;
  }
  if (!stream_swiglu(a.M, a.N, a.K)) {
    launch_skinny_fused<true>(a, a.K, 1, nullptr, nullptr);
    return C;
  }
  by_rows(a.M, [&](auto mt, auto xn) {
    constexpr int MT = decltype(mt)::value, NW = MT == 1 ? 8 : 4;
    gemm_stream_kernel<EPI_SWIGLU, 2, MT, decltype(xn)::value, true, NW, 3 - MT>
        <<<a.N / 32, NW * 64, 0, cur_stream()>>>(a);
  });
  return C;
}

// Where the rotated rows of a fused projection go.
static void rope_args(StreamArgs& a, const torch::Tensor& A, long Hq, long Hkv,
                      const torch::Tensor& cos_t, const torch::Tensor& sin_t,
                      const c10::optional<torch::Tensor>& pos, torch::Tensor& k_pages,
                      torch::Tensor& v_pages, const torch::Tensor& page_table,
                      const torch::Tensor& start_pos) {
  CHECK_DEV_ALL3(k_pages, v_pages, page_table);
  CHECK_DEV_ALL3(cos_t, sin_t, start_pos);
  CHECK_BF16(k_pages); CHECK_BF16(v_pages);
  CHECK_CONTIG(k_pages); CHECK_CONTIG(v_pages); CHECK_CONTIG(page_table);
  a.T = A.size(1);
  a.Hq = Hq; a.Hkv = Hkv;
  a.P = k_pages.size(2); a.D = k_pages.size(3);
  a.maxp = page_table.size(1);
  TORCH_CHECK(a.D % 32 == 0 && a.N == (Hq + 2 * Hkv) * a.D &&
              k_pages.size(1) == Hkv && v_pages.sizes() ==
                  (at::IntArrayRef{k_pages.size(0), Hkv, a.D, a.P}),
              "bad fused qkv shape");
  TORCH_CHECK(page_table.scalar_type() == at::kInt &&
              page_table.size(0) >= A.size(0) &&
              start_pos.scalar_type() == at::kInt &&
              start_pos.numel() >= A.size(0), "bad page table or positions");
  TORCH_CHECK(cos_t.scalar_type() == at::kFloat && cos_t.is_contiguous() &&
              sin_t.scalar_type() == at::kFloat && sin_t.is_contiguous() &&
              cos_t.dim() == 2 && cos_t.size(1) == a.D / 2 &&
              cos_t.sizes() == sin_t.sizes(), "bad rotation tables");
  if (pos.has_value()) {
    CHECK_DEV((*pos));
    TORCH_CHECK(pos->scalar_type() == at::kInt && pos->is_contiguous() &&
                pos->numel() == a.M, "bad position ids");
    a.pos = pos->data_ptr<int>();
  }
  a.cos_t = cos_t.data_ptr<float>();
  a.sin_t = sin_t.data_ptr<float>();
  a.max_pos = cos_t.size(0);
  a.table = page_table.data_ptr<int>();
  a.start = start_pos.data_ptr<int>();
  a.k_pages = bf_ptr_mut(k_pages);
  a.v_pages = bf_ptr_mut(v_pages);
}

// [q | k | v] = rms(A) @ W^T with q turned in the result and k, v in their page slots
// (their columns of the result stay unwritten). A (B, T, K), norm weight folded in.
torch::Tensor gemm_rope_kv(torch::Tensor A, torch::Tensor W, double eps, long Hq,
                           long Hkv,
                           torch::Tensor cos_t, torch::Tensor sin_t,
                           c10::optional<torch::Tensor> pos, torch::Tensor k_pages,
                           torch::Tensor v_pages, torch::Tensor page_table,
                           torch::Tensor start_pos) {
  StreamArgs a = stream_args(A, W);
  TORCH_CHECK(A.dim() == 3 && a.K % 256 == 0 && a.N % 64 == 0,
              "(B, T, K) rows, K%256, N%64 required");
  rope_args(a, A, Hq, Hkv, cos_t, sin_t, pos, k_pages, v_pages, page_table, start_pos);
  auto sizes = A.sizes().vec();
  sizes.back() = a.N;
  auto C = torch::empty(sizes, A.options());
  a.C = bf_ptr_mut(C);
  if (a.M == 0) return C;
  a.eps = eps;
  if ((size_t)W.data_ptr() % 16 == 0 && few_rope(a.M, a.N, a.K)) {
    few_tile(few_width(a.N), [&](auto tile) {
      typedef decltype(tile) T;
      rows_launch(gemm_rows_rope_kernel<T>, ldiv_up(a.N, T::BN), T::THREADS, T::LDS,
                  cur_stream(), a);
    });
    return C;
  }
  if (stream_rope(a.M, a.N, a.K)) {
    by_rows(a.M, [&](auto mt, auto xn) {
      constexpr int MT = decltype(mt)::value;
      gemm_stream_kernel<EPI_ROPE, 2, MT, decltype(xn)::value, true, 4, 4 - MT>
          <<<a.N / 32, 256, 0, cur_stream()>>>(a);
    });
    return C;
  }
  // the split of gemm_skinny's small-N shapes; the fold norms, turns and stores
  const int stages = a.K / 256;
  int ksplit = std::min<int>(
      std::max(1, a.K / 512), std::max(1, std::min(8, 1024 / (a.N / 64))));
  const int per = (stages + ksplit - 1) / ksplit;
  ksplit = (stages + per - 1) / per;
  const long n = (long)ksplit * a.M * a.N;
  auto part = torch::empty({n + ksplit * 32}, A.options().dtype(at::kFloat));
  float* pp = part.data_ptr<float>();
  launch_skinny_fused<false>(a, per * 256, ksplit, pp, pp + n);
  rope_kv_fold_kernel<<<(a.M * (a.N / 2) + 255) / 256, 256, 0, cur_stream()>>>(
      a, pp, pp + n, ksplit);
  return C;
}

// C(M,N) = A(M,K) @ W(N,K)^T [+ residual (M,N)] [+ bias (N,)], M <= 32.
torch::Tensor gemm_skinny(torch::Tensor A, torch::Tensor W,
                          c10::optional<torch::Tensor> residual,
                          c10::optional<torch::Tensor> bias, long ksplit_req,
                          c10::optional<torch::Tensor> norm_w, double eps,
                          c10::optional<torch::Tensor> ss_in,
                          c10::optional<torch::Tensor> ss_out,
                          long norm_mode_req) {
  CHECK_DEV(A); CHECK_BF16(A); CHECK_CONTIG(A);
  CHECK_DEV(W); CHECK_BF16(W); CHECK_CONTIG(W);
  const int K = A.size(-1);
  const int M = A.numel() / K;
  const int N = W.size(0);
  TORCH_CHECK(M <= 32, "gemm_skinny is for M <= 32, got ", M);
  TORCH_CHECK(W.size(1) == K, "A/W K mismatch");
  TORCH_CHECK(K % 32 == 0 && N % 64 == 0 && N > 0, "K%32, N%64 required");
  // norm_mode: 0 none; 1 scale A by invr*norm_w per stage; 2 norm weight
  // pre-folded into W — only the invr accumulator scale remains (cheap).
  int norm_mode = (int)norm_mode_req;
  const unsigned short* nwp = nullptr;
  if (norm_w.has_value()) {
    TORCH_CHECK(norm_w->is_contiguous() && norm_w->numel() == K &&
                norm_w->scalar_type() == at::kBFloat16,
                "norm_w must be contiguous bf16 of length K");
    nwp = bf_ptr(*norm_w);
    if (norm_mode == 0) norm_mode = 1;
  }
  TORCH_CHECK(norm_mode != 1 || nwp, "norm_mode 1 needs norm_w");
  if (norm_mode)
    TORCH_CHECK(K % 256 == 0, "fused rmsnorm needs the v2 (K%256) kernel");
  // ss_in: (nstripes, 32) f32 row sum-of-squares left by the producing
  // GEMM's epilogue — lets the fused rmsnorm skip re-streaming A.
  const float* ssinp = nullptr;
  int nstripes = 0;
  if (ss_in.has_value()) {
    TORCH_CHECK(norm_mode != 0, "ss_in only meaningful with a norm mode");
    TORCH_CHECK(ss_in->is_contiguous() && ss_in->scalar_type() == at::kFloat &&
                ss_in->numel() % 32 == 0, "ss_in must be f32 (nstripes,32)");
    ssinp = ss_in->data_ptr<float>();
    nstripes = (int)(ss_in->numel() / 32);
  }
  float* ssoutp = nullptr;
  if (ss_out.has_value()) {
    TORCH_CHECK(ss_out->is_contiguous() && ss_out->scalar_type() == at::kFloat &&
                ss_out->numel() == (long)(N / 64) * 32,
                "ss_out must be f32 of numel (N/64)*32");
    ssoutp = ss_out->data_ptr<float>();
  }
  auto sizes = A.sizes().vec();
  sizes.back() = N;
  auto C = torch::empty(sizes, A.options());
  if (M == 0) return C;   // missing rows repeat row M - 1
  const unsigned short* rp = nullptr;
  if (residual.has_value()) {
    TORCH_CHECK(residual->is_contiguous() && residual->numel() == (long)M * N);
    rp = bf_ptr(*residual);
  }
  const unsigned short* bp = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_contiguous() && bias->numel() == N);
    bp = bf_ptr(*bias);
  }
  int ksplit = (int)ksplit_req;
  if (ksplit <= 0) {
    // Measured optima (benchmarks/bench_kernels.py gemm): big-N shapes are
    // BW-bound — once N/64 covers the 256 CUs extra splits only add combine
    // traffic; small-N shapes are per-block-latency-bound and want
    // (N/64)*ksplit ~ 512-1024 blocks, capped at 8.
    // BBAMD_GEMM_KSPLIT_BIG: experiment knob for the in-context latency
    // parking the PMC shows on the big MLP GEMMs (prof_ctx r2k).
    static const int ks_big = [] {
      const char* e = std::getenv("BBAMD_GEMM_KSPLIT_BIG");
      return e ? std::atoi(e) : 1;
    }();
    if (N / 64 >= 256) ksplit = ks_big;
    else ksplit = (int)std::min<long>(K / 512,
                                      std::max<long>(1, std::min<long>(8, 1024 / (N / 64))));
    ksplit = std::max(1, ksplit);
  }
  const bool v2 = (K % 256) == 0;
  int kchunk = K;
  if (v2) {
    // v2 stages 256-element chunks: round the K slice to a stage multiple and
    // drop empty trailing splits.
    const int nch = K / 256;
    const int per = (nch + ksplit - 1) / ksplit;
    ksplit = (nch + per - 1) / per;
    kchunk = per * 256;
  }
  torch::Tensor part;
  float* pp = nullptr;
  if (ksplit > 1) {
    part = torch::empty({(long)ksplit, (long)M, (long)N},
                        torch::TensorOptions().device(A.device()).dtype(at::kFloat));
    pp = part.data_ptr<float>();
  }
  dim3 grid(N / 64, ksplit);
  auto launch_v2 = [&](auto mt, auto stage_norm) {
    gemm_skinny_v2_kernel<decltype(mt)::value, decltype(stage_norm)::value>
        <<<grid, 256, 0, cur_stream()>>>(
            bf_ptr(A), bf_ptr(W), ksplit == 1 ? rp : nullptr,
            ksplit == 1 ? bp : nullptr, bf_ptr_mut(C), pp, M, N, K, kchunk,
            ksplit, nwp, (float)eps, norm_mode, ssinp, nstripes,
            ksplit == 1 ? ssoutp : nullptr);
  };
  auto launch = [&](auto mt) {
    if (v2 && norm_mode == 1) launch_v2(mt, std::true_type{});
    else if (v2) launch_v2(mt, std::false_type{});
    else {
      TORCH_CHECK(!norm_mode && (!ssoutp || ksplit > 1),
                  "fused norm / ss_out need the v2 (K%256) kernel");
      gemm_skinny_kernel<decltype(mt)::value><<<grid, 256, 0, cur_stream()>>>(
          bf_ptr(A), bf_ptr(W), ksplit == 1 ? rp : nullptr,
          ksplit == 1 ? bp : nullptr, bf_ptr_mut(C), pp, M, N, K, ksplit);
    }
  };
  if (M <= 16) launch(std::integral_constant<int, 1>{});
  else launch(std::integral_constant<int, 2>{});
  if (ksplit > 1) {
    // the vectorized (float4-per-lane) combine serves both the ss-emitting
    // and plain cases; the flat grid-stride combine remains the fallback
    // for N % 64 != 0 and for narrow N where (N/64, M/16) leaves the grid
    // too small (gemma-class H=2304 -> 36 WGs)
    if (ssoutp || (N % 64 == 0 && N / 64 >= 64)) {
      dim3 cg(N / 64, (M + 15) / 16);
      gemm_skinny_combine_ss_kernel<<<cg, 256, 0, cur_stream()>>>(
          pp, rp, bp, bf_ptr_mut(C), ssoutp, M, N, ksplit);
    } else {
      const long total = (long)M * N;
      const int cgrid = (int)std::min<long>((total + 255) / 256, 2048);
      gemm_skinny_combine_kernel<<<cgrid, 256, 0, cur_stream()>>>(
          pp, rp, bp, bf_ptr_mut(C), M, N, ksplit);
    }
  }
  return C;
}

// ---------------------------------------------------------------------------
// quant4 / selftest
// ---------------------------------------------------------------------------

std::vector<torch::Tensor> quant4_pack(torch::Tensor x) {
  CHECK_DEV(x); CHECK_BF16(x); CHECK_CONTIG(x);
  const long ncols = x.size(-1);
  TORCH_CHECK(ncols % 64 == 0, "quant4 needs cols % 64 == 0");
  const long nrows = x.numel() / ncols;
  auto packed = torch::empty({nrows, ncols / 2},
                             torch::TensorOptions().device(x.device()).dtype(at::kByte));
  auto hopt = torch::TensorOptions().device(x.device()).dtype(at::kHalf);
  auto scale = torch::empty({nrows, ncols / 64}, hopt);
  auto zero = torch::empty({nrows, ncols / 64}, hopt);
  const long ngroups = nrows * (ncols / 64);
  const int wpb = 4;  // waves per block
  quant4_pack_kernel<64><<<(ngroups + wpb - 1) / wpb, wpb * 64, 0, cur_stream()>>>(
      bf_ptr(x), packed.data_ptr<unsigned char>(),
      reinterpret_cast<__half*>(scale.data_ptr()),
      reinterpret_cast<__half*>(zero.data_ptr()), nrows, ncols);
  return {packed, scale, zero};
}

torch::Tensor quant4_unpack(torch::Tensor packed, torch::Tensor scale,
                            torch::Tensor zero) {
  CHECK_DEV(packed);
  const long nrows = packed.size(0), ncols = packed.size(1) * 2;
  auto out = torch::empty({nrows, ncols},
                          torch::TensorOptions().device(packed.device()).dtype(at::kBFloat16));
  const long total = nrows * ncols;
  const int grid = (int)std::min<long>((total + 255) / 256, 4096);
  quant4_unpack_kernel<64><<<grid, 256, 0, cur_stream()>>>(
      packed.data_ptr<unsigned char>(), reinterpret_cast<__half*>(scale.data_ptr()),
      reinterpret_cast<__half*>(zero.data_ptr()), bf_ptr_mut(out), nrows, ncols);
  return out;
}

torch::Tensor kv_stream_probe(torch::Tensor k_pages, torch::Tensor v_pages,
                              torch::Tensor page_table, torch::Tensor ctx_lens,
                              long n_split, bool nt) {
  const int B = page_table.size(0), Hkv = k_pages.size(1);
  const int P = k_pages.size(2), D = k_pages.size(3), maxp = page_table.size(1);
  auto out = torch::empty({(long)B * Hkv * n_split * 4},
                          torch::TensorOptions().device(k_pages.device()).dtype(at::kFloat));
  dim3 grid(B * Hkv, n_split);
  TORCH_CHECK(D == 128);
  if (nt)
    kv_stream_probe_kernel<128, true><<<grid, 256, 0, cur_stream()>>>(
        bf_ptr(k_pages), bf_ptr(v_pages), page_table.data_ptr<int>(),
        ctx_lens.data_ptr<int>(), out.data_ptr<float>(), B, Hkv, P, maxp,
        (int)n_split);
  else
    kv_stream_probe_kernel<128, false><<<grid, 256, 0, cur_stream()>>>(
        bf_ptr(k_pages), bf_ptr(v_pages), page_table.data_ptr<int>(),
        ctx_lens.data_ptr<int>(), out.data_ptr<float>(), B, Hkv, P, maxp,
        (int)n_split);
  return out;
}

torch::Tensor mfma_selftest(torch::Tensor A, torch::Tensor B) {
  CHECK_DEV(A); CHECK_BF16(A); CHECK_CONTIG(A); CHECK_CONTIG(B);
  TORCH_CHECK(A.size(0) == 16 && A.size(1) == 32 && B.size(0) == 32 && B.size(1) == 16);
  auto C = torch::empty({16, 16}, torch::TensorOptions().device(A.device()).dtype(at::kFloat));
  mfma_selftest_kernel<<<1, 64, 0, cur_stream()>>>(bf_ptr(A), bf_ptr(B),
                                                   C.data_ptr<float>());
  return C;
}

// ---------------------------------------------------------------------------
// products of some dozen rows to a thousand (gemm_rows.hip)
// ---------------------------------------------------------------------------

// A tile, what a round of its workgroups costs beside its stages and what a stage of 64
// columns costs, us (a round is 256 workgroups): least squares of the logarithms over 288
// products of 33 to 2000 rows, each with its tiles and splits in a graph; the two lowest
// tiles' stages then by 1116 products, 512 to 49152 columns, K of 512 to 16384, whose W
// comes from memory as a model's does: with .34 and .378 from nearer caches the choice
// took 3.2% more than the best of what it may choose from on average, with these 1.5%
// (6144 x 4096, 250 rows 31.9 us, 29.7; 16384 x 4096, 48 rows 38.2, 32.1).
#define ROWS_TILES(X)                                                                 \
  X(0, 256, 256, 2, 4, 1, 2, 2, 2, 6.0f, 1.08f) X(1, 160, 256, 2, 2, 1, 3, 1, 0, 5.2f, .752f) \
  X(2, 192, 224, 2, 2, 1, 3, 1, 0, 6.0f, .776f) X(3, 256, 160, 2, 2, 1, 3, 1, 0, 6.4f, .757f) \
  X(4, 256, 128, 2, 2, 1, 3, 1, 0, 4.9f, .663f) X(5, 192, 128, 2, 2, 1, 3, 1, 0, 3.7f, .565f) \
  X(6, 128, 128, 2, 2, 1, 4, 1, 0, 2.4f, .462f) X(7, 96, 128, 2, 2, 1, 4, 1, 0, 2.2f, .410f) \
  X(8, 64, 128, 2, 2, 1, 3, 2, 0, 1.1f, .390f) X(9, 96, 64, 2, 1, 2, 3, 1, 0, 2.4f, .265f)

static RowsPlan rows_plan(long M, long N, long K, bool swiglu) {
  static const RowsCost tiles[] = {
#define X(i, bm, bn, wm, wn, wk, st, mw, more, round, stage) {bm, bn, wk, round, stage},
      ROWS_TILES(X)
#undef X
  };
  return rows_best(tiles, 10, M, N, K, swiglu);
}

// The gated product on a tile of its own, unsplit, with what it takes: one wave a SIMD with
// 280 sums a lane reads the least of L2 and of LDS a product, and its height is between
// those whose workgroups leave a round half empty. us, the tile of rows_plan and this: 28672 x
// 4096: 560 rows 135.5, 113.8; 617 134, 112; 640 139, 116; 1200 264, 212; 1900 352, 333. 36864
// x 3072: 300 rows 108, 84. 57344 x 4096: 617 269, 230; 900 365, 333. 14336 x 4096: 1200 135,
// 112. Full rounds of 256 x 256 are faster: 4096 rows of 28672 x 4096 665, 725. Of 224 sizes
// the rule takes 37, all of them faster, by 2 to 25%.
typedef RowsTile<320, 224, 2, 2, 1, 2, 1> TallRows;

static float tall_us(long M, long N, long K) {
  return ldiv_up(ldiv_up(M, TallRows::BM) * ldiv_up(N, TallRows::BN), 256) *
             (6.f + K / 64 * 1.28f) + (N + M) * K / 9.8e6f;
}

static bool rows_tall(long M, long N, long K) {
  return tall_us(M, N, K) < .97f * rows_plan(M, N, K, true).us;
}

// Whether these are the faster form. The library's kernels are at 1.1 to 1.6 PF where
// their tiles fill the chip, which takes many rows or columns; below, and where K is
// long, they leave CUs idle. us in a graph, W from memory, library and these, N x K:
//   28672 x 4096: 97 rows 56, 55; 333 83, 80; 384 85, 81; 450 89, 101; 1000 172, 189
//   4096 x 14336: 97 50, 35; 333 75, 56; 617 114, 79; 1400 165, 159; 2000 184, 185
//   6144 x 4096: 97 24, 23; 333 37, 32; 512 39, 41; 768 51, 48; 2000 78, 93
//   4096 x 4096: 97 17, 16; 333 25, 22; 617 37, 31; 768 35, 35; 1400 52, 50
//   8192 x 28672: 97 198, 108; 512 313, 203; 617 248, 269; 57344 x 8192: 97 183, 178;
//   160 195, 203; 128256 x 4096: 33 208, 189; 87 235, 209; 151936 x 1024: 64 82, 69
//   1024 x 1024: 97 10.7, 7.8; 1024 x 2048: 97 10.8, 9.4; 512 11.4, 13.6; 1024 x 3072: 64
//   11.9, 9.7; 256 10.3, 12.8; 1400 19.4, 18.0
// The last ones' losses are the host's gain where no graph replays them: a call takes 20
// us of its time in the library, 10 to 14 here. Over 1047 products the library takes 1.16
// times as long on average; 1 in 9 is slower here, mostly by 3 to 10%, where its tiles
// happen to fit. Beyond 11.2 million results of up to 384 rows these take 1.08 to 1.11 times
// as long; 385 rows and more are close from 6 to 11 million on (0.9 to 1.07) and left to it.
static bool rows_wins(long M, long N, long K) {
  if (M <= 32 || N <= 0 || N % 8 || K % 64 || K < 256 || K >= 1 << 20) return false;
  return M * N <= (M <= 384 ? 11200000 : 6000000) && (K <= 16384 || M <= 512);
}

// The same for the gated product in one launch: the other way goes over the projection
// once more, which counts the more the shorter K is. 28672 x 4096: 333 rows 73 us (72 +
// 7), 450 116 (106), 768 159 (185), 1400 288 (294), 2800 483 (607), 16384 2674 (2891). Of
// some 390 products that the rule takes, 385 to 16384 rows, 11 are slower by more than 3%,
// where the library's tiles happen to fill its rounds: 1153 rows 276 (262), 2305 507 (487).
static bool rows_swiglu_wins(long M, long N, long K) {
  if (M <= 32 || N <= 0 || N % 16 || K % 64 || K < 256 || (M > 1024 && K > 5120))
    return false;
  if (K >= 1 << 20 || M >= 1 << 24 || N >= 1 << 24) return false;   // rows_args
  const double library = std::max(2e-6 * M * N * K / 1.2e3, (N + M) * K * 2 / 4.7e6);
  return std::min(rows_plan(M, N, K, true).us, tall_us(M, N, K)) * 1.04 <
         library + M * N * 3 / 5e6 + 3;
}

template <typename F>
static void rows_tile(int tile, F f) {
  switch (tile) {
#define X(i, bm, bn, wm, wn, wk, st, mw, more, round, stage) \
  case i:                                              \
    f(RowsTile<bm, bn, wm, wn, wk, st, mw, false, more>{});         \
    break;
    ROWS_TILES(X)
#undef X
    default:
      TORCH_CHECK(false, "no tile");
  }
}

// Both operands come by 16-byte copies: a view that does not begin at 16 bytes is copied
// first.
static RowsArgs rows_args(torch::Tensor& A, torch::Tensor& W) {
  CHECK_DEV(A); CHECK_BF16(A); CHECK_CONTIG(A);
  CHECK_DEV(W); CHECK_BF16(W); CHECK_CONTIG(W);
  if ((size_t)A.data_ptr() % 16) A = A.clone();
  if ((size_t)W.data_ptr() % 16) W = W.clone();
  RowsArgs a{};
  const long K = A.size(-1);
  TORCH_CHECK(W.dim() == 2 && W.size(1) == K && K > 0 && K % 64 == 0 && K < 1 << 20,
              "A/W K mismatch");
  TORCH_CHECK(A.numel() / K < 1 << 24 && W.size(0) < 1 << 24 && W.size(0) > 0);
  a.M = A.numel() / K;
  a.N = W.size(0);
  a.K = K;
  a.splits = 1;
  a.A = bf_ptr(A);
  a.W = bf_ptr(W);
  return a;
}

static void rows_product(RowsArgs& a, const RowsPlan& plan) {
  rows_tile(plan.tile, [&](auto tile) {
    typedef decltype(tile) T;
    rows_launch(a.M <= T::BM ? gemm_rows_kernel<T, true> : gemm_rows_kernel<T>,
                ldiv_up(a.M, T::BM) * ldiv_up(a.N, T::BN) * a.splits, T::THREADS, T::LDS,
                cur_stream(), a);
  });
}

// C(M,N) = A @ W^T [+ bias] [+ residual].
torch::Tensor gemm_rows(torch::Tensor A, torch::Tensor W,
                        c10::optional<torch::Tensor> residual,
                        c10::optional<torch::Tensor> bias) {
  RowsArgs a = rows_args(A, W);
  TORCH_CHECK(a.N % 8 == 0, "N % 8 != 0");
  auto sizes = A.sizes().vec();
  sizes.back() = a.N;
  auto C = torch::empty(sizes, A.options());
  auto operand = [&](c10::optional<torch::Tensor>& t, long n) -> const unsigned short* {
    if (!t.has_value()) return nullptr;
    CHECK_DEV((*t)); CHECK_BF16((*t)); CHECK_CONTIG((*t));
    TORCH_CHECK(t->numel() == n, "size of residual or bias");
    if ((size_t)t->data_ptr() % 16) t = t->clone();
    return bf_ptr(*t);
  };
  a.R = operand(residual, (long)a.M * a.N);
  a.bias = operand(bias, a.N);
  if (a.M == 0) return C;
  const bool few = a.M <= 32 && a.K % 128 == 0;
  const RowsPlan plan =
      few ? few_plan(a.M, a.N, a.K) : rows_plan(a.M, a.N, a.K, false);
  a.splits = plan.splits;
  a.C = plan.splits > 1 ? nullptr : bf_ptr_mut(C);
  torch::Tensor part;
  if (plan.splits > 1) {
    part = torch::empty({plan.splits, a.M, a.N}, A.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  }
  if (few)
    few_tile(plan.tile, [&](auto tile) {
      typedef decltype(tile) T;
      rows_launch(gemm_rows_kernel<T, true>, ldiv_up(a.N, T::BN) * a.splits, T::THREADS,
                  T::LDS, cur_stream(), a);
    });
  else
    rows_product(a, plan);
  if (plan.splits > 1) {
    a.C = bf_ptr_mut(C);
    gemm_rows_fold_kernel<<<ldiv_up((long)a.M * a.N, 2048), 256, 0, cur_stream()>>>(a);
    HIP_OK(hipGetLastError());
  }
  return C;
}

// h = A @ W^T + residual and its RMS norm, (h, y). Where the product is split, its fold makes
// both.
std::vector<torch::Tensor> gemm_rows_norm(torch::Tensor A, torch::Tensor W,
                                          torch::Tensor residual, torch::Tensor weight,
                                          double eps) {
  RowsArgs a = rows_args(A, W);
  TORCH_CHECK(a.N % 8 == 0, "N % 8 != 0");
  auto operand = [&](torch::Tensor& t, long n) {
    CHECK_DEV(t); CHECK_BF16(t); CHECK_CONTIG(t);
    TORCH_CHECK(t.numel() == n, "size of residual or weight");
    if ((size_t)t.data_ptr() % 16) t = t.clone();
    return bf_ptr(t);
  };
  const unsigned short* w = operand(weight, a.N);
  const unsigned short* r = operand(residual, (long)a.M * a.N);
  TORCH_CHECK(a.N <= 16384, "columns");
  const RowsPlan plan = rows_plan(a.M, a.N, a.K, false);
  if (a.M == 0 || plan.splits == 1)
    return rms_norm_residual(gemm_rows(A, W, c10::nullopt, c10::nullopt), residual, weight, eps);
  auto sizes = A.sizes().vec();
  sizes.back() = a.N;
  auto h = torch::empty(sizes, A.options()), y = torch::empty(sizes, A.options());
  auto part = torch::empty({plan.splits, a.M, a.N}, A.options().dtype(at::kFloat));
  a.splits = plan.splits;
  a.part = part.data_ptr<float>();
  rows_product(a, plan);
  a.C = bf_ptr_mut(h);
  a.R = r;
  auto fold = [&](auto iters) {
    gemm_rows_fold_norm_kernel<decltype(iters)::value>
        <<<a.M, 512, 0, cur_stream()>>>(a, w, bf_ptr_mut(y), (float)eps);
  };
  if (a.N <= 4096) fold(std::integral_constant<int, 1>{});
  else if (a.N <= 8192) fold(std::integral_constant<int, 2>{});
  else fold(std::integral_constant<int, 4>{});
  HIP_OK(hipGetLastError());
  return {h, y};
}

// rope_kv_write_ of A @ W^T: (B, T, (Hq + 2 Hkv) * D) with the turned queries; keys and
// values are in the pages. Where the product is split and a sequence has a few tokens (its
// values go to their pages one by one), its fold does it.
torch::Tensor gemm_rows_rope_kv(torch::Tensor A, torch::Tensor W, long Hq, long Hkv,
                                torch::Tensor cos_t, torch::Tensor sin_t,
                                c10::optional<torch::Tensor> pos, torch::Tensor k_pages,
                                torch::Tensor v_pages, torch::Tensor page_table,
                                torch::Tensor start_pos) {
  TORCH_CHECK(A.dim() == 3, "(B, T, K) rows");
  RowsArgs a = rows_args(A, W);
  TORCH_CHECK(a.N % 8 == 0, "N % 8 != 0");
  StreamArgs r{};
  r.M = a.M;
  r.N = a.N;
  rope_args(r, A, Hq, Hkv, cos_t, sin_t, pos, k_pages, v_pages, page_table, start_pos);
  auto C = torch::empty({A.size(0), A.size(1), a.N}, A.options());
  if (a.M == 0) return C;
  const RowsPlan plan = rows_plan(a.M, a.N, a.K, false);
  a.splits = plan.splits;
  const bool fold = plan.splits > 1 && r.T <= 4 && r.D <= 256 && (r.D & (r.D - 1)) == 0 &&
                    (size_t)k_pages.data_ptr() % 16 == 0;
  torch::Tensor part;
  if (plan.splits > 1) {
    part = torch::empty({plan.splits, a.M, a.N}, A.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  } else {
    a.C = bf_ptr_mut(C);
  }
  rows_product(a, plan);
  if (fold) {
    a.C = r.C = bf_ptr_mut(C);
    const long items = (long)a.M * (a.N / 16);
    gemm_rows_fold_rope_kernel<<<ldiv_up(items, 256), 256, 0, cur_stream()>>>(a, r);
    HIP_OK(hipGetLastError());
    return C;
  }
  if (plan.splits > 1) {
    a.C = bf_ptr_mut(C);
    gemm_rows_fold_kernel<<<ldiv_up((long)a.M * a.N, 2048), 256, 0, cur_stream()>>>(a);
    HIP_OK(hipGetLastError());
  }
  rope_kv_write_(C, Hq, Hkv, cos_t, sin_t, pos, k_pages, v_pages, page_table, start_pos,
                 c10::nullopt, c10::nullopt, 0.0);
  return C;
}

template <bool CLAMPED>
static void rows_glu(RowsArgs& a, const RowsGlu& glu) {
  auto launch = [&](auto tile) {
    typedef decltype(tile) T;
    if constexpr (T::WK == 1)
      rows_launch(a.M <= T::BM ? gemm_rows_glu_kernel<T, CLAMPED, false, true>
                               : gemm_rows_glu_kernel<T, CLAMPED>,
                  ldiv_up(a.M, T::BM) * ldiv_up(glu.ldc, T::BN / 2), T::THREADS, T::LDS,
                  cur_stream(), a, glu);
  };
  if (rows_tall(a.M, 2L * glu.F, a.K)) launch(TallRows{});
  else rows_tile(rows_plan(a.M, 2L * glu.F, a.K, true).tile, launch);
}

// swiglu(A @ W^T) of a fused [gate | up] W: (..., N / 2).
torch::Tensor gemm_rows_swiglu(torch::Tensor A, torch::Tensor W) {
  RowsArgs a = rows_args(A, W);
  TORCH_CHECK(a.N % 16 == 0, "N % 16 != 0");
  auto sizes = A.sizes().vec();
  sizes.back() = a.N / 2;
  auto C = torch::empty(sizes, A.options());
  if (a.M == 0) return C;
  a.C = bf_ptr_mut(C);
  rows_glu<false>(a, RowsGlu{a.N / 2, a.N / 2, a.N / 2});
  return C;
}

// The clamped gated product of rows 0 .. F - 1 of W, gates, and up .. up + F - 1:
// (M, cols) with zeros behind F.
torch::Tensor gemm_rows_glu(torch::Tensor A, torch::Tensor W, long up, long F, long cols,
                            c10::optional<torch::Tensor> gate_b,
                            c10::optional<torch::Tensor> up_b, double limit,
                            double slope) {
  RowsArgs a = rows_args(A, W);
  TORCH_CHECK(A.dim() == 2 && F > 0 && F % 8 == 0 && cols % 8 == 0 && cols >= F &&
              up >= 0 && up + F <= a.N && cols < 1 << 24, "bad gated product");
  auto bias = [&](const c10::optional<torch::Tensor>& t) -> const float* {
    if (!t.has_value()) return nullptr;
    TORCH_CHECK(t->is_cuda() && t->scalar_type() == at::kFloat && t->is_contiguous() &&
                t->numel() >= F, "bad bias");
    return t->data_ptr<float>();
  };
  RowsGlu glu{(int)up, (int)F, (int)cols, bias(gate_b), bias(up_b), (float)limit,
              (float)slope};
  auto C = torch::empty({a.M, cols}, A.options());
  if (a.M == 0) return C;
  a.C = bf_ptr_mut(C);
  rows_glu<true>(a, glu);
  return C;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm);
  m.def("rms_norm_residual", &rms_norm_residual);
  m.def("layer_norm", &layer_norm);
  m.def("rope_apply_", &rope_apply_);
  m.def("swiglu", &swiglu);
  m.def("gelu_tanh", &gelu_tanh);
  m.def("add_bf16", &add_bf16);
  m.def("kv_write", &kv_write);
  m.def("kv_gather", &kv_gather);
  m.def("wire_deflate", &wire_deflate);
  m.def("wire_inflate", &wire_inflate);
  m.def("wire_deflate_mt", &wire_deflate_mt);
  m.def("wire_inflate_mt", &wire_inflate_mt);
  m.def("attn_decode", &attn_decode);
  m.def("attn_decode_qkv", &attn_decode_qkv);
  m.def("attn_prefill_qkv", &attn_prefill_qkv, py::arg("qkv"), py::arg("Hq"),
        py::arg("k_pages"), py::arg("v_pages"), py::arg("page_table"),
        py::arg("q_start"), py::arg("scale"), py::arg("window"), py::arg("tree_mask"),
        py::arg("longest") = 0);
  m.def("rope_kv_write_", &rope_kv_write_);
  m.def("norm_route", &norm_route);
  m.def("add_experts", &add_experts);
  m.def("gemm_stream", &gemm_stream);
  m.def("few_sums", &few_sums);
  m.def("few_wins", &few_wins);
  m.def("few_splits", &few_splits);
  m.def("few_swiglu", &few_swiglu);
  m.def("few_width", &few_width);
  m.def("few_rope", &few_rope);
  m.def("few_plan", [](long M, long N, long K) {
    const RowsPlan p = few_plan(M, N, K);
    return std::make_pair(p.tile, p.splits);
  });
  m.def("rows_wins", &rows_wins);
  m.def("rows_swiglu_wins", &rows_swiglu_wins);
  m.def("rows_tall", &rows_tall);
  m.def("decode_even", &decode_even);
  m.def("rows_plan", [](long M, long N, long K, bool swiglu) {
    const RowsPlan p = rows_plan(M, N, K, swiglu);
    return py::make_tuple(p.tile, p.splits);
  });
  m.def("gemm_rows", &gemm_rows);
  m.def("gemm_rows_norm", &gemm_rows_norm);
  m.def("gemm_rows_rope_kv", &gemm_rows_rope_kv);
  m.def("gemm_rows_swiglu", &gemm_rows_swiglu);
  m.def("gemm_rows_glu", &gemm_rows_glu);
  m.def("gemm_swiglu", &gemm_swiglu);
  m.def("gemm_rope_kv", &gemm_rope_kv);
  m.def("stream_rows", &stream_rows);
  m.def("stream_swiglu", &stream_swiglu);
  m.def("stream_sums", &stream_sums);
  m.def("stream_parts", &stream_parts);
  m.def("stream_rope", &stream_rope);
  m.def("attn_prefill", &attn_prefill, py::arg("q"), py::arg("k_pages"),
        py::arg("v_pages"), py::arg("page_table"), py::arg("q_start"), py::arg("scale"),
        py::arg("window"), py::arg("alibi"), py::arg("tree_mask"),
        py::arg("longest") = 0);
  m.def("prefill_plan", [](long B, int Hq, int Hkv, int Tq, int D, int P, long keys,
                           bool tree, int window) {
    const PrefillPlan p = prefill_plan(B * Hkv, Hq / Hkv, Tq, D, P, keys, tree, window);
    return py::make_tuple(p.splits, p.two ? 2 : 1);
  });
  m.def("gemm_skinny", &gemm_skinny, py::arg("A"), py::arg("W"),
        py::arg("residual") = c10::nullopt, py::arg("bias") = c10::nullopt,
        py::arg("ksplit") = 0, py::arg("norm_w") = c10::nullopt,
        py::arg("eps") = 0.0, py::arg("ss_in") = c10::nullopt,
        py::arg("ss_out") = c10::nullopt, py::arg("norm_mode") = 0);
  m.def("moe_gemm", &moe_gemm);
  m.def("gemm_w4", &gemm_w4);
  m.def("quant4_pack", &quant4_pack);
  m.def("quant4_unpack", &quant4_unpack);
  m.def("mfma_selftest", &mfma_selftest);
  m.def("kv_stream_probe", &kv_stream_probe);
}
