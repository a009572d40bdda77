// Torch bindings of the training path's kernels.

#include <torch/extension.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include "attn_train.hip"
#include "gemm_grad.hip"
#include "gemm_rows_host.h"
#include "train_rows.hip"

using torch::Tensor;
using OptTensor = c10::optional<Tensor>;

static hipStream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

#define CHECK_T(x, st)                                                        \
  TORCH_CHECK((x).is_cuda() && (x).is_contiguous() &&                         \
                  (x).scalar_type() == (st),                                  \
              #x " must be a contiguous device tensor of ", toString(st))

// Rows that are read 16 bytes at a time, by the kernels or by copies to LDS.
#define CHECK_ROWS(x)                                                         \
  CHECK_T(x, at::kBFloat16);                                                  \
  TORCH_CHECK((size_t)(x).data_ptr() % 16 == 0,                               \
              #x " must be aligned to 16 bytes")

static void check_launch() {
  const hipError_t e = hipGetLastError();
  TORCH_CHECK(e == hipSuccess, "kernel launch: ", hipGetErrorString(e));
}

static const unsigned short* in(const Tensor& t) {
  return reinterpret_cast<const unsigned short*>(t.data_ptr());
}
static unsigned short* out(const Tensor& t) {
  return reinterpret_cast<unsigned short*>(t.data_ptr());
}

// Sizes of a fused projection (B, T, (Hq + 2 Hkv) * D), positions from `start`.
static TrainAttnArgs attn_args(const Tensor& qkv, long Hq, long Hkv,
                               const Tensor& cos_t, const Tensor& sin_t, long start,
                               double scale) {
  CHECK_ROWS(qkv);
  CHECK_T(cos_t, at::kFloat);
  CHECK_T(sin_t, at::kFloat);
  TORCH_CHECK(Hkv > 0 && Hq > 0 && Hq % Hkv == 0, "heads: ", Hq, " on ", Hkv);
  TORCH_CHECK(qkv.dim() == 3 && qkv.size(2) % (Hq + 2 * Hkv) == 0 &&
                  qkv.numel() > 0,
              "bad fused qkv shape");
  const long D = qkv.size(2) / (Hq + 2 * Hkv);
  TORCH_CHECK(D == 64 || D == 128, "unsupported head_dim ", D);
  TORCH_CHECK(cos_t.dim() == 2 && cos_t.size(1) == D / 2 &&
                  cos_t.sizes() == sin_t.sizes(),
              "bad rotation tables");
  TORCH_CHECK(start >= 0 && start + qkv.size(1) <= cos_t.size(0),
              "positions beyond the rotation tables");
  TORCH_CHECK(qkv.size(1) * (Hq / Hkv) < (1L << 30), "too many rows");
  TORCH_CHECK(scale > 0, "scale must be positive");
  TrainAttnArgs a{};
  a.qkv = in(qkv);
  a.cos_t = cos_t.data_ptr<float>();
  a.sin_t = sin_t.data_ptr<float>();
  a.B = qkv.size(0);
  a.T = qkv.size(1);
  a.Hkv = Hkv;
  a.G = Hq / Hkv;
  a.start = start;
  a.scale = scale;
  return a;
}

template <typename F>
static void by_head(long D, F f) {
  if (D == 128) f(std::integral_constant<int, 128>{});
  else f(std::integral_constant<int, 64>{});
}

// (result, rotated queries and keys, 32-bit result, log-sums); without `grad` the
// last two are empty.
std::vector<Tensor> rope_attention(Tensor qkv, long Hq, long Hkv, Tensor cos_t,
                                   Tensor sin_t, long start, double scale,
                                   bool grad) {
  TrainAttnArgs a = attn_args(qkv, Hq, Hkv, cos_t, sin_t, start, scale);
  const long D = qkv.size(2) / (Hq + 2 * Hkv), B = a.B, T = a.T;
  Tensor qk = torch::empty({B, T, (Hq + Hkv) * D}, qkv.options());
  Tensor o = torch::empty({B, T, Hq * D}, qkv.options());
  const auto f32 = qkv.options().dtype(at::kFloat);
  Tensor o32 = torch::empty({grad ? B : 0, T, Hq * D}, f32);
  Tensor lse = torch::empty({grad ? B * Hkv : 0, T * a.G}, f32);
  a.qk = in(qk);
  a.out = out(o);
  if (grad) {
    a.out32 = o32.data_ptr<float>();
    a.lse = lse.data_ptr<float>();
  }
  const long pairs = B * T * (Hq + Hkv) * D / 16;
  rope_rows_kernel<<<(pairs + 255) / 256, 256, 0, stream()>>>(
      a.qkv, out(qk), a.cos_t, a.sin_t, B * T, T, Hq + Hkv, Hq + 2 * Hkv, D, start);
  by_head(D, [&](auto d) {
    attn_train_kernel<decltype(d)::value>
        <<<dim3(B * Hkv, (T * a.G + 127) / 128), 256, 0, stream()>>>(a);
  });
  check_launch();
  return {o, qk, o32, lse};
}

Tensor rope_attention_grad(Tensor gout, Tensor qkv, Tensor qk, Tensor o32,
                           Tensor lse, long Hq, long Hkv, Tensor cos_t, Tensor sin_t,
                           long start, double scale) {
  TrainAttnArgs a = attn_args(qkv, Hq, Hkv, cos_t, sin_t, start, scale);
  const long D = qkv.size(2) / (Hq + 2 * Hkv), B = a.B, T = a.T;
  CHECK_ROWS(gout);
  CHECK_ROWS(qk);
  CHECK_T(o32, at::kFloat);
  CHECK_T(lse, at::kFloat);
  TORCH_CHECK(gout.numel() == B * T * Hq * D && o32.numel() == gout.numel() &&
                  qk.numel() == B * T * (Hq + Hkv) * D &&
                  lse.numel() == B * T * Hq,
              "gradient of another shape");
  Tensor delta = torch::empty_like(lse);
  Tensor dqkv = torch::empty_like(qkv);
  a.qk = in(qk);
  a.dout = in(gout);
  a.out32 = o32.data_ptr<float>();
  a.lse = lse.data_ptr<float>();
  a.delta = delta.data_ptr<float>();
  a.dqkv = out(dqkv);
  by_head(D, [&](auto d) {
    constexpr int DD = decltype(d)::value;
    attn_train_dq_kernel<DD>
        <<<dim3(B * Hkv, (T * a.G + 127) / 128), 256, 0, stream()>>>(a);
    constexpr int lds = TrainRing<DD>::BYTES;
    TORCH_CHECK(hipFuncSetAttribute(
                    reinterpret_cast<const void*>(attn_train_dkv_kernel<DD>),
                    hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess,
                "cannot reserve ", lds, " bytes of LDS");
    attn_train_dkv_kernel<DD>
        <<<dim3(B * Hkv, (T + 63) / 64), 256, lds, stream()>>>(a);
  });
  check_launch();
  return dqkv;
}

Tensor rms_norm_grad(Tensor x, Tensor w, Tensor gy, OptTensor gx, double eps) {
  CHECK_ROWS(x);
  CHECK_ROWS(w);
  CHECK_ROWS(gy);
  const long H = x.size(-1);
  TORCH_CHECK(H % 8 == 0 && H <= 16384 && w.numel() == H &&
                  gy.numel() == x.numel(),
              "bad norm shapes");
  if (gx.has_value()) {
    CHECK_ROWS((*gx));
    TORCH_CHECK(gx->numel() == x.numel());
  }
  Tensor dx = torch::empty_like(x);
  if (x.numel() == 0) return dx;
  auto launch = [&](auto it) {
    rms_norm_grad_kernel<decltype(it)::value>
        <<<x.numel() / H, 256, 0, stream()>>>(
            in(x), in(w), in(gy), gx.has_value() ? in(*gx) : nullptr, out(dx), H,
            (float)eps);
  };
  if (H <= 2048) launch(std::integral_constant<int, 1>{});
  else if (H <= 4096) launch(std::integral_constant<int, 2>{});
  else if (H <= 8192) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 8>{});
  check_launch();
  return dx;
}

Tensor swiglu_grad(Tensor gu, Tensor gm) {
  CHECK_ROWS(gu);
  CHECK_ROWS(gm);
  const long I = gm.size(-1);
  TORCH_CHECK(I % 8 == 0 && gu.size(-1) == 2 * I && gu.numel() == 2 * gm.numel(),
              "bad product shapes");
  Tensor dgu = torch::empty_like(gu);
  if (gm.numel() == 0) return dgu;
  const long N = gm.numel() / I;
  swiglu_grad_kernel<<<std::min<long>((N * I / 8 + 255) / 256, 4096), 256, 0,
                       stream()>>>(in(gu), in(gm), out(dgu), N, I);
  check_launch();
  return dgu;
}

// Tiles of gemm_rows.hip whose sums run over rows of w, and what their rounds and stages
// cost: fitted to 192 products, 33 to 2000 rows, where the choice takes 2.5% more than
// the best of eleven tiles and up to 16 splits.
#define GRAD_TILES(X)                                                                     \
  X(0, 256, 256, 2, 4, 2, 2, 2, 6.0f, 1.15f) X(1, 160, 256, 2, 2, 3, 1, 0, 6.7f, .854f)         \
  X(2, 128, 256, 2, 4, 3, 2, 0, 3.3f, .664f) X(3, 192, 128, 2, 2, 3, 1, 0, 5.1f, .587f)          \
  X(4, 128, 128, 2, 2, 4, 1, 0, 4.2f, .476f) X(5, 96, 128, 2, 2, 4, 1, 0, 3.8f, .406f)           \
  X(6, 64, 128, 2, 2, 3, 2, 0, 2.6f, .340f)

static RowsPlan grad_plan(long M, long N, long K) {
  static const RowsCost tiles[] = {
#define X(i, bm, bn, wm, wn, st, mw, more, round, stage) {bm, bn, 1, round, stage},
      GRAD_TILES(X)
#undef X
  };
  return rows_best(tiles, 7, M, K, N, false, true);
}

// Whether linear_grad beats the library's GEMM, which leaves CUs idle where the result
// has few tiles. us in a graph, w from memory, library and here, rows of w x columns:
//   28672 x 4096: 1 row 146, 47; 33 160, 48; 128 143, 57; 450 276, 110; 1024 344, 186; 1400
//   305, 330;  38400 x 4096: 1024 460, 247;  57344 x 4096: 1024 532, 351
//   4096 x 14336: 1 29, 26; 33 37, 27; 450 67, 59; 768 87, 81; 1700 165, 174
//   6144 x 4096: 1 34, 14; 33 29, 15; 450 54, 38; 1400 73, 70; 2000 95, 84; 2500 107, 111
//   4096 x 4096: 450 39, 30; 2000 67, 58; 2500 75, 78;  1024 x 2048: 1 6, 8; 64 9, 8
//   8192 x 28672: 200 143, 129; 333 161, 178; 900 369, 349
//   57344 x 8192: 128 298, 172; 333 351, 369; 450 543, 362; 513 501, 515; 900 742, 685
// Its form for rows of w to sum over is 4 to 8% slower than that for columns, these are
// not, but take tiles of 256 x 256, and 3000 rows of few columns leave a quarter of the
// chip idle: 28672 x 4096, 3000 rows 550, 600; 4000 700, 660; 8000 1392, 1337. 4096 x 14336:
// 3000 315, 284; 8000 737, 682. 6144 x 4096: 3000 125, 128; 4000 158, 149; 8000 305, 287.
static bool linear_grad_wins(long M, long N, long K) {
  return N > 0 && N % 64 == 0 && K > 0 && K % 256 == 0 &&
         (M >= (N >= 3 * K ? 3600 : 3000) || (M <= 1024 && N >= 4 * K && K <= 5120) ||
          (M * K <= 8500000 && (M <= 512 || M * K * N <= 150000000000L)));
}

// g (M, N) @ w (N, K) -> (M, K); splits <= 0: as many as the sizes want.
Tensor linear_grad(Tensor g, Tensor w, long splits) {
  CHECK_ROWS(g);
  CHECK_ROWS(w);
  TORCH_CHECK(g.dim() == 2 && w.dim() == 2 && g.size(1) == w.size(0) &&
                  g.size(0) < (1L << 30) && w.size(0) % 32 == 0 &&
                  w.size(1) % 256 == 0 && w.numel() > 0 && w.numel() < (1L << 40),
              "need (M, N) @ (N, K), N % 32 == 0, K % 256 == 0");
  const long M = g.size(0), N = w.size(0), K = w.size(1);
  Tensor c = torch::empty({M, K}, g.options());
  if (M == 0) return c;
  Tensor part;
  auto parts = [&](long n) {
    part = torch::empty({n, M, K}, g.options().dtype(at::kFloat));
    return part.data_ptr<float>();
  };
  // a tile's 256 rows of g and a stage's 64 of w lie within 32 bits of bytes
  if (N % 64 == 0 && K < (1L << 24) && N < (1L << 23)) {
    RowsPlan plan = grad_plan(M, N, K);
    if (splits > 0) plan.splits = (int)std::min<long>(splits, N / 64);
    RowsArgs a{};
    a.A = in(g);
    a.W = in(w);
    a.M = M;
    a.N = K;
    a.K = N;
    a.splits = plan.splits;
    if (a.splits > 1) a.part = parts(a.splits);
    else a.C = out(c);
    switch (plan.tile) {
#define X(i, bm, bn, wm, wn, st, mw, more, round, stage)                                      \
  case i: {                                                                             \
    typedef RowsTile<bm, bn, wm, wn, 1, st, mw, true, more> T;                                \
    rows_launch(gemm_rows_kernel<T>, ldiv_up(M, bm) * ldiv_up(K, bn) * a.splits,        \
                T::THREADS, T::LDS, stream(), a);                                       \
    break;                                                                              \
  }
      GRAD_TILES(X)
#undef X
    }
    if (a.splits > 1) {
      a.C = out(c);
      gemm_rows_fold_kernel<<<ldiv_up(M * K, 2048), 256, 0, stream()>>>(a);
      check_launch();
    }
    return c;
  }
  GemmGradArgs a{};
  a.A = in(g);
  a.W = in(w);
  a.M = M;
  a.N = N;
  a.K = K;
  const long tiles = ((a.M + 127) / 128) * (a.K / 256);
  if (splits <= 0) splits = std::min<long>(32, 512 / std::max<long>(1, tiles));
  a.splits = (int)std::max<long>(1, std::min<long>(splits, a.N / 256));
  if (a.splits > 1) a.part = parts(a.splits);
  else a.C = out(c);
  gemm_grad_kernel<<<tiles * a.splits, 256, 0, stream()>>>(a);
  check_launch();
  if (a.splits > 1) {
    gemm_grad_fold_kernel<<<(c.numel() / 8 + 255) / 256, 256, 0, stream()>>>(
        a.part, out(c), c.numel(), a.splits);
    check_launch();
  }
  return c;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("linear_grad", &linear_grad);
  m.def("linear_grad_wins", &linear_grad_wins);
  m.def("linear_grad_plan", [](long M, long N, long K) {
    const RowsPlan p = grad_plan(M, N, K);
    return py::make_tuple(p.tile, p.splits);
  });
  m.def("rope_attention", &rope_attention);
  m.def("rope_attention_grad", &rope_attention_grad);
  m.def("rms_norm_grad", &rms_norm_grad);
  m.def("swiglu_grad", &swiglu_grad);
}
