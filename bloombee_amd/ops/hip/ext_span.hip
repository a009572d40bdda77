// Torch bindings of the one-launch decode step (module _hip_span).
#include "host.h"
#include "decode_span.hip"

namespace {

bool aligned16(const Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

template <class Sizes>
int most_units(int M, int H, int I, int qkv_rows) {
  constexpr int QU = Sizes::Qkv::UNITS, OU = Sizes::O::UNITS, GU = Sizes::Glu::UNITS,
                DU = Sizes::Down::UNITS;
  auto padded = [](long all, int per, int U) {
    const long slots = span::SLOTS - (Sizes::SPARES ? span::MOST_SPARED : 0);
    const long most = (all + slots - 1) / slots;
    return (int)((most + per - 1) / per * U);
  };
  return std::max({padded(qkv_rows / 4, QU, QU), padded(H / 4, OU, OU),
                   padded(I / 4, GU / 2, GU), padded(H / 4, DU, DU)});
}

struct Lds { int units, wide, sums, squares, control, all; };

Lds lds_of(int M, int H, int I, int Hq, int Hkv, int units) {
  Lds l;
  l.units = units;
  l.wide = M * H * 2;
  l.sums = l.wide + std::max({M * Hq * span::HEAD * 2, M * I * 2,
                              span::attention_lds(Hq / Hkv),
                              span::SLOTS / (M * Hkv) * span::PART_FLOATS * 4});
  l.sums = (l.sums + 15) / 16 * 16;
  l.squares = l.sums + units * M * span::PITCH * 4;
  l.control = l.squares + span::NW * 16 * 4;
  l.all = l.control + (int)sizeof(span::Control);
  return l;
}

// Everything that a slot of a small model has of a layer is in registers at once, also
// where some slots have attention only.
bool small_model(int H, int I, int Hq, int Hkv) {
  auto most = [](long units) {
    const long slots = span::SLOTS - span::MOST_SPARED;
    return (units + slots - 1) / slots;
  };
  using S = span::SmallSizes;
  return H <= 1024 && Hq * span::HEAD <= 2048 && I <= 3072 &&
         most((Hq + 2L * Hkv) * span::HEAD / 4) <= S::Qkv::UNITS &&
         most(H / 4) <= S::O::UNITS && most(I / 4) <= S::Glu::UNITS / 2;
}

Lds lds_of(int M, int H, int I, int Hq, int Hkv) {
  const int rows = (Hq + 2 * Hkv) * span::HEAD;
  return lds_of(M, H, I, Hq, Hkv,
                small_model(H, I, Hq, Hkv)
                    ? most_units<span::SmallSizes>(M, H, I, rows)
                    : most_units<span::LargeSizes>(M, H, I, rows));
}

}  // namespace

// Whether these sizes can be run.
bool span_fits(long M, long H, long I, long Hq, long Hkv, long D, long P) {
  if (M < 1 || M > span::MAX_ROWS || D != span::HEAD || Hkv < 1 || Hq % Hkv ||
      Hq / Hkv > 8 || M * Hkv > span::SLOTS || (P != 8 && P != 16 && P != 32) ||
      H < 128 || I < 128 || H % 256 || I % 256 || Hq % 2 || H > 16384 || I > 65536 || Hq > 128 ||
      4 * I * H >= 1L << 32 || (Hq + 2 * Hkv) * D * H * 2 >= 1L << 32)
    return false;
  return lds_of((int)M, (int)H, (int)I, (int)Hq, (int)Hkv).all <= 160 * 1024;
}

namespace {

bool plain(const Tensor& t, at::ScalarType type, const Tensor& like) {
  return t.is_cuda() && t.is_contiguous() && t.scalar_type() == type &&
         t.device() == like.device();
}

}  // namespace

// Whether decode_span takes these; the same arguments.
static bool span_takes(Tensor hidden, std::vector<Tensor> weights, long Hq, Tensor cos_t,
                Tensor sin_t, OptTensor pos, Tensor start, Tensor table) {
  if (!plain(hidden, at::kBFloat16, hidden) || hidden.dim() != 3 || hidden.size(1) != 1 ||
      weights.empty() || weights.size() % 8 || weights[6].dim() != 4 ||
      weights[3].dim() != 2)
    return false;
  const long M = hidden.size(0), H = hidden.size(2), I = weights[3].size(1);
  const long np = weights[6].size(0), Hkv = weights[6].size(1), P = weights[6].size(2);
  const long D = weights[6].size(3);
  if (!span_fits(M, H, I, Hq, Hkv, D, P)) return false;
  if (!plain(start, at::kInt, hidden) || start.numel() != M || !table.is_cuda() ||
      table.device() != hidden.device() || table.scalar_type() != at::kInt ||
      table.dim() != 2 || table.size(0) != M || table.size(1) < 1 ||
      table.stride(1) != 1 || (M > 1 && table.stride(0) < table.size(1)))
    return false;
  for (const Tensor& t : {cos_t, sin_t})
    if (!plain(t, at::kFloat, hidden) || t.dim() != 2 || t.size(1) != D / 2 ||
        t.size(0) < 1 || t.size(0) != cos_t.size(0))
      return false;
  if (pos && (!plain(*pos, at::kInt, hidden) || pos->numel() != M)) return false;
  const std::vector<std::vector<long>> sizes = {
      {(Hq + 2 * Hkv) * D, H}, {H, Hq * D}, {2 * I, H}, {H, I}, {D}, {D},
      {np, Hkv, P, D}, {np, Hkv, D, P}};
  for (size_t i = 0; i < weights.size(); ++i) {
    const Tensor& w = weights[i];
    const size_t k = i % 8;
    if ((k == 4 || k == 5) && w.numel() == 0) continue;
    if (!plain(w, at::kBFloat16, hidden) || w.dim() != (long)sizes[k].size() ||
        !aligned16(w))
      return false;
    for (size_t d = 0; d < sizes[k].size(); ++d)
      if (w.size(d) != sizes[k][d]) return false;
  }
  return true;
}

// A decoded token of each sequence through a span of layers: hidden (M, 1, H). weights:
// eight tensors a layer: qkv, o, gate_up, down, q norm, k norm (both empty: none), k pages,
// v pages; the norms of the rows are folded into them. Columns of table are how far the
// sequences may reach. groups: workgroups, each a slot's; fewer take several. span_takes()
// has said yes.
static Tensor run_span(Tensor hidden, const std::vector<Tensor>& weights, long Hq,
                       const Tensor& cos_t, const Tensor& sin_t, const OptTensor& pos,
                       const Tensor& start, const Tensor& table, double eps, double scale,
                       long groups) {
  const int M = hidden.size(0), H = hidden.size(2), I = weights[3].size(1);
  const int Hkv = weights[6].size(1), P = weights[6].size(2);
  const int layers = (int)(weights.size() / 8);
  if (!aligned16(hidden)) hidden = hidden.clone();
  const Lds lds = lds_of(M, H, I, (int)Hq, Hkv);
  span::Args a;
  a.cos_t = cos_t.data_ptr<float>();
  a.sin_t = sin_t.data_ptr<float>();
  a.pos = pos ? pos->data_ptr<int>() : nullptr;
  a.start = start.data_ptr<int>();
  a.table = table.data_ptr<int>();
  a.M = M; a.H = H; a.I = I; a.Hq = (int)Hq; a.Hkv = Hkv;
  a.plog = P == 8 ? 3 : P == 16 ? 4 : 5;
  a.maxp = (int)table.stride(0);
  a.max_pos = (int)cos_t.size(0);
  a.parts = (int)std::min<long>(
      span::SLOTS / (M * Hkv),
      (table.size(1) * P + span::MIN_PART - 1) / span::MIN_PART);
  a.units = lds.units;
  a.lds_wide = lds.wide; a.lds_sums = lds.sums; a.lds_squares = lds.squares;
  a.lds_control = lds.control;
  a.inv_h = (float)(1.0 / H);
  a.eps = (float)eps; a.scale = (float)scale;
  const long each = span::fill_places(a.at, M, H, I, Hq, Hkv, a.parts);
  TORCH_CHECK(each < 1L << 30, "a span's exchange");
  for (int l0 = 0; l0 < layers; l0 += span::MAX_LAYERS) {
    a.layers = std::min(layers - l0, span::MAX_LAYERS);
    for (int l = 0; l < a.layers; ++l) {
      const Tensor* w = &weights[(l0 + l) * 8];
      auto ptr = [&](int i) {
        return (span::mem16)(w[i].numel() ? w[i].data_ptr() : nullptr);
      };
      a.layer[l] = {ptr(0), ptr(1), ptr(2), ptr(3), ptr(4), ptr(5), ptr(6), ptr(7)};
    }
    const long n = (span::SLOTS + a.layers * each + 3) / 4;
    auto work = torch::empty({n * 4}, start.options());
    auto out = torch::empty_like(hidden);
    a.hidden = static_cast<const bf16_bits*>(hidden.data_ptr());
    a.out = static_cast<bf16_bits*>(out.data_ptr());
    a.work = reinterpret_cast<unsigned*>(work.data_ptr<int>());
    span::decode_span_fill_kernel<<<(int)std::min<long>((n + 255) / 256, 1024), 256, 0,
                                    cur_stream()>>>(
        reinterpret_cast<uint4*>(a.work), n);
    check_launch();
    auto launch = [&](auto kernel) {
      allow_lds(kernel, lds.all);
      kernel<<<(int)groups, span::NT, lds.all, cur_stream()>>>(a);
    };
    if (small_model(H, I, (int)Hq, Hkv))
      launch(span::decode_span_kernel<span::SmallSizes>);
    else
      launch(span::decode_span_kernel<span::LargeSizes>);
    check_launch();
    hidden = out;
  }
  return hidden;
}

Tensor decode_span(Tensor hidden, std::vector<Tensor> weights, long Hq, Tensor cos_t,
                   Tensor sin_t, OptTensor pos, Tensor start, Tensor table, double eps,
                   double scale, long groups) {
  TORCH_CHECK(groups >= 1 && groups <= span::SLOTS, "workgroups of a span");
  TORCH_CHECK(span_takes(hidden, weights, Hq, cos_t, sin_t, pos, start, table),
              "decode_span: sizes, types or layouts that the kernel does not take");
  return run_span(hidden, weights, Hq, cos_t, sin_t, pos, start, table, eps, scale,
                  groups);
}

// None where decode_span would raise.
OptTensor decode_span_if(Tensor hidden, std::vector<Tensor> weights, long Hq, Tensor cos_t,
                         Tensor sin_t, OptTensor pos, Tensor start, Tensor table,
                         double eps, double scale) {
  if (!span_takes(hidden, weights, Hq, cos_t, sin_t, pos, start, table))
    return c10::nullopt;
  return run_span(hidden, weights, Hq, cos_t, sin_t, pos, start, table, eps, scale,
                  span::SLOTS);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("decode_span", &decode_span, py::arg("hidden"), py::arg("weights"), py::arg("Hq"),
        py::arg("cos_t"), py::arg("sin_t"), py::arg("pos"), py::arg("start"),
        py::arg("table"), py::arg("eps"), py::arg("scale"),
        py::arg("groups") = span::SLOTS);
  m.def("decode_span_if", &decode_span_if);
  m.def("span_fits", &span_fits);
}
