// torch operators over the C-ABI: a whole quantized linear (and a set of sibling linears) per call.
//
// svdq::linear and svdq::linear_siblings enqueue the activation pass and the GEMM back to back on the
// current stream, with every intermediate (operand codes, scales, low-rank activations, x_hat) in one
// workspace from the caching allocator.  As two Python operators with five allocations a layer call
// took 75 us on the host, three times a prompt-sized layer's GPU time; as one native operator 21 us
// (four sibling layers 172 -> 42 us).
// Registered with the dispatcher like any operator: tracing, vmap, dispatch modes and autograd meet
// them there (no gradient is defined).  The shape functions are registered from Python (ops.py).
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/library.h>

#include "../../include/svdq_gfx950.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

const char* status_name(int s) {
  switch (s) {
    case SVDQ_ERR_ARG: return "SVDQ_ERR_ARG";
    case SVDQ_ERR_SHAPE: return "SVDQ_ERR_SHAPE";
    case SVDQ_ERR_ALIGN: return "SVDQ_ERR_ALIGN";
    case SVDQ_ERR_UNSUPPORTED: return "SVDQ_ERR_UNSUPPORTED";
    case SVDQ_ERR_LAUNCH: return "SVDQ_ERR_LAUNCH";
  }
  return "SVDQ_ERR";
}
void check_status(const char* fn, int status) {
  TORCH_CHECK(status == SVDQ_OK, fn, " failed with ", status_name(status), ": ", svdq_last_error());
}

void check_tensor(const char* name, const Tensor& t, c10::Device dev, at::ScalarType dtype) {
  TORCH_CHECK_VALUE(t.device() == dev, name, " is on ", t.device(), ", expected ", dev);
  TORCH_CHECK_TYPE(t.scalar_type() == dtype, name, " must be ", dtype, ", got ", t.scalar_type());
  TORCH_CHECK_VALUE(t.is_contiguous(), name, " must be contiguous");
}

template <class T = void>
T* ptr(const Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}
template <class T = void>
T* ptr(const OptTensor& t) {
  return t.has_value() ? static_cast<T*>(t->data_ptr()) : nullptr;
}

// One layer's operands, checked, and where its intermediates go in the workspace.
struct Layer {
  const Tensor *srs, *l2, *w, *ws, *l1cat;
  OptTensor lora_down, lora_mult, bias;
  int64_t rtp, n, r, rl;
  int splits;
  int64_t qa, sx, xhat, mid;   // byte offsets, -1: not used
};

constexpr int64_t kNone = -1;   // operand: x_hat only, the W4A16 path
bool fast_group(int64_t g) { return g == 64 || g == 128; }

int64_t operand_bytes(int64_t rows, int64_t k, int64_t operand) {
  return operand == SVDQ_OPERAND_E3M2 ? ((rows + 1) & ~int64_t(1)) * k * 3 / 4 : rows * k;
}

struct Call {
  c10::Device dev;
  int64_t m, k, group, operand, bytes = 0;
  bool quant, want_xhat;
  std::vector<int64_t> lead;
  Tensor x;

  // x [..., K'] with K' <= K: flattened to contiguous rows, zero columns up to K
  Call(const Tensor& xin, int64_t k_, int64_t group_, int64_t operand_)
      : dev(xin.device()), k(k_), group(group_), operand(operand_) {
    TORCH_CHECK(xin.is_cuda(), "svdq::linear needs a GPU tensor");
    TORCH_CHECK_TYPE(xin.scalar_type() == at::kBFloat16, "x must be bfloat16, got ", xin.scalar_type());
    TORCH_CHECK_VALUE(xin.dim() >= 2, "expected [..., K] activation, got shape ", xin.sizes());
    TORCH_CHECK_VALUE(group > 0 && k > 0 && k % group == 0, "K=", k, " must be a multiple of group_size=", group);
    TORCH_CHECK_VALUE(operand == kNone || operand == SVDQ_OPERAND_E4M3 || operand == SVDQ_OPERAND_I8 ||
                          operand == SVDQ_OPERAND_E3M2,
                      "operand=", operand);
    const int64_t kx = xin.size(-1);
    TORCH_CHECK_VALUE(kx <= k, "activation K=", kx, " exceeds packed weight K=", k);
    lead = xin.sizes().vec();
    lead.pop_back();
    m = 1;
    for (int64_t d : lead) m *= d;
    TORCH_CHECK_VALUE(m <= INT32_MAX && k <= INT32_MAX, "M=", m, ", K=", k, " exceed 2^31 - 1");
    x = xin.reshape({m, kx}).contiguous();
    if (kx != k) x = at::constant_pad_nd(x, {0, k - kx}, 0);
    quant = operand != kNone;
    want_xhat = !quant || !fast_group(group);
  }

  int64_t take(int64_t n) {
    const int64_t at = bytes;
    bytes += (n + 255) / 256 * 256;
    return at;
  }

  Layer layer(const Tensor& srs, const Tensor& l2, OptTensor lora_down, OptTensor lora_mult, int64_t rtp,
              const Tensor& w, const Tensor& ws, const Tensor& l1cat, OptTensor bias) {
    Layer l{&srs, &l2, &w, &ws, &l1cat, std::move(lora_down), std::move(lora_mult), std::move(bias)};
    l.rtp = rtp;
    check_tensor("srs", srs, dev, at::kFloat);
    TORCH_CHECK_VALUE(srs.numel() == 2 * k, "srs has ", srs.numel(), " elements, expected ", 2 * k);
    check_tensor("l2", l2, dev, at::kBFloat16);
    TORCH_CHECK_VALUE(l2.dim() == 2 && l2.size(1) == k, "l2 must be [r, ", k, "], got ", l2.sizes());
    l.r = l2.size(0);
    l.rl = 0;
    if (l.lora_down.has_value()) {
      check_tensor("lora_down", *l.lora_down, dev, at::kBFloat16);
      TORCH_CHECK_VALUE(l.lora_down->dim() == 2 && l.lora_down->size(1) == k, "lora_down must be [rl, ", k, "], got ",
                        l.lora_down->sizes());
      l.rl = l.lora_down->size(0);
      TORCH_CHECK_VALUE(l.lora_mult.has_value() && l.lora_mult->numel() == l.rl, "lora_mult must have rl entries");
      check_tensor("lora_mult", *l.lora_mult, dev, at::kFloat);
    }
    check_tensor("weight", w, dev, at::kByte);
    check_tensor("weight scales", ws, dev, quant ? at::kInt : at::kHalf);
    TORCH_CHECK_VALUE(ws.dim() == 2 && ws.size(quant ? 0 : 1) == k / group, "weight scales do not match K=", k,
                      ", group_size=", group, ": ", ws.sizes());
    l.n = ws.size(quant ? 1 : 0);
    TORCH_CHECK_VALUE(l.n <= INT32_MAX, "N=", l.n, " exceeds 2^31 - 1");
    TORCH_CHECK_VALUE(w.numel() == (quant ? operand_bytes(l.n, k, operand) : l.n * k / 2), "weight holds ", w.numel(),
                      " bytes for N=", l.n, ", K=", k);
    check_tensor("l1cat", l1cat, dev, at::kBFloat16);
    TORCH_CHECK_VALUE(l1cat.dim() == 2 && l1cat.size(0) == l.n && l1cat.size(1) == rtp, "l1cat must be [", l.n, ", ",
                      rtp, "], got ", l1cat.sizes());
    if (l.bias.has_value()) {
      check_tensor("bias", *l.bias, dev, at::kBFloat16);
      TORCH_CHECK_VALUE(l.bias->numel() == l.n, "bias must have ", l.n, " entries");
    }
    int64_t mid_floats = 0;
    check_status("svdq_act_quant_workspace",
                 svdq_act_quant_workspace((int)m, (int)k, (int)group, (int)rtp, &l.splits, &mid_floats));
    l.qa = quant ? take(operand_bytes(m, k, operand)) : -1;
    l.sx = quant ? take(4 * m * (k / group)) : -1;
    l.xhat = want_xhat ? take(2 * m * k) : -1;
    l.mid = take(4 * mid_floats);
    return l;
  }

  unsigned flags(bool exact) const {
    return (operand == SVDQ_OPERAND_E4M3 ? SVDQ_ACT_OPERAND_E4M3 : 0u) |
           (operand == SVDQ_OPERAND_I8 ? SVDQ_ACT_OPERAND_I8 : 0u) |
           (operand == SVDQ_OPERAND_E3M2 ? SVDQ_ACT_OPERAND_E3M2 : 0u) | (want_xhat ? SVDQ_ACT_XHAT : 0u) |
           (exact ? SVDQ_ACT_EXACT_DIV : 0u) | (quant ? SVDQ_ACT_SX_PAIRS : 0u);
  }

  void act_quant(const Layer& l, uint8_t* base, bool exact, hipStream_t st) const {
    auto at = [&](int64_t off) -> void* { return off < 0 ? nullptr : base + off; };
    check_status("svdq_act_quant",
                 svdq_act_quant(ptr(x), k, ptr<float>(*l.srs), ptr(*l.l2), (int)l.r, ptr(l.lora_down), (int)l.rl,
                                ptr<float>(l.lora_mult), (int)m, (int)k, (int)group, (int)l.rtp, flags(exact),
                                at(l.qa), at(l.sx), nullptr, at(l.xhat), k, static_cast<float*>(at(l.mid)), l.splits,
                                st));
  }

  Tensor output(const Layer& l, bool out_f32) const {
    std::vector<int64_t> shape = lead;
    shape.push_back(l.n);
    return at::empty(shape, x.options().dtype(out_f32 ? at::kFloat : at::kBFloat16));
  }
};

Tensor linear(const Tensor& x, const Tensor& srs, const Tensor& l2, const OptTensor& lora_down,
              const OptTensor& lora_mult, int64_t group, int64_t rtp, const Tensor& weight, const Tensor& weight_scales,
              const Tensor& l1cat, const OptTensor& bias, int64_t operand, bool out_f32, bool exact, int64_t epi,
              const OptTensor& aux, const OptTensor& vec) {
  TORCH_CHECK_VALUE(srs.numel() % 2 == 0, "srs must hold 2 K values");
  Call c(x, srs.numel() / 2, group, operand);
  const c10::DeviceGuard guard(c.dev);
  const Layer l = c.layer(srs, l2, lora_down, lora_mult, rtp, weight, weight_scales, l1cat, bias);
  if (epi != SVDQ_EPI_NONE) {
    TORCH_CHECK_VALUE(!out_f32, "epilogue ops need bf16 output");
    TORCH_CHECK_VALUE(aux.has_value(), "epilogue op needs aux");
    check_tensor("aux", *aux, c.dev, at::kBFloat16);
    TORCH_CHECK_VALUE(aux->numel() == c.m * l.n, "aux must be [", c.m, ", ", l.n, "], got ", aux->sizes());
    TORCH_CHECK_VALUE(vec.has_value() == (epi == SVDQ_EPI_RESIDUAL_GATE), "vec is for residual_gate");
    if (vec.has_value()) {
      check_tensor("vec", *vec, c.dev, at::kBFloat16);
      TORCH_CHECK_VALUE(vec->numel() == l.n, "vec must have ", l.n, " entries");
    }
  } else {
    TORCH_CHECK_VALUE(!aux.has_value() && !vec.has_value(), "aux / vec given without an epilogue op");
  }
  Tensor y = c.output(l, out_f32);
  const Tensor work = at::empty({c.bytes}, c.x.options().dtype(at::kByte));
  uint8_t* base = ptr<uint8_t>(work);
  const hipStream_t st = c10::hip::getCurrentHIPStream(c.dev.index());
  c.act_quant(l, base, exact, st);
  const int m = (int)c.m, n = (int)l.n, k = (int)c.k, rt = (int)rtp, f32 = out_f32;
  if (c.quant)
    check_status("svdq_w4a4_gemm_epi",
                 svdq_w4a4_gemm_epi(base + l.qa, (int)operand, base + l.sx, ptr(weight), ptr(weight_scales),
                                    base + l.mid, ptr(l1cat), rt, ptr(bias), m, n, k, (int)group, ptr(y), n, f32,
                                    (int)epi, ptr(aux), n, ptr(vec), st));
  else
    check_status("svdq_w4a16_gemm_epi",
                 svdq_w4a16_gemm_epi(base + l.xhat, k, ptr(weight), ptr(weight_scales), base + l.mid, ptr(l1cat), rt,
                                     ptr(bias), m, n, k, (int)group, ptr(y), n, f32, (int)epi, ptr(aux), n, ptr(vec),
                                     st));
  return y;
}

std::vector<Tensor> linear_siblings(const Tensor& x, const std::vector<Tensor>& srs, const std::vector<Tensor>& l2,
                                    const c10::List<OptTensor>& lora_down, const c10::List<OptTensor>& lora_mult,
                                    int64_t group, c10::IntArrayRef rtp, const std::vector<Tensor>& weight,
                                    const std::vector<Tensor>& weight_scales, const std::vector<Tensor>& l1cat,
                                    const c10::List<OptTensor>& bias, int64_t operand, bool out_f32, bool exact) {
  const size_t count = srs.size();
  TORCH_CHECK_VALUE(count >= 1 && count <= SVDQ_MAX_SIBLINGS, "1..", SVDQ_MAX_SIBLINGS, " sibling layers, got ", count);
  TORCH_CHECK_VALUE(l2.size() == count && lora_down.size() == count && lora_mult.size() == count &&
                        rtp.size() == count && weight.size() == count && weight_scales.size() == count &&
                        l1cat.size() == count && bias.size() == count,
                    "one entry per layer in every list");
  TORCH_CHECK_VALUE(srs[0].numel() % 2 == 0, "srs must hold 2 K values");
  Call c(x, srs[0].numel() / 2, group, operand);
  TORCH_CHECK_VALUE(fast_group(group), "sibling launch needs group size 64 or 128, got ", group);
  const c10::DeviceGuard guard(c.dev);
  Layer l[SVDQ_MAX_SIBLINGS];
  std::vector<Tensor> ys;
  bool one_pass = operand == SVDQ_OPERAND_E3M2 || !c.quant;   // one launch for the activation passes
  for (size_t i = 0; i < count; ++i) {
    l[i] = c.layer(srs[i], l2[i], lora_down.get(i), lora_mult.get(i), rtp[i], weight[i], weight_scales[i], l1cat[i],
                   bias.get(i));
    ys.push_back(c.output(l[i], out_f32));
    one_pass = one_pass && !l[i].rl && rtp[i] == rtp[0];
  }
  const Tensor work = at::empty({c.bytes}, c.x.options().dtype(at::kByte));
  uint8_t* base = ptr<uint8_t>(work);
  const hipStream_t st = c10::hip::getCurrentHIPStream(c.dev.index());
  const int m = (int)c.m, k = (int)c.k, f32 = out_f32;
  if (one_pass) {
    svdq_act_sibling a[SVDQ_MAX_SIBLINGS];
    for (size_t i = 0; i < count; ++i)
      a[i] = {ptr<float>(srs[i]), ptr(l2[i]), (int)l[i].r, base + (c.quant ? l[i].qa : l[i].xhat),
              c.quant ? base + l[i].sx : nullptr, reinterpret_cast<float*>(base + l[i].mid)};
    if (c.quant)
      check_status("svdq_act_quant_siblings", svdq_act_quant_siblings(ptr(c.x), k, a, (int)count, m, k, (int)group,
                                                                      (int)rtp[0], c.flags(exact), l[0].splits, st));
    else
      check_status("svdq_act_xhat_siblings", svdq_act_xhat_siblings(ptr(c.x), k, a, (int)count, m, k, (int)group,
                                                                    (int)rtp[0], exact, l[0].splits, st));
  } else {
    for (size_t i = 0; i < count; ++i) c.act_quant(l[i], base, exact, st);
  }
  if (c.quant) {
    svdq_w4a4_sibling g[SVDQ_MAX_SIBLINGS];
    for (size_t i = 0; i < count; ++i)
      g[i] = {base + l[i].qa, base + l[i].sx, ptr(weight[i]), ptr(weight_scales[i]), base + l[i].mid, ptr(l1cat[i]),
              (int)rtp[i], ptr(l[i].bias), (int)l[i].n, ptr(ys[i]), l[i].n};
    check_status("svdq_w4a4_gemm_siblings",
                 svdq_w4a4_gemm_siblings(g, (int)count, (int)operand, m, k, (int)group, f32, st));
  } else {
    svdq_w4a16_sibling g[SVDQ_MAX_SIBLINGS];
    for (size_t i = 0; i < count; ++i)
      g[i] = {base + l[i].xhat, k, ptr(weight[i]), ptr(weight_scales[i]), base + l[i].mid, ptr(l1cat[i]), (int)rtp[i],
              ptr(l[i].bias), (int)l[i].n, ptr(ys[i]), l[i].n};
    check_status("svdq_w4a16_gemm_siblings", svdq_w4a16_gemm_siblings(g, (int)count, m, k, (int)group, f32, st));
  }
  return ys;
}

}  // namespace

// The torch that this file was compiled against, found in the file by kernels/hip/lib.py ahead of
// loading it: the C++ interfaces used here hold for that build of torch only.
extern "C" __attribute__((used, visibility("default"))) const char svdq_torch_build[] = "svdq_torch built with torch " SVDQ_TORCH_BUILD;

TORCH_LIBRARY_FRAGMENT(svdq, m) {
  m.def(
      "linear(Tensor x, Tensor srs, Tensor l2, Tensor? lora_down, Tensor? lora_mult, int group_size, int rtp, "
      "Tensor weight, Tensor weight_scales, Tensor l1cat, Tensor? bias, int operand, bool out_f32, bool exact, "
      "int epi=0, Tensor? aux=None, Tensor? vec=None) -> Tensor");
  m.def(
      "linear_siblings(Tensor x, Tensor[] srs, Tensor[] l2, Tensor?[] lora_down, Tensor?[] lora_mult, "
      "int group_size, int[] rtp, Tensor[] weight, Tensor[] weight_scales, Tensor[] l1cat, Tensor?[] bias, "
      "int operand, bool out_f32, bool exact) -> Tensor[]");
}
TORCH_LIBRARY_IMPL(svdq, CUDA, m) {
  m.impl("linear", TORCH_FN(linear));
  m.impl("linear_siblings", TORCH_FN(linear_siblings));
}
TORCH_LIBRARY_IMPL(svdq, Autograd, m) {
  m.impl("linear", torch::autograd::autogradNotImplementedFallback());
  m.impl("linear_siblings", torch::autograd::autogradNotImplementedFallback());
}
