// The jit_thc operators on GPU tensors: argument checks, output allocation and the launch through include/lthc.h for
// the CUDA dispatch key, and the autograd formulas of every device.  The schemas and the fake (meta) kernels are
// registered from Python (ops.py, ops_branch.py, ops_triangular.py), which also refuse tensors of other devices; the
// reference's formulas each node follows are cited there.
//
// Why native: one interface step is 2L + 4 of these calls on kernels of a few microseconds, and a call through a
// Python kernel costs 12-16 us of host time (25-60 us where autograd records it, as much again in the backward) against
// 5-6 us here, so below about B = 8 the host set the pace.  B = 1 interface forward (16 calls) 253 -> 98 us; a 6-layer
// fp32 interface training step at B = 5 0.96-1.1 -> 0.41 ms.

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <array>
#include <cmath>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/lthc.h"

namespace {

using at::Tensor;
using at::TensorList;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int64_t S = 4;       // cell side
constexpr int64_t K = S * S;   // taps
constexpr int64_t kQkHeadDim = 64;
constexpr int64_t kAttnMaxTokens = 256;
constexpr int64_t kNormMaxChannels = 2048;
constexpr int64_t kMaxWsDepth = 24;

// ---------------------------------------------------------------------------
// checks and operands
// ---------------------------------------------------------------------------
std::string shape(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

bool has_shape(const Tensor& t, at::IntArrayRef want) { return t.sizes() == want; }

int code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return LTHC_F32;
    case at::kBFloat16: return LTHC_BF16;
    case at::kHalf: return LTHC_F16;
    default: break;
  }
  TORCH_CHECK_VALUE(false, "unsupported dtype ", t.scalar_type(), "; expected float32, bfloat16 or float16");
}

bool known_dtype(const Tensor& t) {
  return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf;
}

void same_device(const Tensor& first, const Tensor& t) {
  TORCH_CHECK_VALUE(t.device() == first.device(), "all tensors must be on ", first.device(), ", got one on ", t.device());
}

void on_gpu(const Tensor& t) {
  TORCH_CHECK_VALUE(t.is_cuda(), "LTHC HIP ops need GPU tensors, got a ", t.device(),
                    " tensor (there is no CPU fallback)");
}

template <typename... Ts>
void on_gpu(const Tensor& first, const Ts&... rest) {
  on_gpu(first);
  (same_device(first, rest), ...);
}

void on_gpu_list(const Tensor& first, TensorList list) {
  for (const Tensor& t : list) same_device(first, t);
}

bool aligned(const Tensor& t, uintptr_t bytes) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0; }

// Contiguous and aligned to 4 elements, as the C ABI requires.
Tensor prep(const Tensor& t) {
  Tensor c = t.contiguous();
  return aligned(c, 4 * c.element_size()) ? c : c.clone();
}

Tensor prep_as(const Tensor& t, at::ScalarType dtype) {
  Tensor c = prep(t);
  return c.scalar_type() == dtype ? c : c.to(dtype);
}

// Contiguous with a 16-byte aligned start.
Tensor prep16(const Tensor& t) {
  Tensor c = t.contiguous();
  return aligned(c, 16) ? c : c.clone();
}

// Cell weights in fp32 or the activation dtype (the compiled pairs), 16-byte aligned.
Tensor prep_w(const Tensor& w, at::ScalarType act) {
  return prep16(w.scalar_type() == at::kFloat || w.scalar_type() == act ? w : w.to(at::kFloat));
}

std::vector<Tensor> prep_ws(TensorList ws, at::ScalarType act) {
  std::vector<Tensor> out;
  out.reserve(ws.size());
  bool mixed = false;
  for (const Tensor& w : ws) {
    out.push_back(prep_w(w, act));
    mixed |= out.back().scalar_type() != out.front().scalar_type();
  }
  if (mixed)
    for (Tensor& w : out) w = prep_w(w.to(at::kFloat), act);
  return out;
}

std::vector<Tensor> prep_all(TensorList ts, at::ScalarType dtype) {
  std::vector<Tensor> out;
  out.reserve(ts.size());
  for (const Tensor& t : ts) out.push_back(prep_as(t, dtype));
  return out;
}

struct Geom {
  int64_t b, g, c;
};

Geom hi_geom(const Tensor& x, const char* name) {
  TORCH_CHECK_VALUE(x.dim() == 4 && x.size(1) == x.size(2), name, " must be NHWC [B,H,H,C], got ", shape(x));
  TORCH_CHECK_VALUE(x.size(1) % S == 0, name, ": high-res side ", x.size(1), " is not a multiple of the cell side ", S);
  TORCH_CHECK_VALUE(x.size(3) % 4 == 0, name, ": channels ", x.size(3), " must be a multiple of 4");
  return {x.size(0), x.size(1) / S, x.size(3)};
}

Geom lo_geom(const Tensor& z, const char* name) {
  TORCH_CHECK_VALUE(z.dim() == 3, name, " must be [B,M,C], got ", shape(z));
  const int64_t m = z.size(1);
  int64_t g = static_cast<int64_t>(std::llround(std::sqrt(static_cast<double>(m))));
  TORCH_CHECK_VALUE(g * g == m, name, ": workspace token count ", m, " is not a square");
  TORCH_CHECK_VALUE(z.size(2) % 4 == 0, name, ": channels ", z.size(2), " must be a multiple of 4");
  return {z.size(0), g, z.size(2)};
}

void check_weight(const Tensor& w, int64_t c, const std::string& name) {
  TORCH_CHECK_VALUE(has_shape(w, {c, K}), name, " must be [", c, ",", K, "], got ", shape(w));
  code(w);
}

void check_like(const Tensor& t, at::IntArrayRef want, const std::string& name) {
  TORCH_CHECK_VALUE(has_shape(t, want), name, " must be ", want, ", got ", shape(t));
}

template <typename T = const void>
std::vector<T*> pointers(TensorList ts) {
  std::vector<T*> p;
  p.reserve(ts.size());
  for (const Tensor& t : ts) p.push_back(t.data_ptr());
  return p;
}

void* data(const Tensor& t) { return t.data_ptr(); }

// The launch's device and stream: torch's current stream on t's device.
struct Launch {
  c10::DeviceGuard guard;
  void* stream;
  explicit Launch(const Tensor& t) : guard(t.device()), stream(c10::hip::getCurrentHIPStream(t.get_device()).stream()) {}
};

void check(int rc, const char* what) {
  if (rc == LTHC_OK) return;
  const char* msg = lthc_last_error();
  if (msg == nullptr || *msg == 0) msg = what;
  TORCH_CHECK_VALUE(rc != LTHC_ERR_INVALID && rc != LTHC_ERR_UNSUPPORTED, msg);
  TORCH_CHECK(false, msg);
}

Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({static_cast<int64_t>(std::max<size_t>(bytes, 16))}, like.options().dtype(at::kByte));
}

Tensor fp32_like(at::IntArrayRef sizes, const Tensor& like) { return at::empty(sizes, like.options().dtype(at::kFloat)); }

void check_depth(size_t dzs, size_t betas) {
  TORCH_CHECK_VALUE(dzs == betas && dzs >= 1 && dzs <= LTHC_MAX_LAYERS, "expected 1..", LTHC_MAX_LAYERS,
                    " dz and as many beta tensors, got ", dzs, " and ", betas);
}

void check_layers(const Geom& g, TensorList dzs, TensorList betas, const char* dz, const char* beta, const char* end) {
  for (size_t i = 0; i < dzs.size(); ++i)
    check_like(dzs[i], {g.b, g.g * g.g, g.c}, dz + std::to_string(i) + end);
  for (size_t i = 0; i < betas.size(); ++i) check_weight(betas[i], g.c, beta + std::to_string(i) + end);
}

// ---------------------------------------------------------------------------
// the interface
// ---------------------------------------------------------------------------
Tensor read_cuda(const Tensor& x_, const Tensor& weight) {
  on_gpu(x_, weight);
  const Geom g = hi_geom(x_, "x");
  check_weight(weight, g.c, "weight");
  const Tensor x = prep(x_), w = prep_w(weight, x.scalar_type());
  Tensor z = at::empty({g.b, g.g * g.g, g.c}, x.options());
  const Launch l(x);
  check(lthc_read_fwd(data(x), code(x), data(w), code(w), data(z), g.b, g.g, S, g.c, l.stream), "lthc_read_fwd");
  return z;
}

// out = base (may be undefined) + sum_l beta_l dz_l; operands prepared.
void materialise(const Tensor& base, TensorList dzs, TensorList betas, const Tensor& out) {
  const Geom g = lo_geom(dzs[0], "dz");
  const auto dp = pointers(dzs), bp = pointers(betas);
  const Launch l(out);
  check(lthc_materialise_fwd(base.defined() ? data(base) : nullptr, dp.data(), code(out), bp.data(), code(betas[0]),
                             data(out), g.b, g.g, S, g.c, static_cast<int>(dzs.size()), l.stream),
        "lthc_materialise_fwd");
}

Tensor write_cuda(const Tensor& z_, const Tensor& weight) {
  on_gpu(z_, weight);
  const Geom g = lo_geom(z_, "z");
  check_weight(weight, g.c, "weight");
  const Tensor z = prep(z_), w = prep_w(weight, z.scalar_type());
  Tensor out = at::empty({g.b, g.g * S, g.g * S, g.c}, z.options());
  materialise(Tensor(), {z}, {w}, out);
  return out;
}

Tensor write_add_cuda(const Tensor& z_, const Tensor& weight, const Tensor& x_) {
  on_gpu(z_, weight, x_);
  const Geom g = lo_geom(z_, "z"), h = hi_geom(x_, "x");
  TORCH_CHECK_VALUE(h.b == g.b && h.g == g.g && h.c == g.c, "z ", shape(z_), " and x ", shape(x_),
                    " do not describe the same cells");
  check_weight(weight, g.c, "weight");
  const Tensor x = prep(x_), z = prep_as(z_, x.scalar_type()), w = prep_w(weight, x.scalar_type());
  Tensor out = at::empty_like(x);
  materialise(x, {z}, {w}, out);
  return out;
}

Tensor materialise_checked(const Tensor& x0_, TensorList dzs, TensorList betas) {
  const Tensor x0 = prep(x0_);
  Tensor out = at::empty_like(x0);
  materialise(x0, prep_all(dzs, x0.scalar_type()), prep_ws(betas, x0.scalar_type()), out);
  return out;
}

Tensor final_list_cuda(const Tensor& x0, TensorList dzs, TensorList betas) {
  on_gpu(x0);
  on_gpu_list(x0, dzs);
  on_gpu_list(x0, betas);
  const Geom g = hi_geom(x0, "x0");
  check_depth(dzs.size(), betas.size());
  check_layers(g, dzs, betas, "dz[", "beta[", "]");
  return materialise_checked(x0, dzs, betas);
}

#define LTHC_T12(p)                                                                                               \
  const Tensor &p##0, const Tensor &p##1, const Tensor &p##2, const Tensor &p##3, const Tensor &p##4,             \
      const Tensor &p##5, const Tensor &p##6, const Tensor &p##7, const Tensor &p##8, const Tensor &p##9,         \
      const Tensor &p##10, const Tensor &p##11
#define LTHC_TYPES12                                                                                              \
  const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,        \
      const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&
#define LTHC_A12(p) p##0, p##1, p##2, p##3, p##4, p##5, p##6, p##7, p##8, p##9, p##10, p##11

Tensor final_12_cuda(const Tensor& x0, LTHC_T12(dz), LTHC_T12(beta)) {
  const std::array<Tensor, 12> dzs{LTHC_A12(dz)}, betas{LTHC_A12(beta)};
  on_gpu(x0);
  on_gpu_list(x0, dzs);
  on_gpu_list(x0, betas);
  check_layers(hi_geom(x0, "x0"), dzs, betas, "dz", "beta", "");
  return materialise_checked(x0, dzs, betas);
}

// gW[l] = sum high * low_l, fp32 [L, C, 16]; operands prepared.
Tensor weight_grad(const Tensor& high, TensorList lows) {
  const Geom g = hi_geom(high, "high");
  const int L = static_cast<int>(lows.size());
  Tensor out = fp32_like({L, g.c, K}, high);
  const Tensor ws = workspace(lthc_weight_grad_workspace_bytes(g.b, g.g, S, g.c, L), high);
  const auto lp = pointers(lows);
  const Launch l(high);
  check(lthc_weight_grad(data(high), lp.data(), code(high), static_cast<float*>(data(out)), g.b, g.g, S, g.c, L,
                         data(ws), ws.numel(), l.stream),
        "lthc_weight_grad");
  return out;
}

Tensor weight_grad_cuda(const Tensor& high_, const Tensor& low) {
  on_gpu(high_, low);
  const Geom g = hi_geom(high_, "high"), h = lo_geom(low, "low");
  TORCH_CHECK_VALUE(h.b == g.b && h.g == g.g && h.c == g.c, "high ", shape(high_), " and low ", shape(low),
                    " do not match");
  const Tensor high = prep(high_);
  return weight_grad(high, {prep_as(low, high.scalar_type())}).select(0, 0);
}

std::tuple<Tensor, Tensor> final_backward_cuda(const Tensor& grad_out, TensorList dzs_, TensorList betas_) {
  on_gpu(grad_out);
  on_gpu_list(grad_out, dzs_);
  on_gpu_list(grad_out, betas_);
  const Geom g = hi_geom(grad_out, "grad_out");
  check_depth(dzs_.size(), betas_.size());
  check_layers(g, dzs_, betas_, "dz[", "beta[", "]");
  const Tensor gr = prep(grad_out);
  const auto dzs = prep_all(dzs_, gr.scalar_type()), betas = prep_ws(betas_, gr.scalar_type());
  const int L = static_cast<int>(dzs.size());
  Tensor gdz = at::empty({L, g.b, g.g * g.g, g.c}, gr.options());
  Tensor gb = fp32_like({L, g.c, K}, gr);
  const Tensor ws = workspace(lthc_materialise_bwd_workspace_bytes(g.b, g.g, S, g.c, L), gr);
  const auto dp = pointers(dzs), bp = pointers(betas);
  std::vector<void*> op;
  const int64_t step = g.b * g.g * g.g * g.c * gr.element_size();
  for (int i = 0; i < L; ++i) op.push_back(static_cast<char*>(data(gdz)) + i * step);
  const Launch l(gr);
  check(lthc_materialise_bwd(data(gr), code(gr), dp.data(), bp.data(), code(betas[0]), op.data(),
                             static_cast<float*>(data(gb)), g.b, g.g, S, g.c, L, data(ws), ws.numel(), l.stream),
        "lthc_materialise_bwd");
  return {gdz, gb};
}

int64_t check_recur(const Tensor& z, const Tensor& dz, const Tensor& gamma) {
  TORCH_CHECK_VALUE(z.sizes() == dz.sizes() && z.dim() >= 1, "z ", shape(z), " and dz ", shape(dz),
                    " must have the same shape");
  const int64_t c = z.size(-1);
  TORCH_CHECK_VALUE(has_shape(gamma, {c}), "gamma must be [", c, "], got ", shape(gamma));
  TORCH_CHECK_VALUE(c % 4 == 0, "channels ", c, " must be a multiple of 4");
  code(gamma);
  return c;
}

Tensor recur_cuda(const Tensor& z_, const Tensor& dz_, const Tensor& gamma_) {
  on_gpu(z_, dz_, gamma_);
  const int64_t c = check_recur(z_, dz_, gamma_);
  const auto dt = at::promote_types(z_.scalar_type(), dz_.scalar_type());
  const Tensor z = prep(z_.to(dt)), dz = prep(dz_.to(dt)), gamma = prep(gamma_);
  Tensor out = at::empty_like(z);
  const Launch l(z);
  check(lthc_recur_fwd(data(z), data(dz), code(z), data(gamma), code(gamma), data(out), c ? z.numel() / c : 0, c, l.stream),
        "lthc_recur_fwd");
  return out;
}

std::optional<Tensor> prep_add(const std::optional<Tensor>& add, const Tensor& grad) {
  if (!add.has_value() || !add->defined()) return std::nullopt;
  TORCH_CHECK_VALUE(add->sizes() == grad.sizes(), "gdz_add ", shape(*add), " must match grad ", shape(grad));
  return prep_as(*add, grad.scalar_type());
}

std::tuple<Tensor, Tensor> recur_backward_cuda(const Tensor& grad_, const Tensor& dz_, const Tensor& gamma_,
                                               const std::optional<Tensor>& gdz_add) {
  on_gpu(grad_, dz_, gamma_);
  const int64_t c = check_recur(grad_, dz_, gamma_);
  const Tensor grad = prep(grad_), dz = prep_as(dz_, grad.scalar_type()), gamma = prep(gamma_);
  const auto add = prep_add(gdz_add, grad);
  const int64_t rows = c ? grad.numel() / c : 0;
  Tensor gdz = at::empty_like(grad), gg = fp32_like({c}, grad);
  const Tensor ws = workspace(lthc_recur_bwd_workspace_bytes(rows, c), grad);
  const Launch l(grad);
  check(lthc_recur_bwd(data(grad), data(dz), add ? data(*add) : nullptr, code(grad), data(gamma), code(gamma), data(gdz),
                       static_cast<float*>(data(gg)), rows, c, data(ws), ws.numel(), l.stream),
        "lthc_recur_bwd");
  return {gdz, gg};
}

std::tuple<Tensor, Tensor, Tensor> recur_backward_sum_cuda(const Tensor& grad_, const Tensor& branch_, const Tensor& dz_,
                                                           const Tensor& gamma_, const std::optional<Tensor>& gdz_add) {
  on_gpu(grad_, branch_, dz_, gamma_);
  const int64_t c = check_recur(grad_, dz_, gamma_);
  TORCH_CHECK_VALUE(branch_.sizes() == grad_.sizes(), "grad_branch ", shape(branch_), " must match grad ", shape(grad_));
  const Tensor grad = prep(grad_), dz = prep_as(dz_, grad.scalar_type()), gamma = prep(gamma_);
  const Tensor branch = prep_as(branch_, grad.scalar_type());
  const auto add = prep_add(gdz_add, grad);
  const int64_t rows = c ? grad.numel() / c : 0;
  Tensor gsum = at::empty_like(grad), gdz = at::empty_like(grad), gg = at::empty({c}, gamma.options());
  const Tensor ws = workspace(lthc_recur_bwd_workspace_bytes(rows, c), grad);
  const Launch l(grad);
  check(lthc_recur_bwd_sum(data(grad), data(branch), data(dz), add ? data(*add) : nullptr, code(grad), data(gamma),
                           code(gamma), data(gsum), data(gdz), data(gg), code(gg), rows, c, data(ws), ws.numel(),
                           l.stream),
        "lthc_recur_bwd_sum");
  return {gsum, gdz, gg};
}

Tensor gamma_stack_cuda(const Tensor& alpha_, const Tensor& stack_) {
  on_gpu(alpha_, stack_);
  TORCH_CHECK_VALUE(alpha_.dim() == 2 && stack_.dim() == 3 && stack_.size(1) == alpha_.size(0) &&
                        stack_.size(2) == alpha_.size(1),
                    "alpha [C,K] and beta_stack [L,C,K] expected, got ", shape(alpha_), ", ", shape(stack_));
  const int64_t L = stack_.size(0), c = alpha_.size(0), k = alpha_.size(1);
  TORCH_CHECK_VALUE(L >= 1 && L <= LTHC_MAX_LAYERS, "depth ", L, " outside 1..", LTHC_MAX_LAYERS);
  const Tensor alpha = alpha_.contiguous(), stack = stack_.to(alpha.scalar_type()).contiguous();
  Tensor out = fp32_like({L, c}, alpha);
  std::vector<const void*> bp;
  for (int64_t i = 0; i < L; ++i) bp.push_back(static_cast<const char*>(data(stack)) + i * c * k * stack.element_size());
  const Launch l(alpha);
  check(lthc_gamma(data(alpha), bp.data(), code(alpha), data(out), LTHC_F32, c, k, static_cast<int>(L), l.stream),
        "lthc_gamma");
  return out;
}

std::vector<Tensor> one_dtype(TensorList ts) {
  std::vector<Tensor> out;
  for (const Tensor& t : ts) out.push_back(t.to(ts[0].scalar_type()).contiguous());
  return out;
}

void check_gamma_rounded(const Tensor& alpha, TensorList betas) {
  bool same = alpha.dim() == 2 && !betas.empty();
  for (const Tensor& b : betas) same &= b.sizes() == alpha.sizes();
  TORCH_CHECK_VALUE(same, "alpha [C,K] and L betas of the same shape expected, got ", shape(alpha));
  TORCH_CHECK_VALUE(betas.size() <= LTHC_MAX_LAYERS, "depth ", betas.size(), " outside 1..", LTHC_MAX_LAYERS);
}

Tensor gamma_rounded_cuda(const Tensor& alpha_, TensorList betas_, at::ScalarType dtype) {
  on_gpu(alpha_);
  on_gpu_list(alpha_, betas_);
  check_gamma_rounded(alpha_, betas_);
  const auto betas = one_dtype(betas_);
  const Tensor alpha = alpha_.contiguous();
  const int64_t c = alpha.size(0), k = alpha.size(1);
  Tensor out = at::empty({static_cast<int64_t>(betas.size()), c}, alpha.options().dtype(dtype));
  const auto bp = pointers(betas);
  const Launch l(alpha);
  check(lthc_gamma_rounded(data(alpha), code(alpha), bp.data(), code(betas[0]), data(out), code(out), c, k,
                           static_cast<int>(betas.size()), l.stream),
        "lthc_gamma_rounded");
  return out;
}

std::tuple<Tensor, std::vector<Tensor>> gamma_rounded_backward_cuda(const Tensor& grad_, const Tensor& alpha_,
                                                                    TensorList betas_, bool need_alpha,
                                                                    bool need_beta) {
  on_gpu(grad_, alpha_);
  on_gpu_list(grad_, betas_);
  check_gamma_rounded(alpha_, betas_);
  check_like(grad_, {static_cast<int64_t>(betas_.size()), alpha_.size(0)}, "grad");
  const auto betas = one_dtype(betas_);
  const Tensor alpha = alpha_.contiguous(), grad = grad_.contiguous();
  Tensor ga = need_alpha ? at::empty_like(alpha) : at::empty({0}, alpha.options());
  std::vector<Tensor> gbs;
  if (need_beta)
    for (const Tensor& b : betas) gbs.push_back(at::empty_like(b));
  const auto bp = pointers(betas);
  const auto gp = pointers<void>(gbs);
  const Launch l(alpha);
  check(lthc_gamma_rounded_bwd(data(grad), data(alpha), code(alpha), bp.data(), code(betas[0]),
                               need_alpha ? data(ga) : nullptr, need_beta ? gp.data() : nullptr, code(grad),
                               alpha.size(0), alpha.size(1), static_cast<int>(betas.size()), l.stream),
        "lthc_gamma_rounded_bwd");
  return {ga, gbs};
}

// ---------------------------------------------------------------------------
// the non-shared interface
// ---------------------------------------------------------------------------
void check_alpha_stack(const Geom& g, const Tensor& a) {
  TORCH_CHECK_VALUE(a.dim() == 3 && a.size(1) == g.c && a.size(2) == K && a.size(0) >= 1 && a.size(0) <= kMaxWsDepth,
                    "alpha_stack must be [L,", g.c, ",", K, "] with 1 <= L <= ", kMaxWsDepth, ", got ", shape(a));
}

std::vector<Tensor> all_base_split_cuda(const Tensor& x0_, const Tensor& alpha_stack) {
  on_gpu(x0_, alpha_stack);
  const Geom g = hi_geom(x0_, "x0");
  check_alpha_stack(g, alpha_stack);
  const Tensor x0 = prep(x0_);
  const auto alphas = prep_w(alpha_stack, x0.scalar_type()).unbind(0);
  std::vector<Tensor> outs;
  for (size_t i = 0; i < alphas.size(); ++i) outs.push_back(at::empty({g.b, g.g * g.g, g.c}, x0.options()));
  const auto ap = pointers(alphas);
  const auto op = pointers<void>(outs);
  const Launch l(x0);
  check(lthc_read_multi_fwd(data(x0), code(x0), ap.data(), code(alphas[0]), op.data(), g.b, g.g, S, g.c,
                            static_cast<int>(alphas.size()), l.stream),
        "lthc_read_multi_fwd");
  return outs;
}

// Gradients of the bases R_l(x0) for x0 (sum_l R_l^T g_l) and the [L, C, 16] read weights (fp32), the g_l as separate
// tensors; an empty tensor for a gradient that is not wanted.
std::tuple<Tensor, Tensor> all_base_backward_cuda(const Tensor& x0_, TensorList grads_, const Tensor& alpha_stack,
                                                  bool need_x, bool need_alpha) {
  on_gpu(x0_, alpha_stack);
  on_gpu_list(x0_, grads_);
  const Geom g = hi_geom(x0_, "x0");
  check_alpha_stack(g, alpha_stack);
  TORCH_CHECK_VALUE(static_cast<int64_t>(grads_.size()) == alpha_stack.size(0), "expected ", alpha_stack.size(0),
                    " gradients, got ", grads_.size());
  for (size_t i = 0; i < grads_.size(); ++i)
    check_like(grads_[i], {g.b, g.g * g.g, g.c}, "grads[" + std::to_string(i) + "]");
  const Tensor x0 = prep(x0_);
  const auto grads = prep_all(grads_, x0.scalar_type());
  Tensor gx = at::empty({0}, x0.options()), ga = fp32_like({0}, x0);
  if (need_x) {
    gx = at::empty_like(x0);
    materialise(Tensor(), grads, prep_w(alpha_stack, x0.scalar_type()).unbind(0), gx);
  }
  if (need_alpha) ga = weight_grad(x0, grads);
  return {gx, ga};
}

Tensor ws_forward(const Tensor& base_, TensorList dzs_, const Tensor& gamma_) {
  on_gpu(base_, gamma_);
  on_gpu_list(base_, dzs_);
  TORCH_CHECK_VALUE(base_.dim() == 3, "base must be [B,M,C], got ", shape(base_));
  const int64_t c = base_.size(2), L = static_cast<int64_t>(dzs_.size());
  TORCH_CHECK_VALUE(L >= 1 && L <= kMaxWsDepth, "depth ", L, " outside 1..", kMaxWsDepth);
  for (int64_t i = 0; i < L; ++i)
    TORCH_CHECK_VALUE(dzs_[i].sizes() == base_.sizes(), "dz", i, " shape ", shape(dzs_[i]), " does not match base ",
                      shape(base_));
  TORCH_CHECK_VALUE(gamma_.dim() == 2 && gamma_.size(0) >= L && gamma_.size(1) == c, "gamma must be [>= ", L, ", ", c,
                    "], got ", shape(gamma_));
  TORCH_CHECK_VALUE(c % 4 == 0, "channels ", c, " must be a multiple of 4");
  code(gamma_);
  const Tensor base = prep(base_), gamma = gamma_.contiguous();
  const auto dzs = prep_all(dzs_, base.scalar_type());
  Tensor out = at::empty_like(base);
  const auto dp = pointers(dzs);
  const Launch l(base);
  check(lthc_ws_accumulate_fwd(data(base), dp.data(), code(base), data(gamma), code(gamma), data(out),
                               c ? base.numel() / c : 0, c, static_cast<int>(L), l.stream),
        "lthc_ws_accumulate_fwd");
  return out;
}

Tensor tri_list_cuda(const Tensor& base, TensorList dzs, const Tensor& gamma) { return ws_forward(base, dzs, gamma); }

Tensor tri12_forward(const Tensor& base, TensorList dzs, const Tensor& gamma, int64_t active) {
  TORCH_CHECK_VALUE(base.dim() == 3 && gamma.dim() == 2 && gamma.size(0) == 12 && gamma.size(1) == base.size(2),
                    "triangular_accumulate_b4_12 expects base [B,M,C] and gamma [12,C], got ", shape(base), " and ",
                    shape(gamma));
  for (size_t i = 0; i < dzs.size(); ++i)
    TORCH_CHECK_VALUE(dzs[i].sizes() == base.sizes(), "triangular_accumulate_b4_12 dz", i, " shape ", shape(dzs[i]),
                      " does not match base ", shape(base));
  return ws_forward(base, dzs.slice(0, active), gamma);
}

int64_t check_active(int64_t active) {
  TORCH_CHECK_VALUE(active >= 1 && active <= 11, "active must be in [1, 11], got ", active);
  return active;
}

template <int ACTIVE>
Tensor tri12_cuda(const Tensor& base, LTHC_T12(dz), const Tensor& gamma) {
  const std::array<Tensor, 12> dzs{LTHC_A12(dz)};
  return tri12_forward(base, dzs, gamma, ACTIVE);
}

Tensor tri12_active_cuda(const Tensor& base, LTHC_T12(dz), const Tensor& gamma, int64_t active) {
  const std::array<Tensor, 12> dzs{LTHC_A12(dz)};
  return tri12_forward(base, dzs, gamma, check_active(active));
}

std::tuple<std::vector<Tensor>, Tensor> ws_backward_cuda(const Tensor& grad_, TensorList dzs_, const Tensor& gamma_,
                                                         int64_t L, bool want_dz) {
  on_gpu(grad_, gamma_);
  on_gpu_list(grad_, dzs_);
  const int64_t c = grad_.size(-1), rows = c ? grad_.numel() / c : 0;
  TORCH_CHECK_VALUE(L >= 1 && L <= kMaxWsDepth, "depth ", L, " outside 1..", kMaxWsDepth);
  TORCH_CHECK_VALUE(gamma_.dim() == 2 && gamma_.size(0) >= L && gamma_.size(1) == c, "gamma must be [>= ", L, ", ", c,
                    "], got ", shape(gamma_));
  TORCH_CHECK_VALUE(dzs_.empty() || static_cast<int64_t>(dzs_.size()) >= L, "expected ", L, " dz, got ", dzs_.size());
  for (const Tensor& dz : dzs_)
    TORCH_CHECK_VALUE(dz.numel() == grad_.numel(), "dz ", shape(dz), " does not match grad ", shape(grad_));
  const Tensor grad = prep(grad_), gamma = gamma_.contiguous();
  std::vector<Tensor> gdz;
  if (want_dz)
    for (int64_t i = 0; i < L; ++i) gdz.push_back(at::empty_like(grad));
  std::vector<Tensor> dzs;
  Tensor gg = fp32_like({0}, grad), ws;
  if (!dzs_.empty()) {
    dzs = prep_all(dzs_.slice(0, L), grad.scalar_type());
    gg = fp32_like({L, c}, grad);
    ws = workspace(lthc_ws_accumulate_bwd_workspace_bytes(rows, c, static_cast<int>(L)), grad);
  }
  const auto dp = pointers(dzs);
  const auto gp = pointers<void>(gdz);
  const Launch l(grad);
  check(lthc_ws_accumulate_bwd(data(grad), dzs.empty() ? nullptr : dp.data(), code(grad), data(gamma), code(gamma),
                               want_dz ? gp.data() : nullptr, dzs.empty() ? nullptr : static_cast<float*>(data(gg)),
                               rows, c, static_cast<int>(L), ws.defined() ? data(ws) : nullptr,
                               ws.defined() ? ws.numel() : 0, l.stream),
        "lthc_ws_accumulate_bwd");
  return {gdz, gg};
}

// ---------------------------------------------------------------------------
// the transformer branch
// ---------------------------------------------------------------------------
// Per-sample [B, C] rows: strided rows of one buffer (chunks of the shared AdaLN vector) in place when their rows are
// contiguous, share a stride that is a multiple of `elems` and start `elems`-element aligned; else copies of stride C.
template <size_t NR>
int64_t mod_rows(std::array<Tensor, NR>& ts, int64_t elems) {
  const int64_t c = ts[0].size(1), ld = ts[0].stride(0);
  auto starts = [&](const Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) / t.element_size() % elems == 0;
  };
  bool ok = ld >= c && ld % elems == 0;
  for (const Tensor& t : ts) ok = ok && t.stride(1) == 1 && t.stride(0) == ld && starts(t);
  if (ok) return ld;
  for (Tensor& t : ts) {
    t = t.contiguous();
    if (!starts(t)) t = t.clone();
  }
  return c;
}

// A norm weight or gamma row as the kernels take it: fp32, bf16 or fp16, aligned to 4 elements.
Tensor norm_weight(const Tensor& w) { return prep(known_dtype(w) ? w : w.to(at::kFloat)); }

struct Bnc {
  int64_t b, n, c;
};

Bnc check_norm(const Tensor& x, const Tensor& weight, const Tensor& shift, const Tensor& scale) {
  TORCH_CHECK_VALUE(x.dim() == 3, "x must be [B,N,C], got ", shape(x));
  const int64_t b = x.size(0), n = x.size(1), c = x.size(2);
  TORCH_CHECK_VALUE(has_shape(weight, {c}) && has_shape(shift, {b, c}) && has_shape(scale, {b, c}), "weight [", c,
                    "], shift and scale [", b, ",", c, "] expected, got ", shape(weight), ", ", shape(shift), ", ",
                    shape(scale));
  TORCH_CHECK_VALUE(shift.scalar_type() == x.scalar_type() && scale.scalar_type() == x.scalar_type(),
                    "shift and scale must have x's dtype ", x.scalar_type(), ", got ", shift.scalar_type(), ", ",
                    scale.scalar_type());
  TORCH_CHECK_VALUE(c % 4 == 0 && c <= kNormMaxChannels, "channels ", c, " must be a multiple of 4 and at most ",
                    kNormMaxChannels);
  code(x);
  return {b, n, c};
}

std::tuple<Tensor, Tensor> norm_modulate_cuda(const Tensor& x_, const Tensor& weight, const Tensor& shift,
                                              const Tensor& scale, double eps) {
  on_gpu(x_, weight, shift, scale);
  const Bnc s = check_norm(x_, weight, shift, scale);
  const Tensor x = prep(x_), w = norm_weight(weight);
  std::array<Tensor, 2> r{shift, scale};
  const int64_t ld = mod_rows(r, 4);
  Tensor y = at::empty_like(x), inv = fp32_like({s.b * s.n}, x);
  const Launch l(x);
  check(lthc_norm_modulate_fwd(data(x), code(x), data(w), code(w), data(r[0]), data(r[1]), ld, data(y),
                               static_cast<float*>(data(inv)), s.b, s.n, s.c, static_cast<float>(eps), l.stream),
        "lthc_norm_modulate_fwd");
  return {y, inv};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> norm_modulate_backward_cuda(const Tensor& grad_, const Tensor& x_,
                                                                       const Tensor& weight, const Tensor& scale,
                                                                       const Tensor& inv_) {
  on_gpu(grad_, x_, weight, scale, inv_);
  const Bnc s = check_norm(x_, weight, scale, scale);
  check_like(grad_, {s.b, s.n, s.c}, "grad");
  TORCH_CHECK_VALUE(inv_.numel() == s.b * s.n, "inv must hold ", s.b * s.n, " values, got ", shape(inv_));
  const Tensor x = prep(x_), grad = prep_as(grad_, x.scalar_type()), w = norm_weight(weight);
  const Tensor inv = inv_.to(at::kFloat).contiguous();
  std::array<Tensor, 1> r{scale};
  const int64_t ld = mod_rows(r, 4);
  Tensor gx = at::empty_like(x), gw = fp32_like({s.c}, x), gsh = fp32_like({s.b, s.c}, x), gsc = fp32_like({s.b, s.c}, x);
  const Tensor ws = workspace(lthc_norm_modulate_bwd_workspace_bytes(s.b, s.n, s.c), x);
  const Launch l(x);
  check(lthc_norm_modulate_bwd(data(grad), data(x), code(x), data(w), code(w), data(r[0]), ld,
                               static_cast<const float*>(data(inv)), data(gx), static_cast<float*>(data(gw)),
                               static_cast<float*>(data(gsh)), static_cast<float*>(data(gsc)), s.b, s.n, s.c, data(ws),
                               ws.numel(), l.stream),
        "lthc_norm_modulate_bwd");
  return {gx, gw, gsh, gsc};
}

struct QkGeom {
  int64_t b, n, h;
};

QkGeom check_qk(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos, const Tensor& sin) {
  TORCH_CHECK_VALUE(qkv.dim() == 5 && qkv.size(2) == 3 && qkv.size(4) == kQkHeadDim, "qkv must be [B,N,3,H,", kQkHeadDim,
                    "], got ", shape(qkv));
  const int64_t n = qkv.size(1), d = kQkHeadDim;
  TORCH_CHECK_VALUE(has_shape(qw, {d}) && has_shape(kw, {d}), "q/k norm weights must be [", d, "], got ", shape(qw), ", ",
                    shape(kw));
  TORCH_CHECK_VALUE(has_shape(cos, {n, d}) && has_shape(sin, {n, d}), "RoPE tables must be [", n, ",", d, "], got ",
                    shape(cos), ", ", shape(sin));
  code(qkv);
  return {qkv.size(0), n, qkv.size(3)};
}

// q and k weights, cos and sin as the kernels take them: fp32 or the activation dtype (bf16 parameters and buffers are
// used as they are), each pair in one dtype, 16-byte aligned.
struct QkOperands {
  Tensor qw, kw, cos, sin;
  QkOperands(const Tensor& qkv, const Tensor& q, const Tensor& k, const Tensor& c, const Tensor& s) {
    auto pair = [&](const Tensor& a, const Tensor& b, Tensor& x, Tensor& y) {
      auto own = [&](const Tensor& t) { return t.scalar_type() == qkv.scalar_type() ? t : t.to(at::kFloat); };
      x = own(a);
      y = own(b);
      if (x.scalar_type() != y.scalar_type()) {
        x = x.to(at::kFloat);
        y = y.to(at::kFloat);
      }
      x = prep16(x);
      y = prep16(y);
    };
    pair(q, k, qw, kw);
    pair(c, s, cos, sin);
  }
};

void check_attention(const Tensor& qkv) {
  const int64_t n = qkv.size(1);
  TORCH_CHECK_VALUE((qkv.scalar_type() == at::kBFloat16 || qkv.scalar_type() == at::kHalf) && n % 64 == 0 && n > 0 &&
                        n <= kAttnMaxTokens,
                    "qkv must be bf16 or fp16 [B,N,3,H,64] with N a multiple of 64 up to ", kAttnMaxTokens, ", got ",
                    shape(qkv), " ", qkv.scalar_type());
}

std::tuple<Tensor, Tensor> qk_norm_rope_cuda(const Tensor& qkv_, const Tensor& q_weight, const Tensor& k_weight,
                                             const Tensor& cos, const Tensor& sin, double eps) {
  on_gpu(qkv_, q_weight, k_weight, cos, sin);
  const QkGeom s = check_qk(qkv_, q_weight, k_weight, cos, sin);
  const Tensor qkv = prep16(qkv_);
  const QkOperands o(qkv, q_weight, k_weight, cos, sin);
  Tensor q = at::empty({s.b, s.n, s.h, kQkHeadDim}, qkv.options()), k = at::empty_like(q);
  const Launch l(qkv);
  check(lthc_qk_norm_rope(data(qkv), code(qkv), data(o.qw), data(o.kw), code(o.qw), data(o.cos), data(o.sin),
                          code(o.cos), data(q), data(k), s.b, s.n, s.h, kQkHeadDim, static_cast<float>(eps), l.stream),
        "lthc_qk_norm_rope");
  return {q, k};
}

std::tuple<Tensor, Tensor> qk_norm_rope_backward_cuda(const Tensor& grad_q, const Tensor& grad_k, const Tensor& qkv_,
                                                      const Tensor& q_weight, const Tensor& k_weight, const Tensor& cos,
                                                      const Tensor& sin, double eps) {
  on_gpu(qkv_, grad_q, grad_k, q_weight, k_weight, cos, sin);
  const QkGeom s = check_qk(qkv_, q_weight, k_weight, cos, sin);
  check_like(grad_q, {s.b, s.n, s.h, kQkHeadDim}, "grad_q");
  check_like(grad_k, {s.b, s.n, s.h, kQkHeadDim}, "grad_k");
  const Tensor qkv = prep16(qkv_);
  const Tensor gq = prep16(grad_q.to(qkv.scalar_type())), gk = prep16(grad_k.to(qkv.scalar_type()));
  const QkOperands o(qkv, q_weight, k_weight, cos, sin);
  Tensor dqkv = at::empty_like(qkv), dw = fp32_like({2, kQkHeadDim}, qkv);
  const Tensor ws = workspace(lthc_qk_norm_rope_bwd_workspace_bytes(s.b, s.n, s.h, kQkHeadDim), qkv);
  const Launch l(qkv);
  check(lthc_qk_norm_rope_bwd(data(qkv), data(gq), data(gk), code(qkv), data(o.qw), data(o.kw), code(o.qw), data(o.cos),
                              data(o.sin), code(o.cos), data(dqkv), data(dw), LTHC_F32, s.b, s.n, s.h, kQkHeadDim,
                              static_cast<float>(eps), data(ws), ws.numel(), l.stream),
        "lthc_qk_norm_rope_bwd");
  return {dqkv, dw};
}

const float kAttnScale = 0.125f;  // 1 / sqrt(64)

Tensor attention_cuda(const Tensor& qkv_, const Tensor& q_weight, const Tensor& k_weight, const Tensor& cos,
                      const Tensor& sin, double eps) {
  on_gpu(qkv_, q_weight, k_weight, cos, sin);
  const QkGeom s = check_qk(qkv_, q_weight, k_weight, cos, sin);
  check_attention(qkv_);
  const Tensor qkv = prep16(qkv_);
  const QkOperands o(qkv, q_weight, k_weight, cos, sin);
  Tensor out = at::empty({s.b, s.n, s.h, kQkHeadDim}, qkv.options());
  const Launch l(qkv);
  check(lthc_qk_norm_rope_attention(data(qkv), code(qkv), data(o.qw), data(o.kw), code(o.qw), data(o.cos), data(o.sin),
                                    code(o.cos), data(out), s.b, s.n, s.h, kQkHeadDim, static_cast<float>(eps),
                                    kAttnScale, l.stream),
        "lthc_qk_norm_rope_attention");
  return out;
}

std::tuple<Tensor, Tensor> attention_backward_cuda(const Tensor& grad_, const Tensor& qkv_, const Tensor& q_weight,
                                                   const Tensor& k_weight, const Tensor& cos, const Tensor& sin,
                                                   double eps) {
  on_gpu(qkv_, grad_, q_weight, k_weight, cos, sin);
  const QkGeom s = check_qk(qkv_, q_weight, k_weight, cos, sin);
  check_attention(qkv_);
  check_like(grad_, {s.b, s.n, s.h, kQkHeadDim}, "grad");
  const Tensor qkv = prep16(qkv_), grad = prep16(grad_.to(qkv.scalar_type()));
  const QkOperands o(qkv, q_weight, k_weight, cos, sin);
  Tensor dqkv = at::empty_like(qkv), dw = fp32_like({2, kQkHeadDim}, qkv);
  const Tensor ws = workspace(lthc_qk_norm_rope_attention_bwd_workspace_bytes(s.b, s.n, s.h, kQkHeadDim), qkv);
  const Launch l(qkv);
  check(lthc_qk_norm_rope_attention_bwd(data(qkv), data(grad), code(qkv), data(o.qw), data(o.kw), code(o.qw),
                                        data(o.cos), data(o.sin), code(o.cos), data(dqkv), data(dw), LTHC_F32, s.b, s.n,
                                        s.h, kQkHeadDim, static_cast<float>(eps), kAttnScale, data(ws), ws.numel(),
                                        l.stream),
        "lthc_qk_norm_rope_attention_bwd");
  return {dqkv, dw};
}

Tensor swiglu_cuda(const Tensor& x_) {
  on_gpu(x_);
  const int64_t two_f = x_.size(-1);
  TORCH_CHECK_VALUE(two_f % 16 == 0, "last dimension ", two_f, " must be 2F with F a multiple of 8");
  code(x_);
  const Tensor x = prep16(x_);
  auto sizes = x.sizes().vec();
  sizes.back() = two_f / 2;
  Tensor out = at::empty(sizes, x.options());
  const Launch l(x);
  check(lthc_swiglu(data(x), code(x), data(out), two_f ? x.numel() / two_f : 0, two_f / 2, l.stream), "lthc_swiglu");
  return out;
}

Tensor swiglu_backward_cuda(const Tensor& grad_, const Tensor& x_) {
  on_gpu(x_, grad_);
  const int64_t two_f = x_.size(-1);
  auto sizes = x_.sizes().vec();
  sizes.back() = two_f / 2;
  TORCH_CHECK_VALUE(two_f % 16 == 0 && grad_.sizes() == at::IntArrayRef(sizes),
                    "x [..., 2F] with F % 8 == 0 and grad [..., F] expected, got ", shape(x_), ", ", shape(grad_));
  code(x_);
  const Tensor x = prep16(x_), grad = prep16(grad_.to(x.scalar_type()));
  Tensor gx = at::empty_like(x);
  const Launch l(x);
  check(lthc_swiglu_bwd(data(x), data(grad), code(x), data(gx), two_f ? x.numel() / two_f : 0, two_f / 2, l.stream),
        "lthc_swiglu_bwd");
  return gx;
}

void check_bnc(const char* name, const Tensor& t, at::IntArrayRef want, at::ScalarType dtype) {
  TORCH_CHECK_VALUE(t.sizes() == want && t.scalar_type() == dtype, name, " must be ", want, " ", dtype, ", got ", shape(t),
                    " ", t.scalar_type());
}

std::tuple<Tensor, Tensor> gate_add_norm_modulate_cuda(const Tensor& z_, const Tensor& a_, const Tensor& gate,
                                                       const Tensor& weight, const Tensor& shift, const Tensor& scale,
                                                       double eps) {
  on_gpu(z_, a_, gate, weight, shift, scale);
  TORCH_CHECK_VALUE(z_.dim() == 3, "z must be [B,N,C], got ", shape(z_));
  const int64_t b = z_.size(0), n = z_.size(1), c = z_.size(2);
  const auto dt = z_.scalar_type();
  check_bnc("a", a_, {b, n, c}, dt);
  check_bnc("gate", gate, {b, c}, dt);
  check_bnc("shift", shift, {b, c}, dt);
  check_bnc("scale", scale, {b, c}, dt);
  TORCH_CHECK_VALUE(has_shape(weight, {c}), "weight must be [", c, "], got ", shape(weight));
  code(z_);
  const Tensor z = prep16(z_), a = prep16(a_), w = norm_weight(weight);
  std::array<Tensor, 3> r{gate, shift, scale};
  const int64_t ld = mod_rows(r, 4);
  Tensor d = at::empty_like(z), y = at::empty_like(z);
  const Launch l(z);
  check(lthc_gate_add_norm_modulate_fwd(data(z), data(a), data(r[0]), code(z), data(w), code(w), data(r[1]), data(r[2]),
                                        ld, data(d), data(y), nullptr, b, n, c, static_cast<float>(eps), l.stream),
        "lthc_gate_add_norm_modulate_fwd");
  return {d, y};
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> gate_add_norm_modulate_backward_cuda(
    const std::optional<Tensor>& grad_d, const Tensor& grad_y, const Tensor& z_, const Tensor& a_, const Tensor& gate,
    const Tensor& weight, const Tensor& scale, double eps) {
  on_gpu(z_, a_, gate, weight, scale, grad_y);
  TORCH_CHECK_VALUE(z_.dim() == 3, "z must be [B,N,C], got ", shape(z_));
  const int64_t b = z_.size(0), n = z_.size(1), c = z_.size(2);
  const auto dt = z_.scalar_type();
  check_like(a_, {b, n, c}, "a");
  check_like(grad_y, {b, n, c}, "grad");
  const bool has_gd = grad_d.has_value() && grad_d->defined();
  if (has_gd) check_like(*grad_d, {b, n, c}, "grad");
  if (has_gd) same_device(z_, *grad_d);
  check_bnc("gate", gate, {b, c}, dt);
  check_bnc("scale", scale, {b, c}, dt);
  TORCH_CHECK_VALUE(has_shape(weight, {c}), "weight must be [", c, "], got ", shape(weight));
  code(z_);
  const Tensor z = prep(z_), a = prep_as(a_, dt), gy = prep_as(grad_y, dt), w = norm_weight(weight);
  const Tensor gd = has_gd ? prep_as(*grad_d, dt) : Tensor();
  std::array<Tensor, 2> r{gate, scale};
  const int64_t ld = mod_rows(r, 4);
  Tensor gz = at::empty_like(z), ga = at::empty_like(z);
  Tensor ggate = at::empty({b, c}, z.options()), gshift = at::empty_like(ggate), gscale = at::empty_like(ggate);
  Tensor gw = at::empty({c}, z.options().dtype(known_dtype(weight) ? weight.scalar_type() : at::kFloat));
  const Tensor ws = workspace(lthc_gate_add_norm_modulate_bwd_workspace_bytes(b, n, c), z);
  const Launch l(z);
  check(lthc_gate_add_norm_modulate_bwd(has_gd ? data(gd) : nullptr, data(gy), data(z), data(a), data(r[0]), code(z),
                                        data(w), code(w), data(r[1]), ld, data(gz), data(ga), data(ggate), data(gshift),
                                        data(gscale), data(gw), code(gw), b, n, c, static_cast<float>(eps), data(ws),
                                        ws.numel(), l.stream),
        "lthc_gate_add_norm_modulate_bwd");
  return {gz, ga, ggate, gw, gshift, gscale};
}

Tensor gate_residual_cuda(const Tensor& d_, const Tensor& gate, const Tensor& m_) {
  on_gpu(d_, gate, m_);
  TORCH_CHECK_VALUE(d_.dim() == 3 && d_.size(2) % 8 == 0, "d must be [B,N,C] with C % 8 == 0, got ", shape(d_));
  const int64_t b = d_.size(0), n = d_.size(1), c = d_.size(2);
  check_bnc("m", m_, {b, n, c}, d_.scalar_type());
  check_bnc("gate", gate, {b, c}, d_.scalar_type());
  code(d_);
  const Tensor d = prep16(d_), m = prep16(m_);
  std::array<Tensor, 1> r{gate};
  const int64_t ld = mod_rows(r, 8);
  Tensor out = at::empty_like(d);
  const Launch l(d);
  check(lthc_gate_residual(data(d), data(r[0]), ld, data(m), code(d), data(out), b, n, c, l.stream), "lthc_gate_residual");
  return out;
}

std::tuple<Tensor, Tensor> gate_residual_backward_cuda(const Tensor& grad_, const Tensor& gate, const Tensor& m_) {
  on_gpu(grad_, gate, m_);
  TORCH_CHECK_VALUE(grad_.dim() == 3, "grad must be [B,N,C], got ", shape(grad_));
  const int64_t b = grad_.size(0), n = grad_.size(1), c = grad_.size(2);
  check_bnc("m", m_, {b, n, c}, grad_.scalar_type());
  check_bnc("gate", gate, {b, c}, grad_.scalar_type());
  const Tensor grad = prep(grad_), m = prep(m_);
  std::array<Tensor, 1> r{gate};
  const int64_t ld = mod_rows(r, 4);
  Tensor gm = at::empty_like(m), ggate = at::empty({b, c}, m.options());
  const Tensor ws = workspace(lthc_gate_residual_bwd_workspace_bytes(b, n, c), m);
  const Launch l(m);
  check(lthc_gate_residual_bwd(data(grad), data(m), data(r[0]), ld, code(m), data(gm), data(ggate), b, n, c, data(ws),
                               ws.numel(), l.stream),
        "lthc_gate_residual_bwd");
  return {ggate, gm};
}

// (gW [N, K], gb [N] or an empty tensor) of a linear layer for the output gradient [..., N] and the input [..., K].
std::tuple<Tensor, Tensor> linear_weight_grad_cuda(const Tensor& grad_, const Tensor& x_, bool need_bias) {
  on_gpu(grad_, x_);
  TORCH_CHECK_VALUE(grad_.dim() >= 1 && grad_.dim() == x_.dim() && grad_.sizes().slice(0, grad_.dim() - 1) ==
                                                                      x_.sizes().slice(0, x_.dim() - 1),
                    "grad [..., N] and x [..., K] expected, got ", shape(grad_), " and ", shape(x_));
  TORCH_CHECK_VALUE(grad_.scalar_type() == x_.scalar_type(), "grad and x must have one dtype, got ", grad_.scalar_type(),
                    ", ", x_.scalar_type());
  const Tensor grad = prep16(grad_), x = prep16(x_);
  const int64_t n = grad.size(-1), k = x.size(-1), m = n ? grad.numel() / n : 0;
  Tensor gw = at::empty({n, k}, grad.options()), gb = at::empty({need_bias ? n : 0}, grad.options());
  const Tensor ws = workspace(lthc_linear_weight_grad_workspace_bytes(m, n, k), grad);
  const Launch l(grad);
  check(lthc_linear_weight_grad(data(grad), data(x), code(grad), data(gw), need_bias ? data(gb) : nullptr, m, n, k, data(ws),
                                ws.numel(), l.stream),
        "lthc_linear_weight_grad");
  return {gw, gb};
}

std::tuple<Tensor, Tensor, Tensor> block_tail_cuda(const Tensor& z_, const Tensor& a_, const Tensor& gate,
                                                   const Tensor& m_, const Tensor& gamma, const Tensor& weight,
                                                   const Tensor& shift, const Tensor& scale, double eps) {
  on_gpu(z_, a_, gate, m_, gamma, weight, shift, scale);
  TORCH_CHECK_VALUE(z_.dim() == 3 && z_.size(2) % 8 == 0, "z must be [B,N,C] with C % 8 == 0, got ", shape(z_));
  const int64_t b = z_.size(0), n = z_.size(1), c = z_.size(2);
  const auto dt = z_.scalar_type();
  check_bnc("a", a_, {b, n, c}, dt);
  check_bnc("m", m_, {b, n, c}, dt);
  check_bnc("gate", gate, {b, c}, dt);
  check_bnc("shift", shift, {b, c}, dt);
  check_bnc("scale", scale, {b, c}, dt);
  TORCH_CHECK_VALUE(has_shape(gamma, {c}), "gamma must be [", c, "], got ", shape(gamma));
  TORCH_CHECK_VALUE(has_shape(weight, {c}), "weight must be [", c, "], got ", shape(weight));
  code(z_);
  const Tensor z = prep16(z_), a = prep16(a_), m = prep16(m_), w = norm_weight(weight), g = norm_weight(gamma);
  std::array<Tensor, 3> r{gate, shift, scale};
  const int64_t ld = mod_rows(r, 4);
  Tensor dz = at::empty_like(z), zn = at::empty_like(z), y = at::empty_like(z);
  const Launch l(z);
  check(lthc_block_tail_fwd(data(z), data(a), data(m), data(r[0]), code(z), data(g), code(g), data(w), code(w), data(r[1]),
                            data(r[2]), ld, data(dz), data(zn), data(y), b, n, c, static_cast<float>(eps), l.stream),
        "lthc_block_tail_fwd");
  return {dz, zn, y};
}

// ---------------------------------------------------------------------------
// autograd
// ---------------------------------------------------------------------------
// The dispatcher's handle of an operator, looked up once.

#define LTHC_OP(fn, name, ...)                                                                                       \
  const c10::TypedOperatorHandle<__VA_ARGS__>& fn() {                                                               \
    static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("jit_thc::" name, "").typed<__VA_ARGS__>(); \
    return op;                                                                                                       \
  }

LTHC_OP(op_read, "local_write_traceable", Tensor(const Tensor&, const Tensor&))
LTHC_OP(op_write, "local_read_traceable", Tensor(const Tensor&, const Tensor&))
LTHC_OP(op_write_add, "local_read_add_traceable", Tensor(const Tensor&, const Tensor&, const Tensor&))
LTHC_OP(op_weight_grad, "local_weight_grad_traceable", Tensor(const Tensor&, const Tensor&))
LTHC_OP(op_final_list, "final_accumulate_list", Tensor(const Tensor&, TensorList, TensorList))
LTHC_OP(op_final_12, "final_accumulate_b4_12_traceable", Tensor(const Tensor&, LTHC_TYPES12, LTHC_TYPES12))
LTHC_OP(op_final_backward, "final_accumulate_backward", std::tuple<Tensor, Tensor>(const Tensor&, TensorList, TensorList))
LTHC_OP(op_list_grad_dz, "final_accumulate_list_grad_dz", std::vector<Tensor>(const Tensor&, TensorList))
LTHC_OP(op_list_grad_beta, "final_accumulate_list_grad_beta", Tensor(const Tensor&, TensorList))
LTHC_OP(op_12_grad_dz, "final_accumulate_b4_12_grad_dz_ptr", Tensor(const Tensor&, LTHC_TYPES12))
LTHC_OP(op_12_grad_beta, "final_accumulate_b4_12_grad_beta_ptr", Tensor(const Tensor&, LTHC_TYPES12))
LTHC_OP(op_recur, "lazy_workspace_update", Tensor(const Tensor&, const Tensor&, const Tensor&))
LTHC_OP(op_recur_backward, "lazy_workspace_update_backward",
        std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const std::optional<Tensor>&))
LTHC_OP(op_recur_backward_sum, "lazy_workspace_update_backward_sum",
        std::tuple<Tensor, Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                           const std::optional<Tensor>&))
LTHC_OP(op_gamma_rounded, "lazy_gamma_rounded", Tensor(const Tensor&, TensorList, at::ScalarType))
LTHC_OP(op_gamma_rounded_backward, "lazy_gamma_rounded_backward",
        std::tuple<Tensor, std::vector<Tensor>>(const Tensor&, const Tensor&, TensorList, bool, bool))
LTHC_OP(op_all_base_split, "all_base_b4_12_split_traceable", std::vector<Tensor>(const Tensor&, const Tensor&))
LTHC_OP(op_all_base_backward, "all_base_backward",
        std::tuple<Tensor, Tensor>(const Tensor&, TensorList, const Tensor&, bool, bool))
LTHC_OP(op_all_base_grad_x, "all_base_b4_12_grad_x", Tensor(const Tensor&, const Tensor&))
LTHC_OP(op_all_base_grad_alpha, "all_base_b4_12_split_grad_alpha", Tensor(const Tensor&, const Tensor&))
LTHC_OP(op_tri_list, "triangular_accumulate_list", Tensor(const Tensor&, TensorList, const Tensor&))
LTHC_OP(op_ws_backward, "ws_accumulate_backward",
        std::tuple<std::vector<Tensor>, Tensor>(const Tensor&, TensorList, const Tensor&, c10::SymInt, bool))
LTHC_OP(op_norm, "norm_modulate",
        std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&, double))
LTHC_OP(op_norm_backward, "norm_modulate_backward",
        std::tuple<Tensor, Tensor, Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                                   const Tensor&))
LTHC_OP(op_qk, "qk_norm_rope",
        std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, double))
LTHC_OP(op_qk_backward, "qk_norm_rope_backward",
        std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                   const Tensor&, const Tensor&, double))
LTHC_OP(op_attention, "qk_norm_rope_attention",
        Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, double))
LTHC_OP(op_attention_backward, "qk_norm_rope_attention_backward",
        std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                   const Tensor&, double))
LTHC_OP(op_swiglu, "swiglu", Tensor(const Tensor&))
LTHC_OP(op_swiglu_backward, "swiglu_backward", Tensor(const Tensor&, const Tensor&))
LTHC_OP(op_ganm, "gate_add_norm_modulate",
        std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                   const Tensor&, double))
LTHC_OP(op_ganm_backward, "gate_add_norm_modulate_backward",
        std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>(const std::optional<Tensor>&, const Tensor&,
                                                                   const Tensor&, const Tensor&, const Tensor&,
                                                                   const Tensor&, const Tensor&, double))
LTHC_OP(op_gres, "gate_residual", Tensor(const Tensor&, const Tensor&, const Tensor&))
LTHC_OP(op_gres_backward, "gate_residual_backward", std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&))

#define LTHC_REPLAY(fn, name) LTHC_OP(fn, name "_backward_replay", std::vector<Tensor>(TensorList, TensorList, double))
LTHC_REPLAY(replay_qk, "qk_norm_rope")
LTHC_REPLAY(replay_attention, "qk_norm_rope_attention")
LTHC_REPLAY(replay_swiglu, "swiglu")
LTHC_REPLAY(replay_ganm, "gate_add_norm_modulate")
LTHC_OP(op_linear_weight_grad, "linear_weight_grad", std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, bool))

using BelowAutograd = at::AutoDispatchBelowADInplaceOrView;

bool records(const Tensor& t) { return t.requires_grad(); }
bool records(TensorList ts) {
  for (const Tensor& t : ts)
    if (t.requires_grad()) return true;
  return false;
}
// Whether autograd records a call on these tensors.
template <typename... Ts>
bool recording(const Ts&... ts) {
  return at::GradMode::is_enabled() && (records(ts) || ...);
}

// In a backward: ops are called below autograd unless a graph of the backward is being built (create_graph), where they
// go through autograd as the formulas of the reference do.
struct BackwardScope {
  std::optional<BelowAutograd> below;
  BackwardScope() {
    if (!at::GradMode::is_enabled()) below.emplace();
  }
};

// For the branch's ops, whose gradients are constants of a graph of the backward.
struct DetachedScope {
  at::NoGradGuard no_grad;
  BelowAutograd below;
};

// Whether the call is being traced (fake, functional or other Python-dispatched tensors, as torch.compile's).  The
// branch's nodes then differentiate the eager sequence in place of their kernels (the *_backward_replay ops): a compiled
// graph keeps the chain's intermediates in fp32, where the kernels round at the eager ops' boundaries.
bool traced(const Tensor& t) {
  return t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::Functionalize}));
}

Tensor as_dtype(const Tensor& t, at::ScalarType dtype) { return t.scalar_type() == dtype ? t : t.to(dtype); }

bool any_needed(AutogradContext* ctx, size_t from, size_t count) {
  for (size_t i = 0; i < count; ++i)
    if (ctx->needs_input_grad(from + i)) return true;
  return false;
}

// Whether a gradient holds a batch of them (is_grads_batched, vmap).  Torch then runs an op once per sample by itself,
// except for ops over tensor lists, which those nodes replace by ops over plain tensors.
bool batched(TensorList ts) {
  const c10::DispatchKeySet keys({c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchBatched});
  for (const Tensor& t : ts)
    if (t.key_set().has_any(keys)) return true;
  return false;
}

Tensor call_12(const c10::TypedOperatorHandle<Tensor(const Tensor&, LTHC_TYPES12)>& op, const Tensor& t, TensorList l) {
  return op.call(t, l[0], l[1], l[2], l[3], l[4], l[5], l[6], l[7], l[8], l[9], l[10], l[11]);
}

struct ReadFn : torch::autograd::Function<ReadFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight) {
    BelowAutograd below;
    ctx->save_for_backward({x, weight});
    return op_read().call(x, weight);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &weight = saved[1];
    Tensor gx, gw;
    if (ctx->needs_input_grad(0)) gx = op_write().call(grads[0], weight);
    if (ctx->needs_input_grad(1)) gw = as_dtype(op_weight_grad().call(x, grads[0]), weight.scalar_type());
    return {gx, gw};
  }
};

struct WriteFn : torch::autograd::Function<WriteFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& z, const Tensor& weight) {
    BelowAutograd below;
    ctx->save_for_backward({z, weight});
    return op_write().call(z, weight);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const Tensor &z = saved[0], &weight = saved[1];
    Tensor gz, gw;
    if (ctx->needs_input_grad(0)) gz = op_read().call(grads[0], weight);
    if (ctx->needs_input_grad(1)) gw = as_dtype(op_weight_grad().call(grads[0], z), weight.scalar_type());
    return {gz, gw};
  }
};

struct WriteAddFn : torch::autograd::Function<WriteAddFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& z, const Tensor& weight, const Tensor& x) {
    BelowAutograd below;
    ctx->save_for_backward({z, weight});
    return op_write_add().call(z, weight, x);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const Tensor &z = saved[0], &weight = saved[1];
    Tensor gz, gw;
    if (ctx->needs_input_grad(0)) gz = op_read().call(grads[0], weight);
    if (ctx->needs_input_grad(1)) gw = as_dtype(op_weight_grad().call(grads[0], z), weight.scalar_type());
    return {gz, gw, grads[0]};
  }
};

// (x, Z0 = R(x)) as one node, x returned as a view of itself: its gradient and Z0's arrive together, and
// dX = g_x + R^T gZ0 is one pass.  The alias is made outside the guard: autograd then knows it as a view that shares
// the saved x's version counter, and refuses an in-place change of it.
struct OpenFn : torch::autograd::Function<OpenFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight) {
    const Tensor alias = x.view_as(x);
    BelowAutograd below;
    ctx->save_for_backward({x, weight});
    ctx->set_materialize_grads(false);  // an unused output's gradient stays undefined
    return {alias, op_read().call(x, weight)};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &weight = saved[1], &gx = grads[0], &gz = grads[1];
    if (!gz.defined()) return {gx, Tensor()};
    Tensor dx, dw;
    if (ctx->needs_input_grad(0))
      dx = gx.defined() ? op_write_add().call(gz, weight, as_dtype(gx, x.scalar_type())) : op_write().call(gz, weight);
    if (ctx->needs_input_grad(1)) dw = as_dtype(op_weight_grad().call(x, gz), weight.scalar_type());
    return {dx, dw};
  }
};

// Gradients of X_L = x0 + sum_l P_l(dz_l): grad_x0 is grad_out itself; gdZ and gbeta from one pass when both are wanted.
variable_list final_grads(AutogradContext* ctx, const Tensor& grad, TensorList dzs, TensorList betas) {
  const size_t L = dzs.size();
  const Tensor grad_out = grad.contiguous();
  const bool want_dz = any_needed(ctx, 1, L), want_beta = any_needed(ctx, 1 + L, L);
  variable_list out(1 + 2 * L);
  out[0] = grad_out;
  Tensor gb;
  if (L == 12 && batched(grad_out)) {
    if (want_dz) {
      const auto parts = call_12(op_12_grad_dz(), grad_out, betas).unbind(0);
      for (size_t i = 0; i < L; ++i) out[1 + i] = parts[i];
    }
    if (want_beta) gb = call_12(op_12_grad_beta(), grad_out, dzs);
  } else if (want_dz && want_beta) {
    Tensor gdz;
    std::tie(gdz, gb) = op_final_backward().call(grad_out, dzs, betas);
    const auto parts = gdz.unbind(0);
    for (size_t i = 0; i < L; ++i) out[1 + i] = parts[i];
  } else if (want_dz) {
    const auto parts = op_list_grad_dz().call(grad_out, betas);
    for (size_t i = 0; i < L; ++i) out[1 + i] = parts[i];
  } else if (want_beta) {
    gb = op_list_grad_beta().call(grad_out, dzs);
  }
  if (want_beta) {
    const auto parts = gb.unbind(0);
    for (size_t i = 0; i < L; ++i) out[1 + L + i] = as_dtype(parts[i], betas[i].scalar_type());
  }
  return out;
}

variable_list concat(TensorList a, TensorList b) {
  variable_list v(a.begin(), a.end());
  v.insert(v.end(), b.begin(), b.end());
  return v;
}

struct FinalListFn : torch::autograd::Function<FinalListFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x0, TensorList dzs, TensorList betas) {
    BelowAutograd below;
    ctx->save_for_backward(concat(dzs, betas));
    return op_final_list().call(x0, dzs, betas);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const TensorList all(saved);
    return final_grads(ctx, grads[0], all.slice(0, saved.size() / 2), all.slice(saved.size() / 2));
  }
};

Tensor call_final_12(const Tensor& x0, TensorList d, TensorList b) {
  return op_final_12().call(x0, d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7], d[8], d[9], d[10], d[11], b[0], b[1], b[2],
                            b[3], b[4], b[5], b[6], b[7], b[8], b[9], b[10], b[11]);
}

struct Final12Fn : torch::autograd::Function<Final12Fn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x0, TensorList dzs, TensorList betas) {
    BelowAutograd below;
    ctx->save_for_backward(concat(dzs, betas));
    return call_final_12(x0, dzs, betas);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    return FinalListFn::backward(ctx, grads);
  }
};

struct RecurFn : torch::autograd::Function<RecurFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& z, const Tensor& dz, const Tensor& gamma) {
    BelowAutograd below;
    ctx->save_for_backward({dz, gamma});
    ctx->saved_data["z"] = static_cast<int64_t>(z.scalar_type());
    return op_recur().call(z, dz, gamma);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const Tensor &dz = saved[0], &gamma = saved[1];
    Tensor gz, gdz, gg;
    if (ctx->needs_input_grad(0)) gz = as_dtype(grads[0], static_cast<at::ScalarType>(ctx->saved_data["z"].toInt()));
    if (ctx->needs_input_grad(1) || ctx->needs_input_grad(2)) {
      std::tie(gdz, gg) = op_recur_backward().call(grads[0], dz, gamma, std::nullopt);
      gdz = ctx->needs_input_grad(1) ? as_dtype(gdz, dz.scalar_type()) : Tensor();
      gg = ctx->needs_input_grad(2) ? as_dtype(gg, gamma.scalar_type()) : Tensor();
    }
    return {gz, gdz, gg};
  }
};

// (Z_{l+1}, dZ_l) as one node, or (Z_{l+1}, Z_{l+1} for the branch, dZ_l) with split: dZ_l's two gradients, and with
// split Z_{l+1}'s two, arrive together and one recurrence-backward launch sums them.
struct StepFn : torch::autograd::Function<StepFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& z, const Tensor& dz, const Tensor& gamma, bool split) {
    ctx->save_for_backward({dz, gamma});
    ctx->saved_data["z"] = static_cast<int64_t>(z.scalar_type());
    ctx->saved_data["split"] = split;
    ctx->set_materialize_grads(false);  // an unused Z_{l+1} (the last step's) skips the recurrence backward
    const Tensor zn = [&] {
      BelowAutograd below;
      return op_recur().call(z, dz, gamma);
    }();
    if (split) return {zn, zn.view_as(zn), dz.view_as(dz)};  // views for autograd, as OpenFn's
    return {zn, dz.view_as(dz)};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const bool split = ctx->saved_data["split"].toBool();
    Tensor gzn = grads[0], branch = split ? grads[1] : Tensor();
    const Tensor gdz_in = grads[split ? 2 : 1];
    const auto saved = ctx->get_saved_variables();
    const Tensor &dz = saved[0], &gamma = saved[1];
    if (!gzn.defined()) std::swap(gzn, branch);
    if (!gzn.defined()) return {Tensor(), gdz_in, Tensor(), Tensor()};
    const bool need_dz = ctx->needs_input_grad(1), need_gamma = ctx->needs_input_grad(2);
    std::optional<Tensor> add;
    if (need_dz && gdz_in.defined()) add = gdz_in;
    Tensor gdz, gg;
    if (branch.defined()) {
      std::tie(gzn, gdz, gg) = op_recur_backward_sum().call(gzn, branch, dz, gamma, add);
    } else if (need_dz || need_gamma) {
      std::tie(gdz, gg) = op_recur_backward().call(gzn, dz, gamma, add);
    }
    Tensor gz;
    if (ctx->needs_input_grad(0)) gz = as_dtype(gzn, static_cast<at::ScalarType>(ctx->saved_data["z"].toInt()));
    gdz = need_dz && gdz.defined() ? as_dtype(gdz, dz.scalar_type()) : Tensor();
    gg = need_gamma && gg.defined() ? as_dtype(gg, gamma.scalar_type()) : Tensor();
    return {gz, gdz, gg, Tensor()};
  }
};

struct GammaRoundedFn : torch::autograd::Function<GammaRoundedFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& alpha, TensorList betas, at::ScalarType dtype) {
    BelowAutograd below;
    ctx->save_for_backward(concat(TensorList(alpha), betas));
    ctx->saved_data["dtype"] = static_cast<int64_t>(dtype);
    return op_gamma_rounded().call(alpha, betas, dtype);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const TensorList betas = TensorList(saved).slice(1);
    variable_list out(2 + betas.size());
    const bool need_a = ctx->needs_input_grad(0), need_b = any_needed(ctx, 1, betas.size());
    if (!need_a && !need_b) return out;
    const Tensor g = as_dtype(grads[0], static_cast<at::ScalarType>(ctx->saved_data["dtype"].toInt()));
    auto [ga, gbs] = op_gamma_rounded_backward().call(g, saved[0], betas, need_a, need_b);
    if (need_a) out[0] = ga;
    for (size_t i = 0; need_b && i < betas.size(); ++i) out[1 + i] = as_dtype(gbs[i], betas[i].scalar_type());
    return out;
  }
};

struct AllBaseSplitFn : torch::autograd::Function<AllBaseSplitFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x0, const Tensor& alpha_stack) {
    BelowAutograd below;
    ctx->save_for_backward({x0, alpha_stack});
    return op_all_base_split().call(x0, alpha_stack);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x0 = saved[0], &alpha_stack = saved[1];
    const bool need_x = ctx->needs_input_grad(0), need_a = ctx->needs_input_grad(1);
    Tensor gx, ga;
    if (batched(grads)) {
      const Tensor base = at::stack(grads);
      if (need_x) gx = op_all_base_grad_x().call(base, alpha_stack);
      if (need_a) ga = op_all_base_grad_alpha().call(x0, base);
    } else {
      std::tie(gx, ga) = op_all_base_backward().call(x0, grads, alpha_stack, need_x, need_a);
    }
    return {need_x ? gx : Tensor(), need_a ? as_dtype(ga, alpha_stack.scalar_type()) : Tensor()};
  }
};

// Gradients of base + sum_{i < active} gamma_i dz_i for (base, dz..., gamma): grad_base is grad_out itself, the layers
// beyond the active prefix get none.
variable_list tri_grads(AutogradContext* ctx, const Tensor& grad, TensorList dzs, const Tensor& gamma, int64_t active) {
  const size_t n = dzs.size();
  const Tensor grad_out = grad.contiguous();
  const bool want_dz = any_needed(ctx, 1, active), want_g = ctx->needs_input_grad(1 + n);
  variable_list out(2 + n);
  out[0] = grad_out;
  if (!want_dz && !want_g) return out;
  auto [gdz, gg] = op_ws_backward().call(grad_out, want_g ? dzs.slice(0, active) : TensorList(), gamma, active, want_dz);
  for (size_t i = 0; i < gdz.size(); ++i) out[1 + i] = gdz[i];
  if (want_g) {
    if (gamma.sym_size(0) != active) {
      Tensor full = at::zeros_symint(gamma.sym_sizes(), gg.options());
      full.narrow(0, 0, active).copy_(gg);
      gg = full;
    }
    out[1 + n] = as_dtype(gg, gamma.scalar_type());
  }
  return out;
}

using Tri12Op = c10::TypedOperatorHandle<Tensor(const Tensor&, LTHC_TYPES12, const Tensor&)>;

const Tri12Op& tri12_op(int64_t active) {  // 1..11: the active{N} ops, 12: the full one
  static const std::vector<Tri12Op> ops = [] {
    std::vector<Tri12Op> v;
    for (int i = 1; i <= 12; ++i) {
      const std::string name = "jit_thc::triangular_accumulate_b4_12_ptr_" +
                               (i < 12 ? "active" + std::to_string(i) : std::string("traceable"));
      v.push_back(c10::Dispatcher::singleton()
                      .findSchemaOrThrow(name.c_str(), "")
                      .typed<Tensor(const Tensor&, LTHC_TYPES12, const Tensor&)>());
    }
    return v;
  }();
  return ops[active - 1];
}

Tensor call_tri12(const Tensor& base, TensorList d, const Tensor& gamma, int64_t active) {
  return tri12_op(active).call(base, d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7], d[8], d[9], d[10], d[11], gamma);
}

struct Tri12Fn : torch::autograd::Function<Tri12Fn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& base, TensorList dzs, const Tensor& gamma, int64_t active) {
    BelowAutograd below;
    ctx->save_for_backward(concat(dzs, TensorList(gamma)));
    ctx->saved_data["active"] = active;
    return call_tri12(base, dzs, gamma, active);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    auto out = tri_grads(ctx, grads[0], TensorList(saved).slice(0, 12), saved[12], ctx->saved_data["active"].toInt());
    out.emplace_back();  // no gradient for `active`
    return out;
  }
};

struct TriListFn : torch::autograd::Function<TriListFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& base, TensorList dzs, const Tensor& gamma) {
    BelowAutograd below;
    ctx->save_for_backward(concat(dzs, TensorList(gamma)));
    return op_tri_list().call(base, dzs, gamma);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    const size_t L = saved.size() - 1;
    return tri_grads(ctx, grads[0], TensorList(saved).slice(0, L), saved[L], static_cast<int64_t>(L));
  }
};

struct NormFn : torch::autograd::Function<NormFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const Tensor& shift,
                               const Tensor& scale, double eps) {
    BelowAutograd below;
    auto [y, inv] = op_norm().call(x, weight, shift, scale, eps);
    ctx->save_for_backward({x, weight, scale, inv});
    ctx->saved_data["shift"] = static_cast<int64_t>(shift.scalar_type());
    return {y, inv};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    BackwardScope scope;
    const auto saved = ctx->get_saved_variables();
    auto [gx, gw, gsh, gsc] = op_norm_backward().call(grads[0].contiguous(), saved[0], saved[1], saved[2], saved[3]);
    auto want = [&](size_t i, const Tensor& t, at::ScalarType dt) {
      return ctx->needs_input_grad(i) ? as_dtype(t, dt) : Tensor();
    };
    return {ctx->needs_input_grad(0) ? gx : Tensor(), want(1, gw, saved[1].scalar_type()),
            want(2, gsh, static_cast<at::ScalarType>(ctx->saved_data["shift"].toInt())),
            want(3, gsc, saved[2].scalar_type()), Tensor()};
  }
};

// Gradients of (qkv, q weight, k weight) from the backward op's dqkv and fp32 [2, 64] weight gradients.
variable_list qk_grads(AutogradContext* ctx, const Tensor& dqkv, const Tensor& dw, const variable_list& saved) {
  auto row = [&](int64_t i) {
    return ctx->needs_input_grad(1 + i) ? as_dtype(dw.select(0, i), saved[1 + i].scalar_type()) : Tensor();
  };
  return {ctx->needs_input_grad(0) ? dqkv : Tensor(), row(0), row(1), Tensor(), Tensor(), Tensor()};
}

// The gradients of the first inputs that are asked for, `total` results in all.
variable_list wanted(AutogradContext* ctx, const std::vector<Tensor>& got, size_t total) {
  variable_list out(total);
  for (size_t i = 0; i < got.size(); ++i)
    if (ctx->needs_input_grad(i)) out[i] = got[i];
  return out;
}

struct QkFn : torch::autograd::Function<QkFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& qw, const Tensor& kw,
                               const Tensor& cos, const Tensor& sin, double eps) {
    BelowAutograd below;
    ctx->save_for_backward({qkv, qw, kw, cos, sin});
    ctx->saved_data["eps"] = eps;
    auto [q, k] = op_qk().call(qkv, qw, kw, cos, sin, eps);
    return {q, k};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto s = ctx->get_saved_variables();
    if (traced(s[0])) return wanted(ctx, replay_qk().call(grads, s, ctx->saved_data["eps"].toDouble()), 6);
    DetachedScope scope;
    auto [dqkv, dw] =
        op_qk_backward().call(grads[0], grads[1], s[0], s[1], s[2], s[3], s[4], ctx->saved_data["eps"].toDouble());
    return qk_grads(ctx, dqkv, dw, s);
  }
};

struct AttentionFn : torch::autograd::Function<AttentionFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos,
                        const Tensor& sin, double eps) {
    BelowAutograd below;
    ctx->save_for_backward({qkv, qw, kw, cos, sin});
    ctx->saved_data["eps"] = eps;
    return op_attention().call(qkv, qw, kw, cos, sin, eps);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto s = ctx->get_saved_variables();
    if (traced(s[0])) return wanted(ctx, replay_attention().call(grads, s, ctx->saved_data["eps"].toDouble()), 6);
    DetachedScope scope;
    auto [dqkv, dw] =
        op_attention_backward().call(grads[0], s[0], s[1], s[2], s[3], s[4], ctx->saved_data["eps"].toDouble());
    return qk_grads(ctx, dqkv, dw, s);
  }
};

struct SwigluFn : torch::autograd::Function<SwigluFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x) {
    BelowAutograd below;
    ctx->save_for_backward({x});
    return op_swiglu().call(x);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto s = ctx->get_saved_variables();
    if (traced(s[0])) return wanted(ctx, replay_swiglu().call(grads, s, 0.), 1);
    DetachedScope scope;
    return {op_swiglu_backward().call(grads[0], s[0])};
  }
};

struct GanmFn : torch::autograd::Function<GanmFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& z, const Tensor& a, const Tensor& gate,
                               const Tensor& weight, const Tensor& shift, const Tensor& scale, double eps) {
    BelowAutograd below;
    ctx->save_for_backward({z, a, gate, weight, shift, scale});
    ctx->saved_data["eps"] = eps;
    auto [d, y] = op_ganm().call(z, a, gate, weight, shift, scale, eps);
    return {d, y};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto s = ctx->get_saved_variables();
    if (traced(s[0])) return wanted(ctx, replay_ganm().call(grads, s, ctx->saved_data["eps"].toDouble()), 7);
    DetachedScope scope;
    auto [gz, ga, ggate, gw, gshift, gscale] =
        op_ganm_backward().call(grads[0], grads[1], s[0], s[1], s[2], s[3], s[5], ctx->saved_data["eps"].toDouble());
    variable_list out{gz, ga, ggate, as_dtype(gw, s[3].scalar_type()), gshift, gscale, Tensor()};
    for (size_t i = 0; i < 6; ++i)
      if (!ctx->needs_input_grad(i)) out[i] = Tensor();
    return out;
  }
};

struct GresFn : torch::autograd::Function<GresFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& d, const Tensor& gate, const Tensor& m) {
    BelowAutograd below;
    ctx->save_for_backward({gate, m});
    return op_gres().call(d, gate, m);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &gate = s[0], &m = s[1], &grad = grads[0];
    Tensor ggate, gm;
    const bool need_gate = ctx->needs_input_grad(1), need_m = ctx->needs_input_grad(2);
    if (need_gate || need_m) {
      if (!at::GradMode::is_enabled() && m.sym_size(2) <= kNormMaxChannels) {
        BelowAutograd below;
        std::tie(ggate, gm) = op_gres_backward().call(grad, gate, m);
      } else {  // a graph of the backward is built, or wider than the kernel's rows
        if (need_gate) ggate = as_dtype(at::sum(as_dtype(grad * m, at::kFloat), 1), gate.scalar_type());
        if (need_m) gm = grad * gate.unsqueeze(1);
      }
    }
    return {ctx->needs_input_grad(0) ? grad : Tensor(), need_gate ? ggate : Tensor(), need_m ? gm : Tensor()};
  }
};

// A linear layer whose weight and bias gradients come from one pass over the rows (linear_weight_grad).  The forward
// and the input's gradient are torch's own products.  Where a graph of the backward is built, or the kernel does not
// take the shapes, the weight's gradient is the product torch's linear has.
struct LinearFn : torch::autograd::Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const std::optional<Tensor>& bias) {
    BelowAutograd below;
    ctx->save_for_backward({x, weight});
    ctx->saved_data["bias"] = bias.has_value() && bias->defined();
    return at::linear(x, weight, bias);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &weight = saved[1], &g = grads[0];
    const bool need_w = ctx->needs_input_grad(1);
    const bool need_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
    Tensor gx, gw, gb;
    if (ctx->needs_input_grad(0)) gx = at::matmul(g, weight);
    if (need_w && !at::GradMode::is_enabled() && x.numel() > 0 && x.size(-1) % 8 == 0 && g.size(-1) % 8 == 0) {
      BelowAutograd below;
      std::tie(gw, gb) = op_linear_weight_grad().call(g, x, need_b);
      if (!need_b) gb = Tensor();
    } else if (need_w || need_b) {
      const Tensor g2 = g.reshape({-1, g.size(-1)});
      if (need_w) gw = g2.t().matmul(x.reshape({-1, x.size(-1)}));
      if (need_b) gb = g2.sum(0);
    }
    return {gx, gw, gb};
  }
};

// ---- autograd kernels: record a node, or go straight below autograd
Tensor read_autograd(const Tensor& x, const Tensor& w) {
  if (recording(x, w)) return ReadFn::apply(x, w);
  BelowAutograd below;
  return op_read().call(x, w);
}

Tensor write_autograd(const Tensor& z, const Tensor& w) {
  if (recording(z, w)) return WriteFn::apply(z, w);
  BelowAutograd below;
  return op_write().call(z, w);
}

Tensor write_add_autograd(const Tensor& z, const Tensor& w, const Tensor& x) {
  if (recording(z, w, x)) return WriteAddFn::apply(z, w, x);
  BelowAutograd below;
  return op_write_add().call(z, w, x);
}

Tensor final_list_autograd(const Tensor& x0, TensorList dzs, TensorList betas) {
  if (recording(x0, dzs, betas) && dzs.size() == betas.size()) return FinalListFn::apply(x0, dzs, betas);
  BelowAutograd below;
  return op_final_list().call(x0, dzs, betas);
}

Tensor final_12_autograd(const Tensor& x0, LTHC_T12(dz), LTHC_T12(beta)) {
  const std::array<Tensor, 12> dzs{LTHC_A12(dz)}, betas{LTHC_A12(beta)};
  if (recording(x0, TensorList(dzs), TensorList(betas))) return Final12Fn::apply(x0, TensorList(dzs), TensorList(betas));
  BelowAutograd below;
  return call_final_12(x0, dzs, betas);
}

Tensor recur_autograd(const Tensor& z, const Tensor& dz, const Tensor& gamma) {
  if (recording(z, dz, gamma)) return RecurFn::apply(z, dz, gamma);
  BelowAutograd below;
  return op_recur().call(z, dz, gamma);
}

Tensor gamma_rounded_autograd(const Tensor& alpha, TensorList betas, at::ScalarType dtype) {
  if (recording(alpha, betas)) return GammaRoundedFn::apply(alpha, betas, dtype);
  BelowAutograd below;
  return op_gamma_rounded().call(alpha, betas, dtype);
}

std::vector<Tensor> all_base_split_autograd(const Tensor& x0, const Tensor& alpha_stack) {
  if (recording(x0, alpha_stack)) return AllBaseSplitFn::apply(x0, alpha_stack);
  BelowAutograd below;
  return op_all_base_split().call(x0, alpha_stack);
}

Tensor tri12_record(const Tensor& base, TensorList dzs, const Tensor& gamma, int64_t active) {
  if (recording(base, dzs, gamma)) return Tri12Fn::apply(base, dzs, gamma, active);
  BelowAutograd below;
  return call_tri12(base, dzs, gamma, active);
}

template <int ACTIVE>
Tensor tri12_autograd(const Tensor& base, LTHC_T12(dz), const Tensor& gamma) {
  const std::array<Tensor, 12> dzs{LTHC_A12(dz)};
  return tri12_record(base, dzs, gamma, ACTIVE);
}

Tensor tri12_active_autograd(const Tensor& base, LTHC_T12(dz), const Tensor& gamma, int64_t active) {
  const std::array<Tensor, 12> dzs{LTHC_A12(dz)};
  return tri12_record(base, dzs, gamma, check_active(active));
}

Tensor tri_list_autograd(const Tensor& base, TensorList dzs, const Tensor& gamma) {
  if (recording(base, dzs, gamma)) return TriListFn::apply(base, dzs, gamma);
  BelowAutograd below;
  return op_tri_list().call(base, dzs, gamma);
}

std::tuple<Tensor, Tensor> pair(const variable_list& v) { return {v[0], v[1]}; }

std::tuple<Tensor, Tensor> norm_autograd(const Tensor& x, const Tensor& w, const Tensor& shift, const Tensor& scale,
                                         double eps) {
  if (recording(x, w, shift, scale)) return pair(NormFn::apply(x, w, shift, scale, eps));
  BelowAutograd below;
  return op_norm().call(x, w, shift, scale, eps);
}

std::tuple<Tensor, Tensor> qk_autograd(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos,
                                       const Tensor& sin, double eps) {
  if (recording(qkv, qw, kw, cos, sin)) return pair(QkFn::apply(qkv, qw, kw, cos, sin, eps));
  BelowAutograd below;
  return op_qk().call(qkv, qw, kw, cos, sin, eps);
}

Tensor attention_autograd(const Tensor& qkv, const Tensor& qw, const Tensor& kw, const Tensor& cos, const Tensor& sin,
                          double eps) {
  if (recording(qkv, qw, kw, cos, sin)) return AttentionFn::apply(qkv, qw, kw, cos, sin, eps);
  BelowAutograd below;
  return op_attention().call(qkv, qw, kw, cos, sin, eps);
}

Tensor swiglu_autograd(const Tensor& x) {
  if (recording(x)) return SwigluFn::apply(x);
  BelowAutograd below;
  return op_swiglu().call(x);
}

std::tuple<Tensor, Tensor> ganm_autograd(const Tensor& z, const Tensor& a, const Tensor& gate, const Tensor& w,
                                         const Tensor& shift, const Tensor& scale, double eps) {
  if (recording(z, a, gate, w, shift, scale)) return pair(GanmFn::apply(z, a, gate, w, shift, scale, eps));
  BelowAutograd below;
  return op_ganm().call(z, a, gate, w, shift, scale, eps);
}

Tensor gres_autograd(const Tensor& d, const Tensor& gate, const Tensor& m) {
  if (recording(d, gate, m)) return GresFn::apply(d, gate, m);
  BelowAutograd below;
  return op_gres().call(d, gate, m);
}

// Composite ops: they only open an autograd node around registered ops.
std::tuple<Tensor, Tensor> read_with_residual(const Tensor& x, const Tensor& weight) {
  return pair(OpenFn::apply(x, weight));
}

Tensor linear(const Tensor& x, const Tensor& weight, const std::optional<Tensor>& bias) {
  if (!at::autocast::is_autocast_enabled(at::kCUDA)) return LinearFn::apply(x, weight, bias);
  // autocast's own conversion, which keeps a parameter's copy for the later calls of the region
  const auto cast = [dt = at::autocast::get_autocast_dtype(at::kCUDA)](const Tensor& t) {
    return at::autocast::cached_cast(dt, t, at::kCUDA);
  };
  std::optional<Tensor> b = bias;
  if (b.has_value() && b->defined()) b = cast(*b);
  return LinearFn::apply(cast(x), cast(weight), b);
}

std::vector<Tensor> lazy_workspace_step(const Tensor& z, const Tensor& dz, const Tensor& gamma, bool split) {
  return StepFn::apply(z, dz, gamma, split);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(jit_thc, m) {
  m.def("read_with_residual(Tensor x, Tensor weight) -> (Tensor, Tensor)", read_with_residual);
  m.def("linear(Tensor x, Tensor weight, Tensor? bias) -> Tensor", linear);
  m.def("lazy_workspace_step(Tensor z, Tensor dz, Tensor gamma, bool split) -> Tensor[]", lazy_workspace_step);
}

#define LTHC_TRI_ACTIVE(m, fn)                                  \
  m.impl("triangular_accumulate_b4_12_ptr_active1", fn<1>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active2", fn<2>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active3", fn<3>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active4", fn<4>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active5", fn<5>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active6", fn<6>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active7", fn<7>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active8", fn<8>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active9", fn<9>);     \
  m.impl("triangular_accumulate_b4_12_ptr_active10", fn<10>);   \
  m.impl("triangular_accumulate_b4_12_ptr_active11", fn<11>);   \
  m.impl("triangular_accumulate_b4_12_ptr_traceable", fn<12>)

TORCH_LIBRARY_IMPL(jit_thc, CUDA, m) {
  m.impl("local_write_traceable", read_cuda);
  m.impl("local_read_traceable", write_cuda);
  m.impl("local_read_add_traceable", write_add_cuda);
  m.impl("local_weight_grad_traceable", weight_grad_cuda);
  m.impl("final_accumulate_list", final_list_cuda);
  m.impl("final_accumulate_b4_12_traceable", final_12_cuda);
  m.impl("final_accumulate_backward", final_backward_cuda);
  m.impl("lazy_workspace_update", recur_cuda);
  m.impl("lazy_workspace_update_backward", recur_backward_cuda);
  m.impl("lazy_workspace_update_backward_sum", recur_backward_sum_cuda);
  m.impl("lazy_gamma_stack", gamma_stack_cuda);
  m.impl("lazy_gamma_rounded", gamma_rounded_cuda);
  m.impl("lazy_gamma_rounded_backward", gamma_rounded_backward_cuda);
  m.impl("all_base_b4_12_split_traceable", all_base_split_cuda);
  m.impl("all_base_backward", all_base_backward_cuda);
  m.impl("triangular_accumulate_list", tri_list_cuda);
  m.impl("triangular_accumulate_b4_12_ptr_active", tri12_active_cuda);
  LTHC_TRI_ACTIVE(m, tri12_cuda);
  m.impl("ws_accumulate_backward", ws_backward_cuda);
  m.impl("norm_modulate", norm_modulate_cuda);
  m.impl("norm_modulate_backward", norm_modulate_backward_cuda);
  m.impl("qk_norm_rope", qk_norm_rope_cuda);
  m.impl("qk_norm_rope_backward", qk_norm_rope_backward_cuda);
  m.impl("qk_norm_rope_attention", attention_cuda);
  m.impl("qk_norm_rope_attention_backward", attention_backward_cuda);
  m.impl("swiglu", swiglu_cuda);
  m.impl("swiglu_backward", swiglu_backward_cuda);
  m.impl("gate_add_norm_modulate", gate_add_norm_modulate_cuda);
  m.impl("gate_add_norm_modulate_backward", gate_add_norm_modulate_backward_cuda);
  m.impl("gate_residual", gate_residual_cuda);
  m.impl("gate_residual_backward", gate_residual_backward_cuda);
  m.impl("linear_weight_grad", linear_weight_grad_cuda);
  m.impl("block_tail", block_tail_cuda);
}

// The nodes hold no device code: meta tensors, fake ones of any device and CPU tensors (whose kernels refuse them, or are
// registered by a program) get the same formulas.
static void autograd_kernels(torch::Library& m) {
  m.impl("local_write_traceable", read_autograd);
  m.impl("local_read_traceable", write_autograd);
  m.impl("local_read_add_traceable", write_add_autograd);
  m.impl("final_accumulate_list", final_list_autograd);
  m.impl("final_accumulate_b4_12_traceable", final_12_autograd);
  m.impl("lazy_workspace_update", recur_autograd);
  m.impl("lazy_gamma_rounded", gamma_rounded_autograd);
  m.impl("all_base_b4_12_split_traceable", all_base_split_autograd);
  m.impl("triangular_accumulate_list", tri_list_autograd);
  m.impl("triangular_accumulate_b4_12_ptr_active", tri12_active_autograd);
  LTHC_TRI_ACTIVE(m, tri12_autograd);
  m.impl("norm_modulate", norm_autograd);
  m.impl("qk_norm_rope", qk_autograd);
  m.impl("qk_norm_rope_attention", attention_autograd);
  m.impl("swiglu", swiglu_autograd);
  m.impl("gate_add_norm_modulate", ganm_autograd);
  m.impl("gate_residual", gres_autograd);
}

TORCH_LIBRARY_IMPL(jit_thc, AutogradCUDA, m) { autograd_kernels(m); }
TORCH_LIBRARY_IMPL(jit_thc, AutogradMeta, m) { autograd_kernels(m); }
TORCH_LIBRARY_IMPL(jit_thc, AutogradCPU, m) { autograd_kernels(m); }
