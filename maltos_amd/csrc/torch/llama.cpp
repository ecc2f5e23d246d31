// The projections, the MLP and the rotary + attention block of maltos_amd/llama.py as C++ autograd nodes, and the record of
// which parameters' gradients a backward pass has written.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <numeric>
#include <unordered_map>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include "common.hpp"

namespace maltos {
namespace {

using torch::autograd::collect_next_edges;
using torch::autograd::compute_requires_grad;
using torch::autograd::set_history;

// ---- which parameters received a gradient -------------------------------------------------------------------------------
// Backward formulas that add into a bound `.grad` return no gradient to autograd, so an optimizer that skips parameters
// without a gradient has to be told another way: a GradMarks holds one flag per parameter it was made for, and listeners
// collect the parameters themselves.  Set from autograd's device thread without the interpreter lock.
struct GradMarks;
std::mutex& marks_mutex = *new std::mutex;  // (never destroyed, like the two below: marks may be released at exit)
auto& marks_by_param = *new std::unordered_map<const c10::TensorImpl*, std::vector<std::pair<GradMarks*, size_t>>>;
auto& listeners = *new std::vector<std::vector<Tensor>*>;

struct GradMarks {
  std::vector<Tensor> params;  // kept alive: their addresses are the keys
  std::vector<uint8_t> written;

  explicit GradMarks(std::vector<Tensor> ps) : params(std::move(ps)), written(params.size(), 0) {
    std::lock_guard<std::mutex> lock(marks_mutex);
    for (size_t i = 0; i < params.size(); ++i) marks_by_param[params[i].unsafeGetTensorImpl()].emplace_back(this, i);
  }
  GradMarks(const GradMarks&) = delete;
  ~GradMarks() {
    std::lock_guard<std::mutex> lock(marks_mutex);
    for (const Tensor& p : params) {
      auto it = marks_by_param.find(p.unsafeGetTensorImpl());
      if (it == marks_by_param.end()) continue;
      auto& v = it->second;
      v.erase(std::remove_if(v.begin(), v.end(), [this](const auto& e) { return e.first == this; }), v.end());
      if (v.empty()) marks_by_param.erase(it);
    }
  }
  std::vector<bool> list() const {
    std::lock_guard<std::mutex> lock(marks_mutex);
    return std::vector<bool>(written.begin(), written.end());
  }
  bool all() const {
    std::lock_guard<std::mutex> lock(marks_mutex);
    return std::find(written.begin(), written.end(), 0) == written.end();
  }
  void fill(bool value) {
    std::lock_guard<std::mutex> lock(marks_mutex);
    std::fill(written.begin(), written.end(), value);
  }
};

}  // namespace

void notify_grad_written(const Tensor& param) {
  std::lock_guard<std::mutex> lock(marks_mutex);
  auto it = marks_by_param.find(param.unsafeGetTensorImpl());
  if (it != marks_by_param.end())
    for (auto& [marks, i] : it->second) marks->written[i] = 1;
  for (std::vector<Tensor>* seen : listeners) seen->push_back(param);
}

namespace {

struct GradListener {
  std::vector<Tensor> seen;
  bool active = false;
  void start() {
    std::lock_guard<std::mutex> lock(marks_mutex);
    if (!active) listeners.push_back(&seen);
    active = true;
  }
  std::vector<Tensor> stop() {
    std::lock_guard<std::mutex> lock(marks_mutex);
    listeners.erase(std::remove(listeners.begin(), listeners.end(), &seen), listeners.end());
    active = false;
    return seen;
  }
  GradListener() = default;
  GradListener(const GradListener&) = delete;
  ~GradListener() { stop(); }
};

// ---- parameters that share one flat buffer --------------------------------------------------------------------------------
// Whether every parameter's `.grad` (or the parameter itself) still is the view of `flat` at its offset: what the flat
// optimizer layouts ask several times a step, for every parameter of the model.
struct FlatViews {
  std::vector<Tensor> params;
  std::vector<int64_t> offsets;
  FlatViews(std::vector<Tensor> ps, std::vector<int64_t> offs) : params(std::move(ps)), offsets(std::move(offs)) {}
  bool grads_are_views_of(const Tensor& flat) const {
    const char* base = static_cast<const char*>(flat.const_data_ptr());
    const int64_t size = flat.element_size();
    for (size_t i = 0; i < params.size(); ++i) {
      const Tensor& g = params[i].grad();
      if (!g.defined() || g.scalar_type() != flat.scalar_type() || !g.is_contiguous() || g.const_data_ptr() != base + offsets[i] * size) return false;
    }
    return true;
  }
  bool grads_defined() const {
    for (const Tensor& p : params)
      if (!p.grad().defined()) return false;
    return true;
  }
};

// ---- products -------------------------------------------------------------------------------------------------------------
Tensor rows2d(const Tensor& t) { return t.dim() == 2 ? t : t.reshape({-1, t.size(-1)}); }

// dW = dy2^T x2 for [rows, out] / [rows, in] operands, large ones as a batch of row-slice products where that fills the chip
// better.  With `grad` (the gradient buffer the weight already owns, a view of a flat gradient buffer) dW is added into it in
// the pass that finishes it and nothing is returned.
Tensor weight_grad(const Tensor& x2, const Tensor& dy2, const Tensor& grad) {
  const int64_t splits = weight_grad_splits(x2.size(0), dy2.size(1), x2.size(1));
  if (splits > 1 && x2.is_contiguous() && dy2.is_contiguous() && !own_product(MLTS_GEMM_TN, dy2, x2)) {
    const int64_t rows = x2.size(0) / splits;
    Tensor part = at::bmm(dy2.view({splits, rows, dy2.size(1)}).transpose(1, 2), x2.view({splits, rows, x2.size(1)}));
    Tensor dw = grad_sum_slices(part, grad.defined() ? OptTensor(grad) : std::nullopt, grad.defined());  // fp32 sum, rounded once
    return grad.defined() ? Tensor() : dw;
  }
  Tensor dw = product(MLTS_GEMM_TN, dy2, x2, grad, grad.defined());
  return grad.defined() ? Tensor() : dw;
}

Tensor project(const Tensor& x, const Tensor& weight) {
  if (x.dim() == 2 && x.is_contiguous()) return product(MLTS_GEMM_NT, x, weight);
  if (!x.is_contiguous()) return at::linear(x, weight);
  c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = weight.size(0);
  return product(MLTS_GEMM_NT, rows2d(x), weight).view(shape);
}

// dx = dy2 w and dw = dy2^T x2 (added into `grad` if that is defined, and then not returned), those of them that are needed: in one
// launch where both run on the own kernels, as neither fills the chip at the sizes they are used for
std::pair<Tensor, Tensor> input_and_weight_grad(const Tensor& dy2, const Tensor& w, const Tensor& x2, const Tensor& grad, bool need_dx, bool need_dw) {
  if (!need_dx || !need_dw) return {need_dx ? product(MLTS_GEMM_NN, dy2, w) : Tensor(), need_dw ? weight_grad(x2, dy2, grad) : Tensor()};
  if (own_product(MLTS_GEMM_NN, dy2, w, Use::WITH_WEIGHT_GRAD) && own_product(MLTS_GEMM_TN, dy2, x2, Use::WITH_WEIGHT_GRAD) && (!grad.defined() || own_output(grad, x2))) {
    Tensor dx = at::empty({dy2.size(0), w.size(1)}, dy2.options());
    Tensor dw = grad.defined() ? grad : at::empty(w.sizes(), dy2.options());
    ProductList list;
    list.add(MLTS_GEMM_TN, dy2, x2, dw, grad.defined());  // the longer contraction first
    list.add(MLTS_GEMM_NN, dy2, w, dx, false);
    list.run();
    return {dx, grad.defined() ? Tensor() : dw};
  }
  Tensor dx = product(MLTS_GEMM_NN, dy2, w);
  return {dx, weight_grad(x2, dy2, grad)};
}

struct LinearBackward final : Formula {
  enum { X, W, COUNT };
  bool into_grad = false;
  LinearBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosLinearBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    const Tensor &x = s[X], &w = s[W], &dy = g[0];
    if (!dy.defined()) return {Tensor(), Tensor()};
    const bool need_dx = task_should_compute_output(0), need_dw = task_should_compute_output(1);
    const Tensor grad = need_dw ? bound_grad(w, into_grad) : Tensor();
    auto [dx, dw] = input_and_weight_grad(rows2d(dy), w, rows2d(x), grad, need_dx, need_dw);
    if (grad.defined()) notify_grad_written(w);  // autograd's hooks on the weight see no gradient for what was added here
    return {need_dx ? dx.view(x.sizes()) : dx, dw};
  }
  variable_list recorded_backward(variable_list&& g, const std::vector<Tensor>& s) override {
    const Tensor &x = s[X], &w = s[W], &dy = g[0];
    if (!dy.defined()) return {Tensor(), Tensor()};
    return {task_should_compute_output(0) ? at::matmul(dy, w) : Tensor(),
            task_should_compute_output(1) ? at::mm(rows2d(dy).t(), rows2d(x)) : Tensor()};
  }
};

// What the nodes below know nothing of (tangents, tensors of function transforms and other subclasses) is left to torch's operators
bool ordinary(const Tensor& t) { return !has_tangent(t) && !at::isTensorSubclassLike(t); }

Tensor linear(const Tensor& x, const Tensor& weight, bool into_grad) {
  if (!ordinary(x) || !ordinary(weight) || weight.dim() != 2) return at::linear(x, weight);
  std::shared_ptr<LinearBackward> fn;
  if (compute_requires_grad(x, weight)) {
    fn = make_formula<LinearBackward>();
    fn->set_next_edges(collect_next_edges(x, weight));
    fn->save(fn->X, x), fn->save(fn->W, weight);
    fn->into_grad = into_grad;
  }
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    y = project(x, weight);
  }
  if (fn) set_history(y, fn);
  return y;
}

// ---- token embedding --------------------------------------------------------------------------------------------------------
struct EmbeddingBackward final : Formula {
  enum { IDS, W, COUNT };
  bool into_grad = false;
  EmbeddingBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosEmbeddingBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return {Tensor()};
    const Tensor &w = s[W], ids = dense(s[IDS].scalar_type() == at::kLong ? s[IDS] : s[IDS].to(at::kLong)), dy = dense(g[0]);
    const int64_t n = ids.numel(), vocab = w.size(0), hidden = w.size(1);
    const Tensor grad = bound_grad(w, into_grad);
    if ((w.scalar_type() != at::kBFloat16 && w.scalar_type() != at::kFloat) || dy.scalar_type() != w.scalar_type() ||
        mlts_embedding_bwd_supports(n, hidden, vocab, dtype_code(w)) != nullptr || !aligned(dy) || (grad.defined() && !aligned(grad)))
      return {at::embedding_dense_backward(dy, ids, vocab, -1, false)};
    Tensor dw = grad.defined() ? grad : at::zeros({vocab, hidden}, w.options());
    check(mlts_embedding_bwd(ids.const_data_ptr<int64_t>(), ptr(dy), mptr(dw), n, hidden, vocab, dtype_code(w), current_stream()));
    if (!grad.defined()) return {dw};
    notify_grad_written(w);
    return {Tensor()};
  }
  variable_list recorded_backward(variable_list&& g, const std::vector<Tensor>& s) override {
    return {g[0].defined() ? at::embedding_dense_backward(g[0], s[IDS], s[W].size(0), -1, false) : Tensor()};
  }
};

Tensor embedding(const Tensor& weight, const Tensor& ids, bool into_grad) {
  if (!ordinary(weight) || !ordinary(ids)) return at::embedding(weight, ids);
  std::shared_ptr<EmbeddingBackward> fn;
  if (compute_requires_grad(weight)) {
    fn = make_formula<EmbeddingBackward>();
    fn->set_next_edges(collect_next_edges(weight));
    fn->save(fn->IDS, ids), fn->save(fn->W, weight);
    fn->into_grad = into_grad;
  }
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    y = at::embedding(weight, ids);
  }
  if (fn) set_history(y, fn);
  return y;
}

// ---- projections that share their input, run as ONE product over adjacent weights -----------------------------------------
// q_proj / k_proj / v_proj (and gate_proj / up_proj) read the same activations.  When their weights are adjacent row blocks
// of one allocation (what the flat optimizer layouts make of them), they ARE one [sum of out_features, in_features] matrix,
// and the three (two) products are one: at LLaMA-50M sizes a 512-wide product has 128 output tiles for 256 compute units,
// the 1536-wide one fills the chip, and the backward's three input-gradient products and their two additions become one.
// Parameters that are not adjacent still share their input: at sizes where the products run on the own kernels, all of a pass are
// one launch, and the outputs are column ranges of one buffer as above (`rows` then has no `weight`).
struct Adjacent {
  Tensor weight;                     // [R, in]; undefined: the parameters are not adjacent
  Tensor grad;                       // their gradients as one matrix like `weight`, when those are adjacent in the same order
  std::vector<int64_t> first;        // output column of parameter i's first row
  std::vector<size_t> order;         // parameters by output column
  int64_t width = 0;                 // their rows together
  bool similar = false;              // not adjacent, but of one input width and type: may run as a group
  // of a parameter: its address and that of its gradient, whether it is trained, its shape and type (another one may come to lie at an
  // address that was given back)
  typedef std::tuple<const void*, const void*, bool, int64_t, int64_t, c10::ScalarType> Key;
  std::vector<Key> key;  // what this was made for

  explicit Adjacent(const std::vector<Tensor>& params) {
    for (const Tensor& p : params) key.push_back(key_of(p));
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    const Tensor& p0 = params[0];
    for (const Tensor& p : params)
      if (p.dim() != 2 || !p.is_cuda() || !p.is_contiguous() || p.scalar_type() != p0.scalar_type() || p.size(1) != p0.size(1)) return;
    order.resize(params.size());
    first.resize(params.size());
    std::iota(order.begin(), order.end(), size_t{0});
    for (size_t i = 0; i < params.size(); ++i) first[i] = width, width += params[i].size(0);
    similar = params.size() <= 3;
    for (const Tensor& p : params)
      if (!p.requires_grad()) return;
    std::vector<size_t> in_order = order;
    std::sort(in_order.begin(), in_order.end(), [&](size_t i, size_t j) { return address(i) < address(j); });
    std::vector<int64_t> at(params.size());
    int64_t rows = 0;
    const char* next = static_cast<const char*>(address(in_order[0]));
    for (size_t i : in_order) {
      if (address(i) != next || !params[i].storage().is_alias_of(p0.storage())) return;
      at[i] = rows;
      rows += params[i].size(0);
      next += params[i].nbytes();
    }
    order = in_order, first = at;
    const Tensor& base = params[order[0]];
    weight = base.as_strided({rows, base.size(1)}, {base.size(1), 1}, base.storage_offset());
    const Tensor g0 = params[order[0]].grad();
    next = nullptr;
    for (size_t i : order) {
      const Tensor& g = params[i].grad();
      if (!g.defined() || !g.is_contiguous() || g.scalar_type() != p0.scalar_type() || g.sizes() != params[i].sizes() ||
          (next && std::get<1>(key[i]) != next) || !g.storage().is_alias_of(g0.storage()))
        return;
      next = static_cast<const char*>(std::get<1>(key[i])) + g.nbytes();
    }
    grad = g0.as_strided(weight.sizes(), weight.strides(), g0.storage_offset());
  }
  const void* address(size_t i) const { return std::get<0>(key[i]); }
  static Key key_of(const Tensor& p) {
    const Tensor& g = p.grad();
    return {p.const_data_ptr(), g.defined() ? g.const_data_ptr() : nullptr, p.requires_grad(), p.dim() == 2 ? p.size(0) : -1, p.numel(), p.scalar_type()};
  }
  bool made_for(const std::vector<Tensor>& params) const {
    if (params.size() != key.size()) return false;
    for (size_t i = 0; i < params.size(); ++i)
      if (key_of(params[i]) != key[i]) return false;
    return true;
  }
};
using AdjacentPtr = std::shared_ptr<Adjacent>;

// the [rows, sum of widths] matrix whose column ranges the given [..., width_i] tensors are, in this order, when they are
// such views of one dense buffer; undefined otherwise (then the caller copies them together)
Tensor adjacent_columns(const std::vector<Tensor>& parts, const std::vector<size_t>& order) {
  const Tensor& first = parts[order[0]];
  const int64_t dims = first.dim();
  int64_t total = 0;
  for (size_t i : order) total += parts[i].size(-1);
  int64_t offset = first.storage_offset();
  for (size_t i : order) {
    const Tensor& p = parts[i];
    if (p.dim() != dims || p.scalar_type() != first.scalar_type() || !p.storage().is_alias_of(first.storage()) || p.storage_offset() != offset ||
        (p.size(-1) > 1 && p.stride(-1) != 1))
      return Tensor();
    int64_t step = total;
    for (int64_t d = dims - 2; d >= 0; --d) {
      if (p.size(d) != first.size(d) || (p.size(d) > 1 && p.stride(d) != step)) return Tensor();
      step *= p.size(d);
    }
    offset += p.size(-1);
  }
  const int64_t rows = first.numel() / first.size(-1);
  return first.as_strided({rows, total}, {total, 1}, first.storage_offset());
}

// whether the products with these parameters, not adjacent, run as one launch
bool runs_as_group(const Adjacent& a, const Tensor& x, const std::vector<Tensor>& weights) {
  if (!a.similar || a.weight.defined() || !x.is_cuda() || !x.is_contiguous() || x.dim() < 2 || x.numel() == 0) return false;
  const Tensor x2 = rows2d(x);
  for (size_t i = 0; i < weights.size(); ++i)
    if (a.first[i] * x.element_size() % 16 || weights[i].size(1) != x.size(-1) || !own_product(MLTS_GEMM_NT, x2, weights[i])) return false;
  return a.width * x.element_size() % 16 == 0;
}

// x times all of the parameters, transposed: their outputs side by side
Tensor project_all(const Tensor& x, const Adjacent& rows, const std::vector<Tensor>& weights) {
  if (rows.weight.defined()) return project(x, rows.weight);
  c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = rows.width;
  Tensor y = at::empty(shape, x.options());
  const Tensor x2 = rows2d(x), y2 = rows2d(y);
  ProductList list;
  for (size_t i = 0; i < weights.size(); ++i) list.add(MLTS_GEMM_NT, x2, weights[i], y2.narrow(1, rows.first[i], weights[i].size(0)), false);
  list.run();
  return y;
}

// gate and up of an MLP side by side (undefined if nobody keeps them), and round(silu(gate)) * up: in one launch where the products run
// on the own kernels: the pass over gate and up costs a launch in small calls and a read of both in large ones.
std::pair<Tensor, Tensor> gate_up_activation(const Tensor& x, const Adjacent& rows, const std::vector<Tensor>& weights, bool keep) {
  const Tensor &wg = weights[0], &wu = weights[1], x2 = rows2d(x);
  const int64_t cols = wg.size(0), es = x.element_size();
  const Use use = keep ? Use::GATE_AND_UP : Use::ACTIVATION;
  if (x.is_contiguous() && wu.sizes() == wg.sizes() && wu.stride(0) == wg.stride(0) && own_product(MLTS_GEMM_NT, x2, rows.weight.defined() ? rows.weight : wg, use) &&
      own_product(MLTS_GEMM_NT, x2, wg, use) && own_product(MLTS_GEMM_NT, x2, wu, use) && (rows.first[0] * es) % 16 == 0 && (rows.first[1] * es) % 16 == 0 &&
      mlts_gemm_swiglu_supports(dtype_code(x), x2.size(0), cols, x2.size(1), x2.stride(0), wg.stride(0), rows.width, cols) == nullptr) {
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = cols;
    const Tensor h = at::empty(shape, x.options());
    Tensor gu;
    char *gate = nullptr, *up = nullptr;
    if (keep) {
      shape.back() = rows.width;
      gu = at::empty(shape, x.options());
      gate = static_cast<char*>(mptr(gu)) + rows.first[0] * es, up = static_cast<char*>(mptr(gu)) + rows.first[1] * es;
    }
    check(mlts_gemm_swiglu(dtype_code(x), x2.size(0), cols, x2.size(1), ptr(x2), x2.stride(0), ptr(wg), ptr(wu), wg.stride(0), gate, up, rows.width, mptr(h),
                           cols, current_stream()));
    return {gu, h};
  }
  const Tensor gu = project_all(x, rows, weights);
  return {gu, swiglu_rows(gu, rows.first[0], rows.first[1], cols)};
}

// whether two dense buffers share memory (the gradient of a parameter that is used twice)
bool share_memory(const Tensor& a, const Tensor& b) {
  if (!a.defined() || !b.defined()) return false;
  const char *pa = static_cast<const char*>(a.const_data_ptr()), *pb = static_cast<const char*>(b.const_data_ptr());
  return pa < pb + b.nbytes() && pb < pa + a.nbytes();
}

// Which gradients a pass asks for: of the input, of the weights that read it (frozen ones are not asked for)
struct Needed {
  bool input = false, any_weight = false, all_weights = true;
  std::vector<bool> weight;
};

// M * N * K of each part up to which the input gradient of weights that are not adjacent is one contraction in parts: it runs on the small
// tiles only, and beyond them the products and their sum one after the other are as fast
constexpr double kOwnLimitParts = 4.0e9;

// The input gradient, then one gradient per parameter, as far as they are needed: added into the gradient buffers where into_grad
// allows it, and then undefined.  dy2: the outputs' gradients side by side.
variable_list grads_of_all(const Adjacent& a, const std::vector<Tensor>& weights, bool into_grad, const Needed& need, const Tensor& x, const Tensor& dy2) {
  variable_list out(1 + weights.size());
  const Tensor x2 = rows2d(x);
  const bool one_matrix = a.weight.defined();
  if (one_matrix && (need.all_weights || !need.any_weight)) {
    const Tensor grad = need.any_weight && into_grad && !at::GradMode::is_enabled() ? a.grad : Tensor();
    Tensor dw;
    std::tie(out[0], dw) = input_and_weight_grad(dy2, a.weight, x2, grad, need.input, need.any_weight);
    for (size_t i = 0; i < weights.size(); ++i) {
      if (grad.defined()) notify_grad_written(weights[i]);
      else if (dw.defined()) out[1 + i] = dw.narrow(0, a.first[i], weights[i].size(0));
    }
  } else {
    std::vector<Tensor> parts, into;
    bool own = !one_matrix;
    for (size_t i = 0; i < weights.size(); ++i) {
      parts.push_back(dy2.narrow(1, a.first[i], weights[i].size(0)));
      into.push_back(need.weight[i] ? bound_grad(weights[i], into_grad) : Tensor());
      own = own && own_product(MLTS_GEMM_NN, parts[i], weights[i]) && own_product(MLTS_GEMM_TN, parts[i], x2) &&
            static_cast<double>(x2.numel()) * weights[i].size(0) <= kOwnLimitParts && (!into[i].defined() || own_output(into[i], x2));
    }
    if (own) {
      ProductList list;
      for (size_t i = 0; i < weights.size(); ++i) {
        if (!need.weight[i]) continue;
        Tensor dw = into[i].defined() ? into[i] : at::empty(weights[i].sizes(), dy2.options());
        // two projections with one weight add into the same buffer: one launch after the other
        if (std::any_of(into.begin(), into.begin() + i, [&](const Tensor& before) { return share_memory(before, into[i]); })) list.run(), list = {};
        list.add(MLTS_GEMM_TN, parts[i], x2, dw, into[i].defined());
        if (!into[i].defined()) out[1 + i] = dw;
      }
      if (need.input) {
        out[0] = at::empty(x2.sizes(), dy2.options());
        for (size_t i = weights.size(); i-- > 0;) {  // last one first: the order in which autograd adds them up
          if (i + 1 == weights.size()) list.add(MLTS_GEMM_NN, parts[i], weights[i], out[0], false);
          else list.add_segment(parts[i], weights[i]);
        }
      }
      if (list.count) list.run();
    } else {
      if (need.input && one_matrix) out[0] = product(MLTS_GEMM_NN, dy2, a.weight);
      for (size_t i = weights.size(); i-- > 0;) {
        if (need.input && !one_matrix) {
          Tensor dx = product(MLTS_GEMM_NN, parts[i], weights[i]);
          out[0] = out[0].defined() ? out[0].add_(dx) : dx;
        }
        if (need.weight[i]) out[1 + i] = weight_grad(x2, parts[i], into[i]);
      }
    }
    for (size_t i = 0; i < weights.size(); ++i)
      if (into[i].defined()) notify_grad_written(weights[i]);
  }
  if (out[0].defined()) out[0] = out[0].view(x.sizes());
  return out;
}

// A formula whose first outputs are the gradients of the shared input and of the weights that read it
struct SharedInputFormula : public Formula {
  AdjacentPtr rows;
  bool into_grad = false;
  std::vector<Tensor> weights;
  std::vector<int64_t> versions;  // of the weights as the forward pass read them
  using Formula::Formula;
  Needed needed() const {
    for (size_t i = 0; i < versions.size(); ++i)
      TORCH_CHECK(weights[i]._version() == versions[i], name(), ": a weight of shape ", weights[i].sizes(),
                  " needed for gradient computation has been modified by an inplace operation: it is at version ", weights[i]._version(),
                  "; expected version ", versions[i], " instead");
    Needed n;
    n.input = task_should_compute_output(0);
    for (size_t i = 0; i < weights.size(); ++i) {
      n.weight.push_back(task_should_compute_output(1 + i));
      n.any_weight = n.any_weight || n.weight[i], n.all_weights = n.all_weights && n.weight[i];
    }
    return n;
  }
};

struct AdjacentLinearsBackward final : SharedInputFormula {
  enum { X, COUNT };
  AdjacentLinearsBackward() : SharedInputFormula(COUNT) {}
  std::string name() const override { return "MaltosAdjacentLinearsBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    bool all = true, any = false;
    for (const Tensor& dy : g) all = all && dy.defined(), any = any || dy.defined();
    variable_list out(1 + weights.size());
    if (!any) return out;
    Tensor dy2;
    if (all) {
      dy2 = adjacent_columns(g, rows->order);  // already side by side (attention's joint gradient buffer)?
      if (!dy2.defined()) {
        std::vector<Tensor> parts;
        for (size_t i : rows->order) parts.push_back(g[i].reshape({-1, g[i].size(-1)}));
        // one launch, through the Python function so that whoever counts the copies of a step sees this one
        pybind11::gil_scoped_acquire gil;
        dy2 = pybind11::module_::import("torch").attr("cat")(parts, 1).cast<Tensor>();
      }
    } else {
      dy2 = at::empty({rows2d(s[X]).size(0), rows->width}, s[X].options());
      for (size_t i = 0; i < weights.size(); ++i) {
        Tensor part = dy2.narrow(1, rows->first[i], weights[i].size(0));
        if (g[i].defined()) part.copy_(g[i].reshape({-1, g[i].size(-1)}));
        else part.zero_();
      }
    }
    return grads_of_all(*rows, weights, into_grad, needed(), s[X], dy2);
  }
};

// the nodes of several projections have no counterpart in torch to fall back to
void refuse_function_transforms(const char* what, const Tensor& x, const std::vector<Tensor>& weights = {}) {
  bool any = of_transform(x);
  refuse_tangents(what, x);
  for (const Tensor& w : weights) refuse_tangents(what, w), any = any || of_transform(w);
  TORCH_CHECK_NOT_IMPLEMENTED(!any, what, ": maltos_amd has no rule of this operator for function transforms");
}

bool any_requires_grad(const std::vector<Tensor>& ts) {
  return std::any_of(ts.begin(), ts.end(), [](const Tensor& t) { return t.requires_grad(); });
}

template <typename F>
std::shared_ptr<F> adjacent_formula(const Tensor& x, const AdjacentPtr& rows, const std::vector<Tensor>& weights, bool into_grad) {
  auto fn = make_formula<F>();
  torch::autograd::edge_list edges = collect_next_edges(x);
  for (const Tensor& w : weights) edges.push_back(torch::autograd::impl::gradient_edge(w));
  fn->set_next_edges(std::move(edges));
  fn->save(fn->X, x);
  fn->rows = rows, fn->weights = weights, fn->into_grad = into_grad;
  // (adjacent parameters are views that flat optimizer layouts write to as one buffer: their versions say nothing)
  if (!rows->weight.defined())
    for (const Tensor& w : weights) fn->versions.push_back(w._version());
  return fn;
}

// (x W_0^T, x W_1^T, ...) as column slices of one buffer: one product with the parameters' common matrix, or their group
std::vector<Tensor> adjacent_linears(const Tensor& x, const AdjacentPtr& rows, const std::vector<Tensor>& weights, bool into_grad) {
  refuse_function_transforms("adjacent_linears", x, weights);
  std::vector<Tensor> out(weights.size());
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    const Tensor y = project_all(x, *rows, weights);
    for (size_t i = 0; i < weights.size(); ++i) out[i] = y.narrow(-1, rows->first[i], weights[i].size(0));
  }
  if (at::GradMode::is_enabled() && (compute_requires_grad(x) || any_requires_grad(weights))) {
    const auto fn = adjacent_formula<AdjacentLinearsBackward>(x, rows, weights, into_grad);
    for (const Tensor& o : out) set_history(o, fn);
  }
  return out;
}

// round(silu(x W_gate^T)) * (x W_up^T) (models/llama.py:205-206) with the two projections as one product; the backward
// writes d gate and d up side by side, so that the input gradient is one product as well
struct GateUpBackward final : SharedInputFormula {
  enum { X, GU, COUNT };
  GateUpBackward() : SharedInputFormula(COUNT) {}
  std::string name() const override { return "MaltosGateUpBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return variable_list(3);
    const Tensor dgu = swiglu_rows_backward(g[0], dense(s[GU]), rows->first[0], rows->first[1], weights[0].size(0));
    const Tensor dgu2 = rows2d(dgu);
    return grads_of_all(*rows, weights, into_grad, needed(), s[X], dgu2);
  }
};

Tensor gate_up(const Tensor& x, const AdjacentPtr& rows, const std::vector<Tensor>& weights, bool into_grad) {
  refuse_function_transforms("gate_up", x, weights);
  const bool recorded = at::GradMode::is_enabled() && (compute_requires_grad(x) || any_requires_grad(weights));
  Tensor gu, h;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(gu, h) = gate_up_activation(x, *rows, weights, recorded);
  }
  if (recorded) {
    const auto fn = adjacent_formula<GateUpBackward>(x, rows, weights, into_grad);
    fn->save(fn->GU, gu);
    set_history(h, fn);
  }
  return h;
}

// ---- attention(rotary(q), rotary(k), v) (models/llama.py:143-150) as one node ---------------------------------------------
// The same kernels as the separate ops, hence the same values.  What the node adds is the layout of its backward: dQ, dK and
// dV are head ranges of one [B, S, Hq + 2 Hkv, D] buffer, dQ and dK rotated back on their way there, so the gradient of q/k/v projections that run as one product arrives as one matrix.
struct RopeAttentionBackward final : Formula {
  enum { Q, K, V, OUT, LSE, COS, SIN, ROPE_POSITIONS, POSITIONS, SEQUENCES, COUNT };
  int64_t position_offset = 0, mask_mode = 0;
  double scale = 0;
  RopeAttentionBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosRopeAttentionBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return variable_list(3);
    const OptTensor pos = optional_tensor(s[POSITIONS]), seq = optional_tensor(s[SEQUENCES]);
    auto [dq, dk, dv] =
        rotated_attention_backward(g[0], s[Q], s[K], s[V], s[OUT], s[LSE], mask_mode, scale, pos, pos, seq, seq, {s[COS], s[SIN], optional_tensor(s[ROPE_POSITIONS]), position_offset});
    return {dq, dk, dv};
  }
};

Tensor rope_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cos, const Tensor& sin, const OptTensor& rope_positions,
                      int64_t position_offset, const OptTensor& positions, const OptTensor& sequences) {
  refuse_function_transforms("rope_attention", q, {k, v, cos, sin});
  std::shared_ptr<RopeAttentionBackward> fn;
  Tensor out;
  const int64_t mask_mode = positions.has_value() ? MLTS_MASK_DOC : MLTS_MASK_CAUSAL;
  const double scale = std::pow(static_cast<double>(q.size(-1)), -0.5);
  if (compute_requires_grad(q, k, v)) {
    fn = make_formula<RopeAttentionBackward>();
    fn->set_next_edges(collect_next_edges(q, k, v));
    fn->save(fn->V, v);
    fn->save(fn->COS, cos), fn->save(fn->SIN, sin);
    fn->save(fn->ROPE_POSITIONS, rope_positions), fn->save(fn->POSITIONS, positions), fn->save(fn->SEQUENCES, sequences);
    fn->position_offset = position_offset, fn->mask_mode = mask_mode, fn->scale = scale;
  }
  Tensor qr, kr, lse;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(qr, kr) = rope_pair(q, k, cos, sin, rope_positions, position_offset, false, false);
    std::tie(out, lse) = attention_forward(qr, kr, v, mask_mode, scale, positions, positions, sequences, sequences);
  }
  if (fn) {
    set_history(out, fn);
    fn->save(fn->Q, qr), fn->save(fn->K, kr), fn->save(fn->LSE, lse), fn->save(fn->OUT, out, true);
  }
  return out;
}

// ---- the layers of a model ------------------------------------------------------------------------------------------------
// What a decoder layer is made of (models/llama.py:217-231) as four autograd nodes and no Python: the two norms above and the two
// blocks below, with the kernels and the values of the modules one by one.  At a thousand tokens a layer's kernels take 60 us
// forward, calling its modules one after the other 110 us of host time, and the views between them cost the backward pass
// another 20.

// [B, H, S, D] as [B * S, H * D] rows: a view of [B, S, H, D] storage (or a column range of wider rows), a copy of any other layout
// (a saved tensor may come back from the user's hooks in another one)
Tensor as_rows(const Tensor& t) {
  const int64_t B = t.size(0), H = t.size(1), S = t.size(2), D = t.size(3);
  if (t.stride(3) == 1 && t.stride(1) == D && t.stride(2) >= H * D && t.stride(0) == S * t.stride(2))
    return t.as_strided({B * S, H * D}, {t.stride(2), 1}, t.storage_offset());
  return t.transpose(1, 2).reshape({B * S, H * D});
}
// columns col .. col + heads * dim of [B, S, width] rows as [B, heads, S, dim]
Tensor as_heads(const Tensor& rows, int64_t batch, int64_t seq, int64_t width, int64_t col, int64_t heads, int64_t dim) {
  return rows.as_strided({batch, heads, seq, dim}, {seq * width, dim, width, 1}, rows.storage_offset() + col);
}

struct BlockWeights {
  AdjacentPtr rows;              // of the projections that share the block's input
  std::vector<Tensor> in;        // q, k, v or gate, up
  Tensor out;                    // o or down
  bool into_grad_in = false, into_grad_out = false;
};

template <typename F>
std::shared_ptr<F> block_formula(const Tensor& x, const BlockWeights& w) {
  auto fn = adjacent_formula<F>(x, w.rows, w.in, w.into_grad_in);
  fn->add_next_edge(torch::autograd::impl::gradient_edge(w.out));
  fn->save(fn->OUT_W, w.out);
  fn->into_grad_out = w.into_grad_out;
  return fn;
}
bool recorded(const Tensor& x, const BlockWeights& w) {
  return at::GradMode::is_enabled() && (compute_requires_grad(x, w.out) || any_requires_grad(w.in));
}

// A formula of a whole block: the last output is the gradient of the last projection's weight
struct BlockFormula : public SharedInputFormula {
  bool into_grad_out = false;
  using SharedInputFormula::SharedInputFormula;
  // the last projection: the gradients of its input (if something in front of it needs one) and of its weight
  std::pair<Tensor, Tensor> output_grads(const Tensor& dy, const Tensor& w, const Tensor& rows, const Needed& in) const {
    const bool need_dw = task_should_compute_output(1 + weights.size());
    const Tensor grad = need_dw ? bound_grad(w, into_grad_out) : Tensor();
    auto grads = input_and_weight_grad(rows2d(dense(dy)), w, rows, grad, in.input || in.any_weight, need_dw);
    if (grad.defined()) notify_grad_written(w);
    return grads;
  }
};

struct AttentionBlockBackward final : BlockFormula {
  enum { X, Q, K, V, OUT, LSE, COS, SIN, ROPE_POSITIONS, POSITIONS, SEQUENCES, OUT_W, COUNT };
  int64_t position_offset = 0, mask_mode = 0;
  double scale = 0;
  AttentionBlockBackward() : BlockFormula(COUNT) {}
  std::string name() const override { return "MaltosAttentionBlockBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return variable_list(5);
    const Tensor &q = s[Q], &k = s[K];
    const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
    const Needed need = needed();
    auto [dvo, dwo] = output_grads(g[0], s[OUT_W], as_rows(s[OUT]), need);
    if (!dvo.defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), dwo};
    const OptTensor pos = optional_tensor(s[POSITIONS]), seq = optional_tensor(s[SEQUENCES]);
    auto [dq, dk, dv] =
        rotated_attention_backward(as_heads(dvo, B, S, H * D, 0, H, D), q, k, s[V], s[OUT], s[LSE], mask_mode, scale, pos, pos, seq, seq, {s[COS], s[SIN], optional_tensor(s[ROPE_POSITIONS]), position_offset});
    const std::vector<Tensor> parts = {as_rows(dq), as_rows(dk), as_rows(dv)};
    Tensor dqkv = adjacent_columns(parts, rows->order);
    if (!dqkv.defined()) {
      std::vector<Tensor> ordered;
      for (size_t i : rows->order) ordered.push_back(parts[i]);
      dqkv = at::cat(ordered, 1);
    }
    variable_list out = grads_of_all(*rows, weights, into_grad, need, s[X], dqkv);
    out.push_back(dwo);
    return out;
  }
};

struct Positions {
  int64_t offset = 0;
  OptTensor rope, ids, sequences;  // int32 rotary positions; positions and sequence ids of a document mask
};

// q, k and v side by side with q and k rotated on the way out of their products, or undefined: sizes, layouts and positions that are left to
// a pass of their own
Tensor project_rotated(const Tensor& x, const BlockWeights& w, int64_t heads, int64_t kv_heads, const Tensor& cos, const Tensor& sin, const Positions& p) {
  const Adjacent& rows = *w.rows;
  const int64_t B = x.size(0), S = x.size(1), D = w.in[0].size(0) / heads, max_pos = cos.dim() == 2 ? cos.size(0) : 0;
  const auto table = [&](const Tensor& t) {
    return t.is_cuda() && t.is_contiguous() && t.dim() == 2 && t.size(0) == max_pos && t.size(1) * 2 == D && t.scalar_type() == x.scalar_type() && aligned(t);
  };
  const bool given = p.rope.has_value() && p.rope->defined();
  if (!x.is_contiguous() || !table(cos) || !table(sin) || max_pos > 0x7fffffff || S > 0x7fffffff) return Tensor();
  if (given ? !p.rope->is_cuda() || p.rope->scalar_type() != at::kInt || !p.rope->is_contiguous() || p.rope->sizes() != at::IntArrayRef({B, S})
            : p.offset < 0 || p.offset + S > max_pos)
    return Tensor();
  const Tensor x2 = rows2d(x);
  if (rows.weight.defined() && !own_product(MLTS_GEMM_NT, x2, rows.weight, Use::ROTATION)) return Tensor();
  const Tensor y = at::empty({B, S, rows.width}, x.options()), y2 = rows2d(y);
  mlts_gemm_rotation r{};
  r.cos = ptr(cos), r.sin = ptr(sin), r.positions = given ? p.rope->const_data_ptr<int32_t>() : nullptr;
  r.max_pos = static_cast<int32_t>(max_pos), r.position_offset = given ? 0 : static_cast<int32_t>(p.offset);
  r.seq = static_cast<int32_t>(S), r.head_dim = static_cast<int32_t>(D);
  ProductList list;
  if (rows.weight.defined()) {
    list.add(MLTS_GEMM_NT, x2, rows.weight, y2, false);
    r.columns[0][0] = rows.first[0], r.columns[0][1] = rows.first[0] + heads * D;
    r.columns[0][2] = rows.first[1], r.columns[0][3] = rows.first[1] + kv_heads * D;
  } else {
    for (size_t i = 0; i < w.in.size(); ++i) list.add(MLTS_GEMM_NT, x2, w.in[i], y2.narrow(1, rows.first[i], w.in[i].size(0)), false);
    r.columns[0][1] = heads * D, r.columns[1][1] = kv_heads * D;
  }
  if (mlts_gemm_rope_supports(list.items, list.count, dtype_code(x), &r) != nullptr) return Tensor();
  check(mlts_gemm_rope(list.items, list.count, dtype_code(x), &r, current_stream()));
  return y;
}

Tensor attention_block(const Tensor& x, const BlockWeights& w, int64_t heads, int64_t kv_heads, const Tensor& cos, const Tensor& sin, const Positions& p) {
  const int64_t B = x.size(0), S = x.size(1), D = w.in[0].size(0) / heads, width = w.rows->width;
  const int64_t mask_mode = p.ids.has_value() ? MLTS_MASK_DOC : MLTS_MASK_CAUSAL;
  const double scale = std::pow(static_cast<double>(D), -0.5);
  Tensor q, k, v, qr, kr, out, lse, y;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    Tensor qkv = project_rotated(x, w, heads, kv_heads, cos, sin, p);
    const bool rotated = qkv.defined();
    if (!rotated) qkv = project_all(x, *w.rows, w.in);
    q = as_heads(qkv, B, S, width, w.rows->first[0], heads, D);
    k = as_heads(qkv, B, S, width, w.rows->first[1], kv_heads, D);
    v = as_heads(qkv, B, S, width, w.rows->first[2], kv_heads, D);
    if (rotated) qr = q, kr = k;
    else std::tie(qr, kr) = rope_pair(q, k, cos, sin, p.rope, p.offset, false, false);
    std::tie(out, lse) = attention_forward(qr, kr, v, mask_mode, scale, p.ids, p.ids, p.sequences, p.sequences);
    y = product(MLTS_GEMM_NT, as_rows(out), w.out).view({B, S, w.out.size(0)});
  }
  if (recorded(x, w)) {
    auto fn = block_formula<AttentionBlockBackward>(x, w);
    fn->save(fn->Q, qr), fn->save(fn->K, kr), fn->save(fn->V, v), fn->save(fn->OUT, out), fn->save(fn->LSE, lse);
    fn->save(fn->COS, cos), fn->save(fn->SIN, sin);
    fn->save(fn->ROPE_POSITIONS, p.rope), fn->save(fn->POSITIONS, p.ids), fn->save(fn->SEQUENCES, p.sequences);
    fn->position_offset = p.offset, fn->mask_mode = mask_mode, fn->scale = scale;
    set_history(y, fn);
  }
  return y;
}

// the gradients of an MLP's gate and up side by side, and (need_dw) of its last projection's weight, in one launch where that runs on the own
// kernels; undefined: sizes and layouts that are left to the products and the pass over gate and up
std::pair<Tensor, Tensor> activation_and_weight_grad(const Tensor& dy2, const Tensor& w, const Tensor& h2, const Tensor& gu, const Adjacent& rows,
                                                     const Tensor& grad, bool need_dw) {
  const int64_t cols = w.size(1), es = gu.element_size(), width = gu.size(-1);
  if (width != 2 * cols || !gu.is_contiguous() || !aligned(gu) || (rows.first[0] * es) % 16 || (rows.first[1] * es) % 16 ||
      !own_product(MLTS_GEMM_NN, dy2, w, Use::ACTIVATION) || (need_dw && !own_product(MLTS_GEMM_TN, dy2, h2, Use::ACTIVATION)) || gu.scalar_type() != dy2.scalar_type() || gu.numel() / width != dy2.size(0) ||
      (grad.defined() && (!own_output(grad, h2) || !grad.is_contiguous())))
    return {};
  int64_t ws_bytes = 0;
  const int dtype = dtype_code(dy2);
  if (mlts_gemm_swiglu_bwd_supports(dtype, need_dw, dy2.size(0), cols, dy2.size(1), dy2.stride(0), w.stride(0), h2.stride(0), width, width,
                                    &ws_bytes) != nullptr)
    return {};
  const Tensor dgu = at::empty(gu.sizes(), gu.options());
  const Tensor dw = !need_dw ? Tensor() : grad.defined() ? grad : at::empty(w.sizes(), dy2.options());
  const Tensor ws = workspace(ws_bytes, dy2);
  const char* in = static_cast<const char*>(ptr(gu));
  char* out = static_cast<char*>(mptr(dgu));
  check(mlts_gemm_swiglu_bwd(dtype, dy2.size(0), cols, dy2.size(1), ptr(dy2), dy2.stride(0), ptr(w), w.stride(0), ptr(h2), h2.stride(0), need_dw ? mptr(dw) : nullptr,
                             grad.defined(), in + rows.first[0] * es, in + rows.first[1] * es, width, out + rows.first[0] * es, out + rows.first[1] * es, width,
                             ws.defined() ? mptr(ws) : nullptr, ws_bytes, current_stream()));
  return {dgu, dw};
}

struct MlpBlockBackward final : BlockFormula {
  enum { X, GU, H, OUT_W, COUNT };
  MlpBlockBackward() : BlockFormula(COUNT) {}
  std::string name() const override { return "MaltosMlpBlockBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return variable_list(4);
    const Needed need = needed();
    Tensor dgu, dw;
    if (need.input || need.any_weight) {
      const bool need_dw = task_should_compute_output(1 + weights.size());
      const Tensor grad = need_dw ? bound_grad(s[OUT_W], into_grad_out) : Tensor();
      std::tie(dgu, dw) = activation_and_weight_grad(rows2d(dense(g[0])), s[OUT_W], rows2d(s[H]), dense(s[GU]), *rows, grad, need_dw);
      if (dgu.defined() && grad.defined()) dw = Tensor(), notify_grad_written(s[OUT_W]);
    }
    if (!dgu.defined()) {
      Tensor dh;
      std::tie(dh, dw) = output_grads(g[0], s[OUT_W], rows2d(s[H]), need);
      if (!dh.defined()) return {Tensor(), Tensor(), Tensor(), dw};
      dgu = swiglu_rows_backward(dh.view(s[H].sizes()), dense(s[GU]), rows->first[0], rows->first[1], weights[0].size(0));
    }
    variable_list out = grads_of_all(*rows, weights, into_grad, need, s[X], rows2d(dgu));
    out.push_back(dw);
    return out;
  }
};

Tensor mlp_block(const Tensor& x, const BlockWeights& w) {
  const bool keep = recorded(x, w);
  Tensor gu, h, y;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(gu, h) = gate_up_activation(x, *w.rows, w.in, keep);
    y = project(h, w.out);
  }
  if (keep) {
    auto fn = block_formula<MlpBlockBackward>(x, w);
    fn->save(fn->GU, gu), fn->save(fn->H, h);
    set_history(y, fn);
  }
  return y;
}

// A borrowed look at a module: its attributes without going through Python's attribute lookup.
struct ModuleView {
  PyObject* module;
  PyObject* dict;
  explicit ModuleView(PyObject* m) : module(m) {
    PyObject** p = m ? _PyObject_GetDictPtr(m) : nullptr;
    dict = p ? *p : nullptr;
  }
  PyObject* item(const char* name) const { return dict ? PyDict_GetItemString(dict, name) : nullptr; }
  PyObject* in(const char* table, const char* name) const {
    PyObject* t = item(table);
    return t && PyDict_Check(t) ? PyDict_GetItemString(t, name) : nullptr;
  }
  // exactly of this class, and nothing hangs on its call
  bool stock(const pybind11::handle& type) const {
    if (!dict || reinterpret_cast<PyObject*>(Py_TYPE(module)) != type.ptr() || item("forward")) return false;
    for (const char* hooks : {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"}) {
      PyObject* h = item(hooks);
      if (!h || !PyDict_Check(h) || PyDict_Size(h) != 0) return false;
    }
    return true;
  }
  Tensor tensor(const char* table, const char* name) const {
    PyObject* t = in(table, name);
    return t && THPVariable_CheckExact(t) ? THPVariable_Unpack(t) : t && THPVariable_Check(t) ? THPVariable_Unpack(t) : Tensor();
  }
  bool flag(const char* name) const {  // on the instance or its class
    PyObject* v = item(name);
    if (v) return PyObject_IsTrue(v) == 1;
    v = PyObject_GetAttrString(reinterpret_cast<PyObject*>(Py_TYPE(module)), name);
    if (!v) PyErr_Clear();
    const bool on = v && PyObject_IsTrue(v) == 1;
    Py_XDECREF(v);
    return on;
  }
  int64_t integer(const char* name) const {
    PyObject* v = item(name);
    return v && PyLong_Check(v) ? PyLong_AsLongLong(v) : 0;
  }
};

// The rows of `params` (see Adjacent), kept on the module until a parameter or gradient moves
AdjacentPtr rows_of_module(const ModuleView& m, const std::vector<Tensor>& params) {
  static const char* const kept = "_maltos_hip_fused_rows";
  if (PyObject* r = m.item(kept); r && r != Py_None) {
    AdjacentPtr rows = pybind11::cast<AdjacentPtr>(pybind11::handle(r));
    if (rows->made_for(params)) return rows;
  }
  auto rows = std::make_shared<Adjacent>(params);
  PyDict_SetItemString(m.dict, kept, pybind11::cast(rows).ptr());
  return rows;
}

struct LayerParts {
  BlockWeights attention, mlp;
  Tensor norm1, norm2, cos, sin;
  double eps1 = 0, eps2 = 0;
  bool into_norm1 = false, into_norm2 = false;
  int64_t heads = 0, kv_heads = 0;
};

// types: the classes of the stock modules; backends: the attention backend names that route to the kernels here
bool read_layer(PyObject* layer, const pybind11::dict& types, const pybind11::handle& backends, const Tensor& x, LayerParts& out) {
  auto child = [](const ModuleView& m, const char* name) { return ModuleView(m.in("_modules", name)); };
  auto type = [&](const char* name) { return pybind11::handle(PyDict_GetItemString(types.ptr(), name)); };
  const ModuleView l(layer);
  if (!l.stock(type("layer"))) return false;
  const ModuleView attn = child(l, "self_attn"), mlp = child(l, "mlp"), n1 = child(l, "input_layernorm"), n2 = child(l, "post_attention_layernorm");
  if (!attn.stock(type("attention")) || !mlp.stock(type("mlp")) || !n1.stock(type("norm")) || !n2.stock(type("norm"))) return false;
  const ModuleView core = child(attn, "attn_core"), rotary = child(attn, "rotary_emb");
  if (!core.stock(type("core")) || !rotary.stock(type("rotary"))) return false;
  PyObject* backend = core.item("attention_backend");
  if (!backend || PySequence_Contains(backends.ptr(), backend) != 1) return false;
  if (!attn.flag("fuse_projections") || !attn.flag("fuse_rope_attention") || !mlp.flag("fuse_projections")) return false;

  auto fits = [&](const Tensor& t, int64_t dims) {
    return t.defined() && ordinary(t) && t.dim() == dims && t.is_cuda() && t.scalar_type() == x.scalar_type() && t.is_contiguous() && t.device() == x.device();
  };
  auto block = [&](const ModuleView& m, std::initializer_list<const char*> ins, const char* last, BlockWeights& w) {
    w.into_grad_in = true;
    for (const char* name : ins) {
      const ModuleView p = child(m, name);
      w.in.push_back(p.stock(type("linear")) && p.in("_parameters", "bias") == Py_None ? p.tensor("_parameters", "weight") : Tensor());
      if (!fits(w.in.back(), 2)) return false;
      w.into_grad_in = w.into_grad_in && p.flag("accumulate_into_grad");
    }
    const ModuleView p = child(m, last);
    w.out = p.stock(type("linear")) && p.in("_parameters", "bias") == Py_None ? p.tensor("_parameters", "weight") : Tensor();
    w.into_grad_out = p.dict && p.flag("accumulate_into_grad");
    if (!fits(w.out, 2) || w.in[0].size(1) != x.size(-1)) return false;
    w.rows = rows_of_module(m, w.in);
    return w.rows->weight.defined() || runs_as_group(*w.rows, x, w.in);
  };
  if (!block(attn, {"q_proj", "k_proj", "v_proj"}, "o_proj", out.attention) || !block(mlp, {"gate_proj", "up_proj"}, "down_proj", out.mlp)) return false;
  const auto &a = out.attention, &m = out.mlp;
  out.heads = attn.integer("num_heads"), out.kv_heads = attn.integer("num_kv_heads");
  const int64_t dim = attn.integer("head_dim");
  if (out.heads <= 0 || out.kv_heads <= 0 || dim <= 0 || dim > 192 || a.in[0].size(0) != out.heads * dim || a.in[1].size(0) != out.kv_heads * dim ||
      a.in[2].size(0) != out.kv_heads * dim || a.out.size(1) != out.heads * dim || a.out.size(0) != x.size(-1))
    return false;
  if (m.in[0].size(0) != m.in[1].size(0) || m.out.size(1) != m.in[0].size(0) || m.out.size(0) != x.size(-1) ||
      m.in[0].size(0) % (16 / x.element_size()) != 0)
    return false;
  out.cos = rotary.tensor("_buffers", "cos"), out.sin = rotary.tensor("_buffers", "sin");
  out.norm1 = n1.tensor("_parameters", "weight"), out.norm2 = n2.tensor("_parameters", "weight");
  PyObject *e1 = n1.item("eps"), *e2 = n2.item("eps");
  if (!fits(out.cos, 2) || !fits(out.sin, 2) || !fits(out.norm1, 1) || !fits(out.norm2, 1) || !e1 || !e2 || !PyFloat_Check(e1) || !PyFloat_Check(e2))
    return false;
  out.eps1 = PyFloat_AsDouble(e1), out.eps2 = PyFloat_AsDouble(e2);
  out.into_norm1 = n1.flag("accumulate_into_grad"), out.into_norm2 = n2.flag("accumulate_into_grad");
  return true;
}

// (x, pending) after all layers of a ModuleList's table, the last residual add left to whoever normalises next; None where a
// layer is not made of stock modules, something hooks into one, or its projections run one by one
pybind11::object run_layers(const pybind11::dict& layers, const pybind11::dict& types, const pybind11::object& backends, const Tensor& x_in,
                            int64_t position_offset, const OptTensor& rope_positions, const OptTensor& positions, const OptTensor& sequences) {
  if (!x_in.is_cuda() || x_in.dim() != 3 || !x_in.is_contiguous() || x_in.numel() == 0 || !ordinary(x_in) ||
      (x_in.scalar_type() != at::kBFloat16 && x_in.scalar_type() != at::kFloat) || c10::impl::dispatch_mode_enabled() ||
      at::autocast::is_autocast_enabled(at::kCUDA))
    return pybind11::none();
  std::vector<LayerParts> parts(PyDict_Size(layers.ptr()));
  size_t count = 0;
  for (auto item : layers)
    if (!read_layer(item.second.ptr(), types, backends, x_in, parts[count++])) return pybind11::none();
  const Positions where{position_offset, rope_positions, positions, sequences};
  Tensor x = x_in, pending;
  {
    pybind11::gil_scoped_release no_gil;
    for (const LayerParts& l : parts) {
      Tensor normed;
      if (pending.defined()) std::tie(x, normed) = add_rms_norm(x, pending, l.norm1, l.eps1, l.into_norm1);
      else normed = rms_norm(x, l.norm1, l.eps1, l.into_norm1);
      const Tensor attn = attention_block(normed, l.attention, l.heads, l.kv_heads, l.cos, l.sin, where);
      std::tie(x, normed) = add_rms_norm(x, attn, l.norm2, l.eps2, l.into_norm2);
      pending = mlp_block(normed, l.mlp);
    }
  }
  return pybind11::make_tuple(x, pending);
}

}  // namespace

void bind_llama(pybind11::module& m) {
  using torch::wrap_pybind_function;
  namespace py = pybind11;
  m.def("run_layers", wrap_pybind_function(run_layers));
  m.def("linear", wrap_pybind_function(linear));
  m.def("embedding", wrap_pybind_function(embedding));
  m.def("product", wrap_pybind_function([](int form, const Tensor& a, const Tensor& b, const OptTensor& out, bool accumulate) {
          at::AutoDispatchBelowADInplaceOrView below_autograd;
          return product(form, a, b, out.value_or(Tensor()), accumulate);
        }), py::arg("form"), py::arg("a"), py::arg("b"), py::arg("out") = py::none(), py::arg("accumulate") = false);
  m.def("adjacent_linears", wrap_pybind_function(adjacent_linears));
  m.def("gate_up", wrap_pybind_function(gate_up));
  m.def("weight_grad_splits", wrap_pybind_function(weight_grad_splits));
  m.def("adjacent_columns", wrap_pybind_function([](const std::vector<Tensor>& parts) {
          std::vector<size_t> order(parts.size());
          std::iota(order.begin(), order.end(), size_t{0});
          const Tensor t = adjacent_columns(parts, order);
          return t.defined() ? OptTensor(t) : std::nullopt;
        }));
  py::class_<Adjacent, AdjacentPtr>(m, "Adjacent")
      .def(py::init<const std::vector<Tensor>&>())
      // (kept on modules, which are copied and pickled: a copy makes its own)
      .def("__reduce__", [](const Adjacent&) { return py::make_tuple(py::type::of(py::none()), py::tuple()); })
      .def("made_for", &Adjacent::made_for)
      .def("runs_as_group", &runs_as_group)
      .def_property_readonly("adjacent", [](const Adjacent& a) { return a.weight.defined(); })
      .def_property_readonly("weight", [](const Adjacent& a) { return a.weight.defined() ? OptTensor(a.weight) : std::nullopt; })
      .def_property_readonly("grad", [](const Adjacent& a) { return a.grad.defined() ? OptTensor(a.grad) : std::nullopt; });
  m.def("rope_attention", wrap_pybind_function(rope_attention));
  m.def("notify_grad_written", wrap_pybind_function(notify_grad_written));
  py::class_<GradMarks>(m, "GradMarks")
      .def(py::init<std::vector<Tensor>>())
      .def("list", &GradMarks::list)
      .def("all", &GradMarks::all)
      .def("fill", &GradMarks::fill);
  py::class_<GradListener>(m, "GradListener").def(py::init<>()).def("start", &GradListener::start).def("stop", &GradListener::stop);
  py::class_<FlatViews>(m, "FlatViews")
      .def(py::init<std::vector<Tensor>, std::vector<int64_t>>())
      .def("grads_are_views_of", &FlatViews::grads_are_views_of)
      .def("grads_defined", &FlatViews::grads_defined);
}

}  // namespace maltos
