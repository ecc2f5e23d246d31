// Host side between torch tensors and the C ABI (include/maltos_hip.h): shared helpers of the sources in this folder.
//
// What an eager training step pays per operator besides its kernels is host time: an operator whose implementation,
// autograd formula and argument checks are Python costs 40-60 us per call (forward and backward together), several times
// the kernel it launches at small sizes.  Here the same operators are C++ from the Python entry point to the launch.
#pragma once
#include <ATen/ATen.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <tuple>
#include <utility>
#include <vector>

#include "../../../include/maltos_hip.h"

namespace maltos {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::Edge;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

[[noreturn]] void raise_status(int status);  // the exception maltos_amd._lib.check raises for this status
inline void check(int status) {
  if (C10_UNLIKELY(status != MLTS_OK)) raise_status(status);
}

inline int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return MLTS_BF16;
  if (t.scalar_type() == at::kFloat) return MLTS_F32;
  TORCH_CHECK_VALUE(false, "maltos_amd kernels take float32 or bfloat16 tensors, got ", t.scalar_type());
}

inline void require_gpu(const Tensor& t) {
  TORCH_CHECK(!t.defined() || t.is_cuda(), "maltos_amd ops run on the GPU only (there is no CPU fallback); got a host tensor");
}
inline void require_gpu(const OptTensor& t) {
  if (t.has_value()) require_gpu(*t);
}

// Forward-mode tangents: the kernels have no formula for them, and an output without one reads as a derivative of zero.
inline bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(0).defined(); }
template <typename... T>
void refuse_tangents(const char* what, const T&... tensors) {
  TORCH_CHECK_NOT_IMPLEMENTED(!(has_tangent(tensors) || ...), what, ": maltos_amd has no forward-mode derivative of this operator");
}

// tensors of function transforms (torch.func)
inline bool of_transform(const Tensor& t) {
  return t.defined() && (t.key_set().has(c10::DispatchKey::FuncTorchBatched) || t.key_set().has(c10::DispatchKey::FuncTorchGradWrapper));
}
// Whether something around the innermost transform differentiates this value: what a node records in there is not seen by it.
bool differentiated_outside(Tensor t);

inline mlts_stream_t current_stream() { return c10::hip::getCurrentHIPStream().stream(); }
inline bool stream_is_capturing() {
  return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

inline const void* ptr(const Tensor& t) { return t.const_data_ptr(); }
inline void* mptr(const Tensor& t) { return t.mutable_data_ptr(); }
inline const void* ptr(const OptTensor& t) { return t.has_value() && t->defined() ? t->const_data_ptr() : nullptr; }

inline bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }  // to 16-byte accesses

inline Tensor workspace(int64_t bytes, const Tensor& like) {
  if (bytes <= 0) return Tensor();
  return at::empty({bytes}, like.options().dtype(at::kByte));
}

// contiguous without a copy where it already is (Tensor::contiguous does the same but goes through the dispatcher)
inline Tensor dense(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }
// the kernels take any (batch, head, seq) strides but need a contiguous head_dim
inline Tensor dense_last(const Tensor& t) { return t.stride(-1) == 1 || t.size(-1) == 1 ? t : t.contiguous(); }

struct Strides3 {
  int64_t v[3];
  explicit Strides3(const Tensor& t) : v{t.stride(0), t.stride(1), t.stride(2)} {}
};

// [B, H, S, D] over [B, S, H, D] storage: the layout a projection output is transposed from and back to
inline Tensor bshd_empty(int64_t B, int64_t H, int64_t S, int64_t D, const at::TensorOptions& opts) {
  return at::empty_strided({B, H, S, D}, {S * H * D, D, H * D, 1}, opts);
}

// ---- raw launches (no autograd) -----------------------------------------------------------------------------------
std::tuple<Tensor, Tensor> attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, int64_t mask_mode, double scale,
                                             const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq);
std::tuple<Tensor, Tensor, Tensor> attention_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                      const Tensor& lse, int64_t mask_mode, double scale, const OptTensor& q_pos,
                                                      const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq);
// rotary positions that q and k were rotated by (rope_pair): their gradients come back rotated back
struct RotatedBy {
  const Tensor &cos, &sin;
  OptTensor positions;
  int64_t offset;
};
std::tuple<Tensor, Tensor, Tensor> rotated_attention_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                              const Tensor& lse, int64_t mask_mode, double scale, const OptTensor& q_pos,
                                                              const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq, const RotatedBy& rotated);
std::tuple<Tensor, Tensor> rope_pair(const Tensor& xa, const Tensor& xb, const Tensor& cos, const Tensor& sin, const OptTensor& positions,
                                     int64_t position_offset, bool inverse, bool in_place);
Tensor swiglu_rows(const Tensor& gu, int64_t gate_col, int64_t up_col, int64_t cols);
Tensor swiglu_rows_backward(const Tensor& dh, const Tensor& gu, int64_t gate_col, int64_t up_col, int64_t cols);
Tensor grad_sum_slices(const Tensor& parts, const OptTensor& out, bool accumulate);

// with autograd; into_grad: the weight's gradient is added into the buffer it owns
Tensor rms_norm(const Tensor& x, const Tensor& w, double eps, bool into_grad);
std::tuple<Tensor, Tensor> add_rms_norm(const Tensor& x, const Tensor& res, const Tensor& w, double eps, bool into_grad);  // (sum, its norm)

int64_t weight_grad_splits(int64_t rows, int64_t out_features, int64_t in_features);  // products.cpp
// What shares a product's launch: nothing; dx and dW of one layer each other; the rotation; the activation, gate and up being kept; the activation alone, or its gradient
enum class Use { ALONE, WITH_WEIGHT_GRAD, ROTATION, GATE_AND_UP, ACTIVATION };
bool own_product(int form, const Tensor& a, const Tensor& b, Use use = Use::ALONE);  // whether it runs on the own kernels: by size, type, layout
// a, b as the form (MLTS_GEMM_*) says -> [M, N], written to `out` (or added onto it) if that is given
Tensor product(int form, const Tensor& a, const Tensor& b, const Tensor& out = Tensor(), bool accumulate = false);  // products.cpp

bool own_output(const Tensor& out, const Tensor& a);  // whether the own kernels can write a product with `a` to `out`
// Products that run on the own kernels (own_product, own_output), in one call: small ones in one launch.
struct ProductList {
  mlts_gemm_product items[4];
  int count = 0;
  Tensor like;
  void add(int form, const Tensor& a, const Tensor& b, const Tensor& out, bool accumulate);
  void add_segment(const Tensor& a, const Tensor& b);  // NN: the last product also gets + a b
  void run() const;
};

void notify_grad_written(const Tensor& param);  // llama.cpp: the parameter's gradient buffer was written past autograd
// the gradient buffer a weight already owns and a backward formula may add into, or undefined (a backward pass that is itself
// recorded leaves the adding to autograd: what the buffer holds has no history)
inline Tensor bound_grad(const Tensor& weight, bool into_grad) {
  if (!into_grad || at::GradMode::is_enabled()) return Tensor();
  const Tensor& g = weight.grad();
  if (!g.defined() || !g.is_contiguous() || g.scalar_type() != weight.scalar_type() || g.sizes() != weight.sizes()) return Tensor();
  return g;
}

void bind_ops(pybind11::module& m);    // ops.cpp
void bind_llama(pybind11::module& m);  // llama.cpp

// A backward formula over saved tensors.  The tensors are unpacked first, with autograd as it is (an unpack hook may run a
// checkpointed forward again), then `backward` runs without autograd recording.  A backward pass that is to be differentiated
// itself (create_graph) goes to `recorded_backward`.
struct Formula : public Node {
  explicit Formula(size_t count) : saved_(count) {}
  virtual variable_list backward(variable_list&& grads, const std::vector<Tensor>& saved) = 0;
  void save(size_t slot, const Tensor& t, bool is_output = false) {
    saved_[slot] = SavedVariable(t, is_output);
    if (is_output) outputs_ |= uint32_t{1} << slot;
  }
  void save(size_t slot, const OptTensor& t) {
    if (t.has_value()) save(slot, *t);
  }
  variable_list apply(variable_list&& grads) final {
    before_unpack(grads);
    std::vector<Tensor> values(saved_.size());
    for (size_t i = 0; i < saved_.size(); ++i) values[i] = saved_[i].unpack((outputs_ >> i) & 1 ? getptr() : nullptr);
    if (at::GradMode::is_enabled()) return recorded_backward(std::move(grads), values);
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    return backward(std::move(grads), values);
  }
  virtual void before_unpack(const variable_list&) {}
  // The backward kernels have no derivatives: their results carry an error as history, so that a second derivative raises where
  // its terms would be missing.  Formulas made of differentiable operators override this.
  virtual variable_list recorded_backward(variable_list&& grads, const std::vector<Tensor>& saved) {
    static const char* const refusal = ": maltos_amd has no second derivative of this operator";
    for (const std::vector<Tensor>* values : {&std::as_const(grads), &saved})
      for (const Tensor& t : *values) TORCH_CHECK(!differentiated_outside(t), name(), refusal);
    torch::autograd::edge_list sources;
    for (const Tensor& g : grads)
      if (g.defined() && g.requires_grad()) sources.push_back(torch::autograd::impl::gradient_edge(g));
    for (const Edge& e : next_edges())
      if (e.is_valid()) sources.push_back(e);
    variable_list out;
    {
      at::AutoDispatchBelowADInplaceOrView below_autograd;
      out = backward(std::move(grads), saved);
      for (Tensor& t : out)
        if (t.defined()) t = t.detach();  // (a result may be one of the gradients, or stand there twice)
    }
    const auto error = std::shared_ptr<Node>(new torch::autograd::Error(name() + refusal, std::move(sources)),
                                             torch::autograd::deleteNode);
    for (const Tensor& t : out)
      if (t.defined()) torch::autograd::set_history(t, error);
    return out;
  }
  void release_variables() override {
    for (SavedVariable& s : saved_) s.reset_data();
  }

 private:
  std::vector<SavedVariable> saved_;
  uint32_t outputs_ = 0;
};

inline OptTensor optional_tensor(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }

template <typename F>
std::shared_ptr<F> make_formula() {
  return std::shared_ptr<F>(new F(), torch::autograd::deleteNode);
}

}  // namespace maltos
