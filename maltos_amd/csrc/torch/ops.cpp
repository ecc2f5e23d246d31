// The maltos:: operators over the C ABI: argument checks, output allocation, launches and autograd formulas.  Their
// schemas and fake kernels are registered by maltos_amd/ops.py.
#include <torch/library.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <iterator>
#include <list>
#include <memory>
#include <mutex>
#include <vector>

#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "common.hpp"

namespace maltos {

void raise_status(int status) {
  const char* text = mlts_last_error();
  const std::string msg = text && *text ? text : "libmaltos_hip status " + std::to_string(status);
  TORCH_CHECK_VALUE(status != MLTS_ERR_INVALID, msg);
  TORCH_CHECK(status != MLTS_ERR_UNSUPPORTED, msg);
  pybind11::gil_scoped_acquire gil;
  const pybind11::object error = pybind11::module_::import("maltos_amd._lib").attr("MaltosHipError");
  PyErr_SetString(error.ptr(), msg.c_str());
  throw pybind11::error_already_set();
}

bool differentiated_outside(Tensor t) {
  if (!of_transform(t)) return false;
  pybind11::gil_scoped_acquire gil;
  const pybind11::object unwrap = pybind11::module_::import("torch._C._functorch").attr("get_unwrapped");
  while (of_transform(t)) {
    t = unwrap(t).cast<Tensor>();
    if (t.requires_grad() || t.key_set().has(c10::DispatchKey::FuncTorchGradWrapper)) return true;
  }
  return false;
}

namespace {

void check_attn_inputs(const Tensor& q, const Tensor& k, const Tensor& v) {
  TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "attention expects q, k, v of shape [batch, heads, seq, head_dim]");
  TORCH_CHECK_VALUE(k.sizes() == v.sizes(), "k and v must have identical shapes, got ", k.sizes(), " vs ", v.sizes());
  TORCH_CHECK_VALUE(q.size(0) == k.size(0) && q.size(3) == k.size(3), "q and k disagree on batch or head_dim: ", q.sizes(), " vs ", k.sizes());
  TORCH_CHECK_VALUE(k.size(1) > 0 && q.size(1) % k.size(1) == 0, "query heads (", q.size(1), ") must be a multiple of kv heads (", k.size(1), ")");
  TORCH_CHECK_VALUE(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(), "q, k, v must share a dtype");
}

double resolve_scale(const std::optional<double>& scale, const Tensor& q) {
  return scale.has_value() ? *scale : std::pow(static_cast<double>(q.size(3)), -0.5);
}

// ---- position / sequence ids --------------------------------------------------------------------------------------
struct Ids {
  OptTensor given[4];  // q_pos, k_pos, q_seq, k_seq as the caller has them
  OptTensor used[4];   // int32 contiguous, what the kernels read
};

OptTensor ids32(const OptTensor& t, int64_t batch, int64_t seq, const char* what) {
  if (!t.has_value() || !t->defined()) return std::nullopt;
  TORCH_CHECK_VALUE(t->dim() == 2 && t->size(0) == batch && t->size(1) == seq, what, " must have shape (", batch, ", ", seq, "), got ", t->sizes());
  if (t->scalar_type() == at::kInt && t->is_contiguous()) return t;
  return t->to(at::kInt).contiguous();
}

void check_tables(const Tensor& x, const Tensor& cos, const Tensor& sin) {
  const int64_t half = x.size(3) / 2;
  TORCH_CHECK_VALUE(cos.sizes() == sin.sizes() && cos.dim() == 2 && cos.size(1) * 2 == x.size(3), "cos/sin tables must be [max_pos, ", half,
                    "], got ", cos.sizes());
  TORCH_CHECK_VALUE(cos.scalar_type() == x.scalar_type() && sin.scalar_type() == x.scalar_type(),
                    "cos/sin tables must have the activation dtype (the reference casts them first)");
}
const int32_t* ids_ptr(const OptTensor& t) { return t.has_value() && t->defined() ? t->const_data_ptr<int32_t>() : nullptr; }

// ---- document-mask plans (mlts_attn_doc_plan) -----------------------------------------------------------------------
// Every layer of a model, forward and backward, attends under the same ids, so the plan of a call is kept and handed to
// later calls with the same ids.  "The same" is judged without reading device memory: same address, dtype, shape, strides
// and autograd version of the four id tensors as given by the caller, which are kept alive with the plan so that their
// addresses cannot be handed to other tensors meanwhile (an in-place change of the ids through torch bumps the version;
// writes behind torch's back are not seen: clear_doc_plan_cache()).  The int32 forms of the ids are kept with it, also for calls
// that have no plan (fp32, other head dims), if they had to be made.
struct PlanKey {
  int64_t shape[7];
  int64_t device;
  void* stream;
  struct Id {
    const void* data;
    int64_t version, dtype, sizes[2], strides[2];
  } ids[4];
};
struct PlanEntry {
  PlanKey key;
  Ids ids;
  Tensor plan;
};
// Forward runs on the caller's thread, backward on autograd's device thread.  A thread that holds the mutex must not wait for Python's
// interpreter lock, whose holder may be waiting for the mutex: no tensor is made, copied or released under it (one that Python has
// an object of may need that lock), only references to entries move.
typedef std::list<std::shared_ptr<const PlanEntry>> PlanList;
PlanList& plan_cache = *new PlanList;  // (never destroyed: its tensors must not outlive the runtime)
std::atomic<size_t> plan_cache_entries{8};
constexpr int64_t kPlanCacheBytes = int64_t{1} << 30;  // most bytes of plans kept (a plan is B * Sq * Sk / 4 bytes)
std::mutex plan_mutex;

bool same_key(const PlanKey& a, const PlanKey& b) { return std::memcmp(&a, &b, sizeof(PlanKey)) == 0; }

PlanKey plan_key(const mlts_attn_shape& s, const Ids& ids, const Tensor& q) {
  PlanKey key;
  std::memset(&key, 0, sizeof(key));
  const int64_t dims[7] = {s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, s.dtype};
  std::copy(dims, dims + 7, key.shape);
  key.device = q.device().index();
  key.stream = current_stream();
  for (int i = 0; i < 4; ++i) {
    const Tensor& t = *ids.given[i];
    PlanKey::Id& id = key.ids[i];
    id.data = t.const_data_ptr();
    id.version = t._version();
    id.dtype = static_cast<int64_t>(t.scalar_type());
    for (int d = 0; d < 2; ++d) id.sizes[d] = t.size(d), id.strides[d] = t.stride(d);
  }
  return key;
}

std::shared_ptr<const PlanEntry> find_plan(const PlanKey& key) {
  std::lock_guard<std::mutex> lock(plan_mutex);
  for (auto it = plan_cache.begin(); it != plan_cache.end(); ++it)
    if (same_key((*it)->key, key)) {
      plan_cache.splice(plan_cache.begin(), plan_cache, it);
      return *it;
    }
  return nullptr;
}

// the oldest entries beyond the limits, for the caller to release once it has let go of the mutex
void evict_plans(PlanList& gone) {
  auto bytes = [] {
    int64_t n = 0;
    for (const auto& e : plan_cache) n += e->plan.defined() ? e->plan.numel() : 0;
    return n;
  };
  while (plan_cache.size() > plan_cache_entries || bytes() > kPlanCacheBytes) gone.splice(gone.begin(), plan_cache, std::prev(plan_cache.end()));
}

void keep_plan(std::shared_ptr<const PlanEntry> entry) {
  PlanList gone;
  std::lock_guard<std::mutex> lock(plan_mutex);
  plan_cache.push_front(std::move(entry));
  evict_plans(gone);
}

void point_at_ids(mlts_attn_shape& s, const Ids& ids) {
  s.q_pos = ids.used[0]->const_data_ptr<int32_t>();
  s.k_pos = ids.used[1]->const_data_ptr<int32_t>();
  s.q_seq = ids.used[2]->const_data_ptr<int32_t>();
  s.k_seq = ids.used[3]->const_data_ptr<int32_t>();
}

void check_supported(const mlts_attn_shape& s, const char* who) {
  const char* why = mlts_attn_supports(&s);
  TORCH_CHECK_VALUE(why == nullptr, who, ": ", why);
}

// int32 ids and, where one may be kept, the plan of a document-masked call.  The returned tensor (and ids.used) must stay
// alive over the launch.
Tensor attach_document_ids(mlts_attn_shape& s, Ids& ids, const Tensor& q, const char* who) {
  static const char* const what[4] = {"q_positions", "k_positions", "q_sequence_ids", "k_sequence_ids"};
  const int64_t seq[4] = {s.Sq, s.Sk, s.Sq, s.Sk};
  bool versioned = true;
  for (int i = 0; i < 4; ++i) {
    const OptTensor& t = ids.given[i];
    TORCH_CHECK_VALUE(t.has_value() && t->defined(), "document-masked attention needs q/k positions and q/k sequence ids");
    TORCH_CHECK_VALUE(t->dim() == 2 && t->size(0) == s.B && t->size(1) == seq[i], what[i], " must have shape (", s.B, ", ", seq[i], "), got ",
                      t->sizes());
    versioned = versioned && !t->is_inference();  // (inference tensors carry no version counter)
  }
  auto convert = [&] {
    for (int i = 0; i < 4; ++i) {
      int same = i;
      while (same > 0 && !ids.given[same - 1]->is_same(*ids.given[i])) --same;
      ids.used[i] = same > 0 ? ids.used[same - 1] : ids32(ids.given[i], s.B, seq[i], what[i]);
    }
    point_at_ids(s, ids);
    check_supported(s, who);
  };
  // (a captured graph must rebuild the plan on every replay: its id buffers are refilled in place)
  if (plan_cache_entries == 0 || !versioned || stream_is_capturing()) {
    convert();
    return Tensor();
  }
  const PlanKey key = plan_key(s, ids, q);
  if (const std::shared_ptr<const PlanEntry> kept = find_plan(key)) {
    for (int i = 0; i < 4; ++i) ids.used[i] = kept->ids.used[i];
    point_at_ids(s, ids);
    check_supported(s, who);
    if (kept->plan.defined()) s.doc_plan = kept->plan.const_data_ptr();
    return kept->plan;
  }
  convert();
  const int64_t bytes = mlts_attn_doc_plan_bytes(&s);
  if (bytes <= 0 || bytes > kPlanCacheBytes) {
    bool converted = false;
    for (int i = 0; i < 4; ++i) converted = converted || !ids.used[i]->is_same(*ids.given[i]);
    if (converted) keep_plan(std::make_shared<const PlanEntry>(PlanEntry{key, ids, Tensor()}));
    return Tensor();
  }
  Tensor plan = workspace(bytes, q);
  check(mlts_attn_doc_plan(&s, mptr(plan), bytes, current_stream()));
  keep_plan(std::make_shared<const PlanEntry>(PlanEntry{key, ids, plan}));
  s.doc_plan = plan.const_data_ptr();
  return plan;
}

mlts_attn_shape attn_shape(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, int64_t mask_mode, double scale) {
  mlts_attn_shape s{};
  s.B = q.size(0), s.Hq = q.size(1), s.Sq = q.size(2), s.D = q.size(3);
  s.Hkv = k.size(1), s.Sk = k.size(2);
  s.dtype = dtype_code(q);
  s.mask_mode = mask_mode;
  s.scale = scale;
  for (int i = 0; i < 3; ++i) {
    s.q_stride[i] = q.stride(i);
    s.k_stride[i] = k.stride(i);
    s.v_stride[i] = v.stride(i);
    s.o_stride[i] = o.stride(i);
  }
  return s;
}

}  // namespace

std::tuple<Tensor, Tensor> attention_forward(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, int64_t mask_mode, double scale,
                                             const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  check_attn_inputs(q_in, k_in, v_in);
  for (const Tensor* t : {&q_in, &k_in, &v_in}) require_gpu(*t);
  for (const OptTensor* t : {&q_pos, &k_pos, &q_seq, &k_seq}) require_gpu(*t);
  const Tensor q = dense_last(q_in), k = dense_last(k_in), v = dense_last(v_in);
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3);
  Tensor o = bshd_empty(B, Hq, Sq, D, q.options());
  Tensor lse = at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));
  if (B == 0 || Sq == 0) return {o, lse};
  mlts_attn_shape s = attn_shape(q, k, v, o, mask_mode, scale);
  Ids ids{{q_pos, k_pos, q_seq, k_seq}, {}};
  Tensor plan;
  if (mask_mode == MLTS_MASK_DOC) plan = attach_document_ids(s, ids, q, "attention_forward");
  else check_supported(s, "attention_forward");
  const int64_t ws_bytes = mlts_attn_fwd_workspace_bytes(&s);
  Tensor ws = workspace(ws_bytes, q);
  check(mlts_attn_fwd(&s, ptr(q), ptr(k), ptr(v), mptr(o), lse.mutable_data_ptr<float>(), ws.defined() ? mptr(ws) : nullptr, ws_bytes,
                      current_stream()));
  return {o, lse};
}

namespace {

// dq / dk / dv written or added to as `mode` (MLTS_BWD_*) says
void attention_backward_into(const Tensor& dout_in, const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& o_in,
                             const Tensor& lse_in, Tensor& dq, Tensor& dk, Tensor& dv, int mode, int64_t mask_mode, double scale,
                             const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq, const RotatedBy* rotated = nullptr) {
  check_attn_inputs(q_in, k_in, v_in);
  for (const Tensor* t : {&dout_in, &q_in, &k_in, &v_in, &o_in, &lse_in}) require_gpu(*t);
  for (const Tensor* t : {&dq, &dk, &dv}) require_gpu(*t);
  for (const OptTensor* t : {&q_pos, &k_pos, &q_seq, &k_seq}) require_gpu(*t);
  const Tensor q = dense_last(q_in), k = dense_last(k_in), v = dense_last(v_in), o = dense_last(o_in), dout = dense_last(dout_in);
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), Sk = k.size(2);
  if (B == 0 || Sq == 0 || Sk == 0) {
    if (mode == MLTS_BWD_OVERWRITE || mode == MLTS_BWD_DQ_STORE) dq.zero_();
    if (mode != MLTS_BWD_ACCUMULATE) dk.zero_(), dv.zero_();
    return;
  }
  TORCH_CHECK_VALUE(dout.sizes() == q.sizes() && o.sizes() == q.sizes(), "dout and out must have the shape of q");
  TORCH_CHECK_VALUE(lse_in.dim() == 3 && lse_in.size(0) == B && lse_in.size(1) == Hq && lse_in.size(2) == Sq && lse_in.scalar_type() == at::kFloat,
                    "softmax_lse must be float32 of shape (", B, ", ", Hq, ", ", Sq, "), got ", lse_in.scalar_type(), " ", lse_in.sizes());
  const Tensor lse = dense(lse_in);
  mlts_attn_shape s = attn_shape(q, k, v, o, mask_mode, scale);
  Ids ids{{q_pos, k_pos, q_seq, k_seq}, {}};
  Tensor plan;
  if (mask_mode == MLTS_MASK_DOC) plan = attach_document_ids(s, ids, q, "attention_backward");
  else check_supported(s, "attention_backward");
  const int64_t ws_bytes = mlts_attn_bwd_workspace_bytes(&s, mode);
  Tensor ws = workspace(ws_bytes, q);
  const Strides3 dos(dout), dqs(dq), dks(dk), dvs(dv);
  if (rotated) {
    require_gpu(rotated->cos), require_gpu(rotated->sin), require_gpu(rotated->positions);
    check_tables(q, rotated->cos, rotated->sin);
    const Tensor cos = dense(rotated->cos), sin = dense(rotated->sin);
    const OptTensor pos = ids32(rotated->positions, B, Sq, "position_ids");
    const mlts_attn_rotation r{ptr(cos), ptr(sin), ids_ptr(pos), static_cast<int32_t>(cos.size(0)), static_cast<int32_t>(rotated->offset)};
    check(mlts_attn_bwd_rope(&s, ptr(dout), dos.v, ptr(q), ptr(k), ptr(v), ptr(o), lse.const_data_ptr<float>(), mptr(dq), dqs.v, mptr(dk), dks.v,
                             mptr(dv), dvs.v, &r, ws.defined() ? mptr(ws) : nullptr, ws_bytes, current_stream()));
    return;
  }
  check(mlts_attn_bwd(&s, ptr(dout), dos.v, ptr(q), ptr(k), ptr(v), ptr(o), lse.const_data_ptr<float>(), mptr(dq), dqs.v, mptr(dk), dks.v,
                      mptr(dv), dvs.v, mode, ws.defined() ? mptr(ws) : nullptr, ws_bytes, current_stream()));
}

// dq, dk, dv in the input dtype, as [B, H, S, D] views of [B, S, H, D] storage.  For self-attention (queries and keys of
// one length) the three are the head ranges [0, Hq), [Hq, Hq + Hkv), [Hq + Hkv, Hq + 2 Hkv) of ONE [B, S, Hq + 2 Hkv, D]
// buffer: next to each other exactly as the input gradient of projections that run as one product wants them.
std::tuple<Tensor, Tensor, Tensor> attention_gradients(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                      const Tensor& lse, int64_t mask_mode, double scale, const OptTensor& q_pos,
                                                      const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq,
                                                       const RotatedBy* rotated) {
  check_attn_inputs(q, k, v);
  require_gpu(q);
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3), Hkv = k.size(1), Sk = k.size(2);
  Tensor dq, dk, dv;
  if (Sk == Sq) {
    const int64_t H = Hq + 2 * Hkv;
    Tensor joint = at::empty({B * Sq * H * D}, q.options());
    const int64_t strides[4] = {Sq * H * D, D, H * D, 1};
    dq = joint.as_strided({B, Hq, Sq, D}, strides, 0);
    dk = joint.as_strided({B, Hkv, Sq, D}, strides, Hq * D);
    dv = joint.as_strided({B, Hkv, Sq, D}, strides, (Hq + Hkv) * D);
  } else {
    dq = bshd_empty(B, Hq, Sq, D, q.options());
    dk = bshd_empty(B, Hkv, Sk, D, k.options());
    dv = bshd_empty(B, Hkv, Sk, D, v.options());
  }
  attention_backward_into(dout, q, k, v, o, lse, dq, dk, dv, MLTS_BWD_OVERWRITE, mask_mode, scale, q_pos, k_pos, q_seq, k_seq, rotated);
  return {dq, dk, dv};
}

}  // namespace

std::tuple<Tensor, Tensor, Tensor> attention_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                      const Tensor& lse, int64_t mask_mode, double scale, const OptTensor& q_pos,
                                                      const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  return attention_gradients(dout, q, k, v, o, lse, mask_mode, scale, q_pos, k_pos, q_seq, k_seq, nullptr);
}
std::tuple<Tensor, Tensor, Tensor> rotated_attention_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                              const Tensor& lse, int64_t mask_mode, double scale, const OptTensor& q_pos,
                                                              const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq, const RotatedBy& rotated) {
  return attention_gradients(dout, q, k, v, o, lse, mask_mode, scale, q_pos, k_pos, q_seq, k_seq, &rotated);
}

namespace {

void attention_backward_accumulate(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
                                   Tensor dq, Tensor dk, Tensor dv, int64_t mask_mode, std::optional<double> scale, const OptTensor& q_pos,
                                   const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  const Tensor* grads[3] = {&dq, &dk, &dv};
  const Tensor* refs[3] = {&q, &k, &v};
  static const char* const names[3] = {"dq", "dk", "dv"};
  for (int i = 0; i < 3; ++i)
    TORCH_CHECK_VALUE(grads[i]->scalar_type() == at::kFloat && grads[i]->sizes() == refs[i]->sizes() && grads[i]->stride(-1) == 1, names[i],
                      " must be float32 with the shape of its input and a contiguous head_dim");
  at::NoGradGuard no_grad;
  attention_backward_into(dout, q, k, v, o, lse, dq, dk, dv, MLTS_BWD_ACCUMULATE, mask_mode, resolve_scale(scale, q), q_pos, k_pos, q_seq, k_seq);
}

void attention_backward_ring_block(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
                                   Tensor dq, Tensor dk, Tensor dv, bool first, int64_t mask_mode, std::optional<double> scale,
                                   const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  TORCH_CHECK_VALUE(dq.scalar_type() == at::kFloat && dq.sizes() == q.sizes() && dq.stride(-1) == 1,
                    "dq must be float32 with the shape of q and a contiguous head_dim");
  const Tensor* grads[2] = {&dk, &dv};
  const Tensor* refs[2] = {&k, &v};
  for (int i = 0; i < 2; ++i)
    TORCH_CHECK_VALUE(grads[i]->scalar_type() == refs[i]->scalar_type() && grads[i]->sizes() == refs[i]->sizes() && grads[i]->stride(-1) == 1,
                      i ? "dv" : "dk", " must have the dtype and shape of its input and a contiguous head_dim");
  at::NoGradGuard no_grad;
  attention_backward_into(dout, q, k, v, o, lse, dq, dk, dv, first ? MLTS_BWD_DQ_STORE : MLTS_BWD_DQ_ACCUMULATE, mask_mode,
                          resolve_scale(scale, q), q_pos, k_pos, q_seq, k_seq);
}

void attention_merge_(Tensor out_acc, Tensor lse_acc, const Tensor& o_blk_in, const Tensor& lse_blk_in, int64_t q_off) {
  for (const Tensor* t : {&out_acc, &lse_acc}) require_gpu(*t);
  for (const Tensor* t : {&o_blk_in, &lse_blk_in}) require_gpu(*t);
  TORCH_CHECK_VALUE(out_acc.scalar_type() == at::kFloat && lse_acc.scalar_type() == at::kFloat && out_acc.is_contiguous() && lse_acc.is_contiguous(),
                    "running_out / running_lse must be contiguous float32");
  TORCH_CHECK_VALUE(out_acc.dim() == 4 && o_blk_in.dim() == 4 && lse_blk_in.dim() == 3 && lse_acc.dim() == 3,
                    "block shapes do not match the running state");
  const int64_t B = out_acc.size(0), H = out_acc.size(1), S = out_acc.size(2), D = out_acc.size(3), q_len = o_blk_in.size(2);
  TORCH_CHECK_VALUE(o_blk_in.sizes() == at::IntArrayRef({B, H, q_len, D}) && lse_blk_in.sizes() == at::IntArrayRef({B, H, q_len}) &&
                        lse_acc.sizes() == at::IntArrayRef({B, H, S}),
                    "block shapes do not match the running state");
  const Tensor o_blk = dense_last(o_blk_in), lse_blk = lse_blk_in.to(at::kFloat).contiguous();
  const Strides3 os(o_blk);
  check(mlts_attn_merge(out_acc.mutable_data_ptr<float>(), lse_acc.mutable_data_ptr<float>(), ptr(o_blk), os.v, dtype_code(o_blk),
                        lse_blk.const_data_ptr<float>(), B, H, S, D, q_off, q_len, current_stream()));
}

// ---- RMSNorm --------------------------------------------------------------------------------------------------------
void check_norm_weight(const Tensor& x, const Tensor& w) {
  TORCH_CHECK_VALUE(w.dim() == 1 && w.size(0) == x.size(-1) && w.scalar_type() == x.scalar_type(),
                    "RMSNorm weight must be [hidden] with the dtype of x");
}
int64_t rows_of(const Tensor& x) { return x.size(-1) ? x.numel() / x.size(-1) : 0; }

std::tuple<Tensor, Tensor> rmsnorm_fwd(const Tensor& x_in, const Tensor& w_in, double eps) {
  require_gpu(x_in), require_gpu(w_in);
  check_norm_weight(x_in, w_in);
  const Tensor x = dense(x_in), w = dense(w_in);
  const int64_t rows = rows_of(x);
  Tensor y = at::empty(x.sizes(), x.options());
  Tensor rstd = at::empty({rows}, x.options().dtype(at::kFloat));
  check(mlts_rmsnorm_fwd(ptr(x), ptr(w), mptr(y), rstd.mutable_data_ptr<float>(), rows, x.size(-1), eps, dtype_code(x), current_stream()));
  return {y, rstd};
}

std::tuple<Tensor, Tensor> rmsnorm_bwd(const Tensor& dy_in, const Tensor& x_in, const Tensor& w_in, const Tensor& rstd) {
  for (const Tensor* t : {&dy_in, &x_in, &w_in, &rstd}) require_gpu(*t);
  const Tensor x = dense(x_in), dy = dense(dy_in), w = dense(w_in);
  const int64_t rows = rows_of(x), hidden = x.size(-1);
  Tensor dx = at::empty(x.sizes(), x.options()), dw = at::empty(w.sizes(), w.options());
  if (rows == 0) return {dx, dw.zero_()};
  const int64_t ws_bytes = mlts_rmsnorm_bwd_workspace_bytes(rows, hidden);
  Tensor ws = workspace(ws_bytes, x);
  check(mlts_rmsnorm_bwd(ptr(dy), ptr(x), ptr(w), rstd.const_data_ptr<float>(), mptr(dx), mptr(dw), mptr(ws), ws_bytes, rows, hidden,
                         dtype_code(x), current_stream()));
  return {dx, dw};
}

std::tuple<Tensor, Tensor, Tensor> add_rmsnorm_fwd(const Tensor& x_in, const Tensor& res_in, const Tensor& w_in, double eps) {
  for (const Tensor* t : {&x_in, &res_in, &w_in}) require_gpu(*t);
  check_norm_weight(x_in, w_in);
  TORCH_CHECK_VALUE(res_in.sizes() == x_in.sizes() && res_in.scalar_type() == x_in.scalar_type(), "the residual must have the shape and dtype of x");
  const Tensor x = dense(x_in), res = dense(res_in), w = dense(w_in);
  const int64_t rows = rows_of(x);
  Tensor h = at::empty(x.sizes(), x.options()), y = at::empty(x.sizes(), x.options());
  Tensor rstd = at::empty({rows}, x.options().dtype(at::kFloat));
  check(mlts_add_rmsnorm_fwd(ptr(x), ptr(res), mptr(h), ptr(w), mptr(y), rstd.mutable_data_ptr<float>(), rows, x.size(-1), eps, dtype_code(x),
                             current_stream()));
  return {h, y, rstd};
}

std::tuple<Tensor, Tensor> add_rmsnorm_bwd(const Tensor& dy_in, const Tensor& dres_in, const Tensor& h_in, const Tensor& w_in, const Tensor& rstd) {
  for (const Tensor* t : {&dy_in, &dres_in, &h_in, &w_in, &rstd}) require_gpu(*t);
  const Tensor h = dense(h_in), dy = dense(dy_in), dres = dense(dres_in), w = dense(w_in);
  const int64_t rows = rows_of(h), hidden = h.size(-1);
  Tensor dx = at::empty(h.sizes(), h.options()), dw = at::empty(w.sizes(), w.options());
  if (rows == 0) return {dx, dw.zero_()};
  const int64_t ws_bytes = mlts_rmsnorm_bwd_workspace_bytes(rows, hidden);
  Tensor ws = workspace(ws_bytes, h);
  check(mlts_add_rmsnorm_bwd(ptr(dy), ptr(h), ptr(w), rstd.const_data_ptr<float>(), ptr(dres), mptr(dx), mptr(dw), mptr(ws), ws_bytes, rows,
                             hidden, dtype_code(h), current_stream()));
  return {dx, dw};
}

// dx, with dw added onto the gradient buffer the weight already owns; dres may be undefined
Tensor rmsnorm_bwd_into(const Tensor& dy_in, const Tensor& dres_in, const Tensor& x_in, const Tensor& w_in, const Tensor& rstd, Tensor grad) {
  const Tensor x = dense(x_in), dy = dense(dy_in), w = dense(w_in), dres = dres_in.defined() ? dense(dres_in) : dres_in;
  const int64_t rows = rows_of(x), hidden = x.size(-1);
  Tensor dx = at::empty(x.sizes(), x.options());
  if (rows == 0) return dx;
  const int64_t ws_bytes = mlts_rmsnorm_bwd_workspace_bytes(rows, hidden);
  Tensor ws = workspace(ws_bytes, x);
  check(mlts_rmsnorm_bwd_accumulate(ptr(dy), ptr(x), ptr(w), rstd.const_data_ptr<float>(), dres.defined() ? ptr(dres) : nullptr, mptr(dx), mptr(grad),
                                    mptr(ws), ws_bytes, rows, hidden, dtype_code(x), current_stream()));
  return dx;
}

// ---- RoPE -----------------------------------------------------------------------------------------------------------
Tensor rope(const Tensor& x_in, const Tensor& cos_in, const Tensor& sin_in, const OptTensor& positions, int64_t position_offset, bool inverse) {
  for (const Tensor* t : {&x_in, &cos_in, &sin_in}) require_gpu(*t);
  require_gpu(positions);
  TORCH_CHECK_VALUE(x_in.dim() == 4, "rope expects [batch, heads, seq, head_dim]");
  check_tables(x_in, cos_in, sin_in);
  const Tensor x = dense_last(x_in), cos = dense(cos_in), sin = dense(sin_in);
  Tensor y = at::empty_like(x);  // keeps the (possibly transposed) layout of x
  const OptTensor pos = ids32(positions, x.size(0), x.size(2), "position_ids");
  const Strides3 xs(x), ys(y);
  check(mlts_rope(ptr(x), xs.v, mptr(y), ys.v, ptr(cos), ptr(sin), cos.size(0), ids_ptr(pos), position_offset, x.size(0), x.size(1), x.size(2),
                  x.size(3), dtype_code(x), inverse, current_stream()));
  return y;
}

std::tuple<Tensor, Tensor> rope_pair_op(const Tensor& xa, const Tensor& xb, const Tensor& cos, const Tensor& sin, const OptTensor& positions,
                                        int64_t position_offset, bool inverse) {
  return rope_pair(xa, xb, cos, sin, positions, position_offset, inverse, false);
}

void rope_pair_(const Tensor& xa, const Tensor& xb, const Tensor& cos, const Tensor& sin, const OptTensor& positions, int64_t position_offset,
                bool inverse) {
  rope_pair(xa, xb, cos, sin, positions, position_offset, inverse, true);
}

}  // namespace

std::tuple<Tensor, Tensor> rope_pair(const Tensor& xa_in, const Tensor& xb_in, const Tensor& cos_in, const Tensor& sin_in,
                                     const OptTensor& positions, int64_t position_offset, bool inverse, bool in_place) {
  for (const Tensor* t : {&xa_in, &xb_in, &cos_in, &sin_in}) require_gpu(*t);
  require_gpu(positions);
  TORCH_CHECK_VALUE(xa_in.dim() == 4 && xb_in.dim() == 4 && xa_in.size(0) == xb_in.size(0) && xa_in.size(2) == xb_in.size(2) &&
                        xa_in.size(3) == xb_in.size(3) && xa_in.scalar_type() == xb_in.scalar_type(),
                    "rope_pair expects two [batch, heads, seq, head_dim] tensors that differ only in heads");
  check_tables(xa_in, cos_in, sin_in);
  TORCH_CHECK_VALUE(!in_place || (xa_in.stride(-1) == 1 && xb_in.stride(-1) == 1), "rope_pair_: the head_dim of both tensors must be contiguous");
  const Tensor xa = dense_last(xa_in), xb = dense_last(xb_in), cos = dense(cos_in), sin = dense(sin_in);
  Tensor ya = in_place ? xa : at::empty_like(xa), yb = in_place ? xb : at::empty_like(xb);
  const OptTensor pos = ids32(positions, xa.size(0), xa.size(2), "position_ids");
  const Strides3 xas(xa), xbs(xb), yas(ya), ybs(yb);
  check(mlts_rope_pair(ptr(xa), xas.v, mptr(ya), yas.v, xa.size(1), ptr(xb), xbs.v, mptr(yb), ybs.v, xb.size(1), ptr(cos), ptr(sin),
                       cos.size(0), ids_ptr(pos), position_offset, xa.size(0), xa.size(2), xa.size(3), dtype_code(xa), inverse,
                       current_stream()));
  return {ya, yb};
}

// ---- SwiGLU ---------------------------------------------------------------------------------------------------------
namespace {

Tensor swiglu_fwd(const Tensor& gate_in, const Tensor& up_in) {
  require_gpu(gate_in), require_gpu(up_in);
  TORCH_CHECK_VALUE(gate_in.sizes() == up_in.sizes() && gate_in.scalar_type() == up_in.scalar_type(), "gate and up must match in shape and dtype");
  const Tensor gate = dense(gate_in), up = dense(up_in);
  Tensor h = at::empty(gate.sizes(), gate.options());
  check(mlts_swiglu_fwd(ptr(gate), ptr(up), mptr(h), gate.numel(), dtype_code(gate), current_stream()));
  return h;
}

std::tuple<Tensor, Tensor> swiglu_bwd(const Tensor& dh_in, const Tensor& gate_in, const Tensor& up_in) {
  for (const Tensor* t : {&dh_in, &gate_in, &up_in}) require_gpu(*t);
  const Tensor dh = dense(dh_in), gate = dense(gate_in), up = dense(up_in);
  Tensor dg = at::empty(gate.sizes(), gate.options()), du = at::empty(gate.sizes(), gate.options());
  check(mlts_swiglu_bwd(ptr(dh), ptr(gate), ptr(up), mptr(dg), mptr(du), gate.numel(), dtype_code(gate), current_stream()));
  return {dg, du};
}

const char* column(const Tensor& t, int64_t col) { return static_cast<const char*>(t.const_data_ptr()) + col * t.element_size(); }

}  // namespace

// round(silu(gate)) * up where gate = gu[..., gate_col : gate_col + cols] and up = gu[..., up_col : up_col + cols] are
// column blocks of one contiguous [..., width] projection output (no autograd: used inside the fused MLP formula)
Tensor swiglu_rows(const Tensor& gu, int64_t gate_col, int64_t up_col, int64_t cols) {
  require_gpu(gu);
  TORCH_CHECK_VALUE(gu.is_contiguous(), "swiglu_rows expects a contiguous projection output");
  const int64_t width = gu.size(-1), rows = gu.numel() / width;
  c10::SmallVector<int64_t, 5> shape(gu.sizes().begin(), gu.sizes().end());
  shape.back() = cols;
  Tensor h = at::empty(shape, gu.options());
  check(mlts_swiglu_fwd_rows(column(gu, gate_col), column(gu, up_col), width, mptr(h), cols, rows, cols, dtype_code(gu), current_stream()));
  return h;
}

// d gate and d up of swiglu_rows, written into the same column blocks of a buffer shaped like `gu`; its other columns, if
// there are any, are zero
Tensor swiglu_rows_backward(const Tensor& dh_in, const Tensor& gu, int64_t gate_col, int64_t up_col, int64_t cols) {
  require_gpu(dh_in), require_gpu(gu);
  const Tensor dh = dense(dh_in);
  const int64_t width = gu.size(-1), rows = gu.numel() / width;
  Tensor dgu = width == 2 * cols ? at::empty(gu.sizes(), gu.options()) : at::zeros(gu.sizes(), gu.options());
  check(mlts_swiglu_bwd_rows(ptr(dh), cols, column(gu, gate_col), column(gu, up_col), width, const_cast<char*>(column(dgu, gate_col)),
                             const_cast<char*>(column(dgu, up_col)), width, rows, cols, dtype_code(gu), current_stream()));
  return dgu;
}

// ---- cross-entropy --------------------------------------------------------------------------------------------------
namespace {

// overwrite: the gradient replaces the logits in their own buffer (they must be contiguous)
std::tuple<Tensor, Tensor, Tensor> ce_fwd_bwd(const Tensor& logits, const Tensor& labels, int64_t ignore_index, bool overwrite) {
  require_gpu(logits), require_gpu(labels);
  const Tensor lg = dense(logits);
  const int64_t vocab = lg.size(-1), rows = rows_of(lg);
  const Tensor lb = dense(labels.scalar_type() == at::kLong ? labels : labels.to(at::kLong));
  TORCH_CHECK_VALUE(lb.numel() == rows, "labels (", lb.numel(), ") do not match logits rows (", rows, ")");
  TORCH_CHECK_VALUE(!overwrite || lg.is_same(logits), "cross_entropy(overwrite_logits=True) needs contiguous logits");
  Tensor dlogits = overwrite ? lg : at::empty(lg.sizes(), lg.options());
  Tensor loss = at::empty({}, lg.options().dtype(at::kFloat)), count = at::empty({}, lg.options().dtype(at::kInt));
  const int64_t ws_bytes = mlts_ce_workspace_bytes(rows);
  Tensor ws = workspace(ws_bytes, lg);
  check(mlts_ce_fwd_bwd(ptr(lg), lb.const_data_ptr<int64_t>(), mptr(dlogits), loss.mutable_data_ptr<float>(), count.mutable_data_ptr<int32_t>(),
                        mptr(ws), ws_bytes, rows, vocab, ignore_index, dtype_code(lg), current_stream()));
  return {loss, dlogits, count};
}

std::tuple<Tensor, Tensor, Tensor> ce_fwd_bwd_op(const Tensor& logits, const Tensor& labels, int64_t ignore_index) {
  return ce_fwd_bwd(logits, labels, ignore_index, false);
}

void scale_by_scalar_(const Tensor& x, const Tensor& scale) {
  require_gpu(x), require_gpu(scale);
  TORCH_CHECK_VALUE(x.is_contiguous(), "scale_by_scalar_ needs a contiguous tensor");
  const Tensor s = scale.to(at::kFloat).contiguous();
  TORCH_CHECK_VALUE(s.numel() == 1, "scale_by_scalar_ needs a single scale");
  check(mlts_scale_by_device_scalar(mptr(x), s.const_data_ptr<float>(), x.numel(), dtype_code(x), current_stream()));
}

Tensor scale_by_scalar(const Tensor& x, const Tensor& scale) {
  require_gpu(x), require_gpu(scale);
  Tensor out = dense(x).clone();
  scale_by_scalar_(out, scale);
  return out;
}

// ---- optimizer-step launches (in place, no autograd) ------------------------------------------------------------------
const Tensor& flat_f32(const Tensor& t, const char* what) {
  TORCH_CHECK_VALUE(t.scalar_type() == at::kFloat && t.is_contiguous(), what, " must be a contiguous float32 tensor");
  return t;
}

void adamw_step_(const Tensor& p, const Tensor& g, const Tensor& m, const Tensor& v, double lr, double beta1, double beta2, double eps,
                 double weight_decay, int64_t step, const OptTensor& p_lowp, double grad_scale, const OptTensor& sq_norm, double max_norm) {
  for (const Tensor* t : {&p, &g, &m, &v}) require_gpu(*t);
  require_gpu(p_lowp), require_gpu(sq_norm);
  const Tensor* all[4] = {&p, &g, &m, &v};
  static const char* const names[4] = {"param", "grad", "exp_avg", "exp_avg_sq"};
  for (int i = 0; i < 4; ++i) {
    flat_f32(*all[i], names[i]);
    TORCH_CHECK_VALUE(all[i]->numel() == p.numel(), "param, grad, exp_avg, exp_avg_sq must have the same number of elements");
  }
  TORCH_CHECK_VALUE(!p_lowp.has_value() || (p_lowp->scalar_type() == at::kBFloat16 && p_lowp->numel() == p.numel() && p_lowp->is_contiguous()),
                    "p_lowp must be a contiguous bfloat16 tensor matching param");
  TORCH_CHECK_VALUE(!sq_norm.has_value() || (sq_norm->scalar_type() == at::kDouble && sq_norm->numel() == 1), "sq_norm must be a float64 scalar tensor");
  TORCH_CHECK_VALUE(step >= 1, "step is the 1-based optimizer step count");
  check(mlts_adamw_step(static_cast<float*>(mptr(p)), static_cast<const float*>(ptr(g)), static_cast<float*>(mptr(m)),
                        static_cast<float*>(mptr(v)), p_lowp.has_value() ? mptr(*p_lowp) : nullptr, p.numel(), lr, beta1, beta2, eps,
                        weight_decay, step, grad_scale, static_cast<const double*>(ptr(sq_norm)), max_norm, current_stream()));
}

constexpr int64_t kSqNormWorkspace = 16384;

Tensor sq_norm(const Tensor& x, const OptTensor& out_in) {
  require_gpu(x), require_gpu(out_in);
  flat_f32(x, "x");
  Tensor out = out_in.has_value() ? *out_in : at::empty({}, x.options().dtype(at::kDouble));
  Tensor ws = workspace(kSqNormWorkspace, x);
  check(mlts_sq_norm(static_cast<const float*>(ptr(x)), x.numel(), out.mutable_data_ptr<double>(), mptr(ws), current_stream()));
  return out;
}

Tensor scale_(const Tensor& x, double scale) {
  require_gpu(x);
  flat_f32(x, "x");
  check(mlts_scale(static_cast<float*>(mptr(x)), scale, x.numel(), current_stream()));
  return x;
}

// the same passes over lists of tensors
struct FlatList {
  std::vector<void*> ptrs;
  std::vector<int64_t> sizes;
  FlatList(const std::vector<Tensor>& ts, const char* what) {
    for (const Tensor& t : ts) {
      require_gpu(t);
      flat_f32(t, what);
      ptrs.push_back(mptr(t));
      sizes.push_back(t.numel());
    }
  }
};

Tensor list_sq_norm(const std::vector<Tensor>& xs) {
  TORCH_CHECK_VALUE(!xs.empty(), "no tensors");
  const FlatList l(xs, "x");
  Tensor out = at::empty({}, xs[0].options().dtype(at::kDouble));
  const int64_t bytes = mlts_list_sq_norm_workspace_bytes(l.sizes.data(), l.sizes.size());
  Tensor ws = workspace(bytes, xs[0]);
  check(mlts_list_sq_norm(reinterpret_cast<const float* const*>(l.ptrs.data()), l.sizes.data(), l.sizes.size(), out.mutable_data_ptr<double>(),
                          mptr(ws), bytes, current_stream()));
  return out;
}

void list_scale_(const std::vector<Tensor>& xs, double scale) {
  const FlatList l(xs, "x");
  check(mlts_list_scale(reinterpret_cast<float* const*>(l.ptrs.data()), l.sizes.data(), l.sizes.size(), scale, current_stream()));
}

void list_adamw_step_(const std::vector<Tensor>& p, const std::vector<Tensor>& g, const std::vector<Tensor>& m, const std::vector<Tensor>& v, double lr,
                      double beta1, double beta2, double eps, double weight_decay, int64_t step, const OptTensor& sq_norm, double max_norm) {
  require_gpu(sq_norm);
  TORCH_CHECK_VALUE(!sq_norm.has_value() || (sq_norm->scalar_type() == at::kDouble && sq_norm->numel() == 1), "sq_norm must be a float64 scalar tensor");
  const FlatList lp(p, "param"), lg(g, "grad"), lm(m, "exp_avg"), lv(v, "exp_avg_sq");
  TORCH_CHECK_VALUE(lp.sizes == lg.sizes && lp.sizes == lm.sizes && lp.sizes == lv.sizes,
                    "param, grad, exp_avg, exp_avg_sq must have the same number of elements");
  check(mlts_list_adamw_step(reinterpret_cast<float* const*>(lp.ptrs.data()), reinterpret_cast<const float* const*>(lg.ptrs.data()),
                             reinterpret_cast<float* const*>(lm.ptrs.data()), reinterpret_cast<float* const*>(lv.ptrs.data()), lp.sizes.data(),
                             lp.sizes.size(), lr, beta1, beta2, eps, weight_decay, step, 1.0, static_cast<const double*>(ptr(sq_norm)), max_norm,
                             current_stream()));
}

Tensor grad_to_f32_(const Tensor& dst, const Tensor& src, bool accumulate, const OptTensor& sq_out) {
  require_gpu(dst), require_gpu(src), require_gpu(sq_out);
  flat_f32(dst, "dst");
  TORCH_CHECK_VALUE(src.numel() == dst.numel() && src.is_contiguous(), "src must be contiguous and match dst in size");
  Tensor ws = sq_out.has_value() ? workspace(kSqNormWorkspace, dst) : Tensor();
  check(mlts_grad_to_f32(static_cast<float*>(mptr(dst)), ptr(src), dtype_code(src), dst.numel(), accumulate,
                         sq_out.has_value() ? sq_out->mutable_data_ptr<double>() : nullptr, ws.defined() ? mptr(ws) : nullptr, current_stream()));
  return dst;
}

}  // namespace

// parts [slices, ...] -> sum over the slices, added in fp32 and rounded once, into `out` (added onto it: accumulate)
Tensor grad_sum_slices(const Tensor& parts, const OptTensor& out_in, bool accumulate) {
  require_gpu(parts), require_gpu(out_in);
  TORCH_CHECK_VALUE(parts.dim() >= 2 && parts.is_contiguous(), "parts must be a contiguous tensor [slices, ...]");
  TORCH_CHECK_VALUE(out_in.has_value() || !accumulate, "accumulate=True needs an output tensor");
  const at::IntArrayRef shape = parts.sizes().slice(1);
  TORCH_CHECK_VALUE(!out_in.has_value() || (out_in->scalar_type() == parts.scalar_type() && out_in->sizes() == shape && out_in->is_contiguous()),
                    "out must be contiguous with the dtype and the per-slice shape of parts");
  Tensor out = out_in.has_value() ? *out_in : at::empty(shape, parts.options());
  check(mlts_grad_sum_slices(mptr(out), ptr(parts), dtype_code(parts), parts.size(0), out.numel(), accumulate, current_stream()));
  return out;
}

// ---- autograd -------------------------------------------------------------------------------------------------------
namespace {

using torch::autograd::collect_next_edges;
using torch::autograd::compute_requires_grad;
using torch::autograd::set_history;

// The operator of this name, called through the dispatcher: formulas below run on whatever backend or tracing mode the
// tensors bring.
#define MALTOS_OP(name, fn)                                                                              \
  const auto& name() {                                                                                   \
    static const auto handle =                                                                           \
        c10::Dispatcher::singleton().findSchemaOrThrow("maltos::" #name, "").typed<decltype(fn)>();      \
    return handle;                                                                                       \
  }
namespace op {
MALTOS_OP(attn_fwd, attention_forward)
MALTOS_OP(attn_bwd, attention_backward)
MALTOS_OP(rmsnorm_fwd, maltos::rmsnorm_fwd)
MALTOS_OP(rmsnorm_bwd, maltos::rmsnorm_bwd)
MALTOS_OP(add_rmsnorm_fwd, maltos::add_rmsnorm_fwd)
MALTOS_OP(add_rmsnorm_bwd, maltos::add_rmsnorm_bwd)
MALTOS_OP(rope, maltos::rope)
MALTOS_OP(rope_pair, maltos::rope_pair_op)
MALTOS_OP(swiglu_fwd, maltos::swiglu_fwd)
MALTOS_OP(swiglu_bwd, maltos::swiglu_bwd)
MALTOS_OP(ce_fwd_bwd, maltos::ce_fwd_bwd_op)
MALTOS_OP(scale_by_scalar_, maltos::scale_by_scalar_)
}  // namespace op
#undef MALTOS_OP

struct AttnBackward final : Formula {
  enum { Q, K, V, O, LSE, IDS, COUNT = IDS + 4 };
  int64_t mask_mode = 0;
  double scale = 0;
  AttnBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosAttnBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    const Tensor dout = g[0].defined() ? g[0] : at::zeros_like(s[O]);
    auto [dq, dk, dv] = op::attn_bwd().call(dout, s[Q], s[K], s[V], s[O], s[LSE], mask_mode, scale, optional_tensor(s[IDS]),
                                            optional_tensor(s[IDS + 1]), optional_tensor(s[IDS + 2]), optional_tensor(s[IDS + 3]));
    return {dq, dk, dv};
  }
};

std::tuple<Tensor, Tensor> attn_fwd_autograd(const Tensor& q, const Tensor& k, const Tensor& v, int64_t mask_mode, double scale,
                                             const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  refuse_tangents("attn_fwd", q, k, v);
  std::shared_ptr<AttnBackward> fn;
  if (compute_requires_grad(q, k, v)) {
    fn = make_formula<AttnBackward>();
    fn->set_next_edges(collect_next_edges(q, k, v));
    fn->save(fn->Q, q), fn->save(fn->K, k), fn->save(fn->V, v);
    fn->save(fn->IDS, q_pos), fn->save(fn->IDS + 1, k_pos), fn->save(fn->IDS + 2, q_seq), fn->save(fn->IDS + 3, k_seq);
    fn->mask_mode = mask_mode, fn->scale = scale;
  }
  Tensor o, lse;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(o, lse) = op::attn_fwd().call(q, k, v, mask_mode, scale, q_pos, k_pos, q_seq, k_seq);
  }
  if (fn) {
    set_history(o, fn);
    set_history(lse, fn);
    fn->save(fn->O, o, true), fn->save(fn->LSE, lse, true);
  }
  return {o, lse};
}

// into_grad: the weight's gradient is added into the buffer it already owns, as the products of the linear layers do it.  A
// weight with tensor hooks is left to autograd, so that the hooks see its gradient.
Tensor norm_grad_buffer(const Tensor& w, bool into_grad) {
  return into_grad && torch::autograd::impl::hooks(w).empty() && !c10::impl::dispatch_mode_enabled() ? bound_grad(w, true) : Tensor();
}

struct RmsNormBackward final : Formula {
  enum { X, W, RSTD, COUNT };
  bool into_grad = false;
  RmsNormBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosRmsNormBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    const Tensor grad = task_should_compute_output(1) && g[0].defined() ? norm_grad_buffer(s[W], into_grad) : Tensor();
    if (grad.defined()) {
      Tensor dx = rmsnorm_bwd_into(g[0], Tensor(), s[X], s[W], s[RSTD], grad);
      notify_grad_written(s[W]);
      return {dx, Tensor()};
    }
    auto [dx, dw] = op::rmsnorm_bwd().call(g[0].defined() ? g[0] : at::zeros_like(s[X]), s[X], s[W], s[RSTD]);
    return {dx, dw};
  }
};

std::tuple<Tensor, Tensor> rmsnorm_recorded(const Tensor& x, const Tensor& w, double eps, bool into_grad) {
  refuse_tangents("rmsnorm_fwd", x, w);
  std::shared_ptr<RmsNormBackward> fn;
  if (compute_requires_grad(x, w)) {
    fn = make_formula<RmsNormBackward>();
    fn->into_grad = into_grad;
    fn->set_next_edges(collect_next_edges(x, w));
    fn->save(fn->X, x), fn->save(fn->W, w);
  }
  Tensor y, rstd;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(y, rstd) = op::rmsnorm_fwd().call(x, w, eps);
  }
  if (fn) {
    set_history(y, fn);
    set_history(rstd, fn);
    fn->save(fn->RSTD, rstd, true);
  }
  return {y, rstd};
}

// g[0]: gradient of the summed row from its later uses (the residual path), g[1]: gradient of the normalised row.  Both
// addends receive the same gradient.
struct AddRmsNormBackward final : Formula {
  enum { H, W, RSTD, COUNT };
  bool into_grad = false;
  AddRmsNormBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosAddRmsNormBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[1].defined()) return {g[0], g[0], Tensor()};
    if (const Tensor grad = task_should_compute_output(2) ? norm_grad_buffer(s[W], into_grad) : Tensor(); grad.defined()) {
      Tensor dx = rmsnorm_bwd_into(g[1], g[0], s[H], s[W], s[RSTD], grad);
      notify_grad_written(s[W]);
      return {dx, dx, Tensor()};
    }
    auto [dx, dw] = g[0].defined() ? op::add_rmsnorm_bwd().call(g[1], g[0], s[H], s[W], s[RSTD]) : op::rmsnorm_bwd().call(g[1], s[H], s[W], s[RSTD]);
    return {dx, dx, dw};
  }
};

std::tuple<Tensor, Tensor, Tensor> add_rmsnorm_recorded(const Tensor& x, const Tensor& res, const Tensor& w, double eps, bool into_grad) {
  refuse_tangents("add_rmsnorm_fwd", x, res, w);
  std::shared_ptr<AddRmsNormBackward> fn;
  if (compute_requires_grad(x, res, w)) {
    fn = make_formula<AddRmsNormBackward>();
    fn->into_grad = into_grad;
    fn->set_next_edges(collect_next_edges(x, res, w));
    fn->save(fn->W, w);
  }
  Tensor h, y, rstd;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(h, y, rstd) = op::add_rmsnorm_fwd().call(x, res, w, eps);
  }
  if (fn) {
    set_history(h, fn);
    set_history(y, fn);
    set_history(rstd, fn);
    fn->save(fn->H, h, true), fn->save(fn->RSTD, rstd, true);
  }
  return {h, y, rstd};
}

std::tuple<Tensor, Tensor> rmsnorm_fwd_autograd(const Tensor& x, const Tensor& w, double eps) { return rmsnorm_recorded(x, w, eps, false); }
std::tuple<Tensor, Tensor, Tensor> add_rmsnorm_fwd_autograd(const Tensor& x, const Tensor& res, const Tensor& w, double eps) {
  return add_rmsnorm_recorded(x, res, w, eps, false);
}

struct RopeBackward final : Formula {
  enum { COS, SIN, POSITIONS, COUNT };
  int64_t position_offset = 0;
  bool inverse = false;
  RopeBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosRopeBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return {Tensor()};
    return {op::rope().call(g[0], s[COS], s[SIN], optional_tensor(s[POSITIONS]), position_offset, !inverse)};
  }
  variable_list recorded_backward(variable_list&& g, const std::vector<Tensor>& s) override { return backward(std::move(g), s); }
};

Tensor rope_autograd(const Tensor& x, const Tensor& cos, const Tensor& sin, const OptTensor& positions, int64_t position_offset, bool inverse) {
  refuse_tangents("rope", x, cos, sin);
  std::shared_ptr<RopeBackward> fn;
  if (compute_requires_grad(x)) {
    fn = make_formula<RopeBackward>();
    fn->set_next_edges(collect_next_edges(x));
    fn->save(fn->COS, cos), fn->save(fn->SIN, sin), fn->save(fn->POSITIONS, positions);
    fn->position_offset = position_offset, fn->inverse = inverse;
  }
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    y = op::rope().call(x, cos, sin, positions, position_offset, inverse);
  }
  if (fn) set_history(y, fn);
  return y;
}

struct RopePairBackward final : Formula {
  enum { COS, SIN, POSITIONS, COUNT };
  int64_t position_offset = 0;
  bool inverse = false;
  RopePairBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosRopePairBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    const OptTensor pos = optional_tensor(s[POSITIONS]);
    if (g[0].defined() && g[1].defined()) {
      auto [da, db] = op::rope_pair().call(g[0], g[1], s[COS], s[SIN], pos, position_offset, !inverse);
      return {da, db};
    }
    variable_list out(2);
    for (int i = 0; i < 2; ++i)
      if (g[i].defined()) out[i] = op::rope().call(g[i], s[COS], s[SIN], pos, position_offset, !inverse);
    return out;
  }
  variable_list recorded_backward(variable_list&& g, const std::vector<Tensor>& s) override { return backward(std::move(g), s); }
};

std::tuple<Tensor, Tensor> rope_pair_autograd(const Tensor& xa, const Tensor& xb, const Tensor& cos, const Tensor& sin, const OptTensor& positions,
                                              int64_t position_offset, bool inverse) {
  refuse_tangents("rope_pair", xa, xb, cos, sin);
  std::shared_ptr<RopePairBackward> fn;
  if (compute_requires_grad(xa, xb)) {
    fn = make_formula<RopePairBackward>();
    fn->set_next_edges(collect_next_edges(xa, xb));
    fn->save(fn->COS, cos), fn->save(fn->SIN, sin), fn->save(fn->POSITIONS, positions);
    fn->position_offset = position_offset, fn->inverse = inverse;
  }
  Tensor ya, yb;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(ya, yb) = op::rope_pair().call(xa, xb, cos, sin, positions, position_offset, inverse);
  }
  if (fn) {
    set_history(ya, fn);
    set_history(yb, fn);
  }
  return {ya, yb};
}

struct SwigluBackward final : Formula {
  enum { GATE, UP, COUNT };
  SwigluBackward() : Formula(COUNT) {}
  std::string name() const override { return "MaltosSwigluBackward"; }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return {Tensor(), Tensor()};
    auto [dg, du] = op::swiglu_bwd().call(g[0], s[GATE], s[UP]);
    return {dg, du};
  }
};

Tensor swiglu_fwd_autograd(const Tensor& gate, const Tensor& up) {
  refuse_tangents("swiglu_fwd", gate, up);
  std::shared_ptr<SwigluBackward> fn;
  if (compute_requires_grad(gate, up)) {
    fn = make_formula<SwigluBackward>();
    fn->set_next_edges(collect_next_edges(gate, up));
    fn->save(fn->GATE, gate), fn->save(fn->UP, up);
  }
  Tensor h;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    h = op::swiglu_fwd().call(gate, up);
  }
  if (fn) set_history(h, fn);
  return h;
}

// d loss / d logits was written by the forward kernel; it is scaled by the upstream gradient in place (the kernel returns
// at once when that is 1, the usual case) and handed on without a copy, so a graph can be walked once.
struct CrossEntropyBackward final : Formula {
  bool consumed = false;
  const char* twice = "";
  CrossEntropyBackward() : Formula(1) {}
  std::string name() const override { return "MaltosCrossEntropyBackward"; }
  void before_unpack(const variable_list& g) override { TORCH_CHECK(!consumed || !g[0].defined(), twice); }
  variable_list backward(variable_list&& g, const std::vector<Tensor>& s) override {
    if (!g[0].defined()) return {Tensor()};
    const Tensor dlogits = dense(s[0]);
    op::scale_by_scalar_().call(dlogits, g[0]);
    consumed = true;
    return {dlogits.detach()};
  }
};

std::tuple<Tensor, Tensor, Tensor> ce_fwd_bwd_autograd(const Tensor& logits, const Tensor& labels, int64_t ignore_index) {
  refuse_tangents("ce_fwd_bwd", logits);
  std::shared_ptr<CrossEntropyBackward> fn;
  if (compute_requires_grad(logits)) {
    fn = make_formula<CrossEntropyBackward>();
    fn->set_next_edges(collect_next_edges(logits));
    fn->twice = "maltos::ce_fwd_bwd: backward ran twice through the same loss; its logits gradient is scaled in place by the first pass, so "
                "recompute the loss instead of retaining the graph";
  }
  Tensor loss, dlogits, count;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    std::tie(loss, dlogits, count) = op::ce_fwd_bwd().call(logits, labels, ignore_index);
  }
  if (fn) {
    set_history(loss, fn);
    set_history(dlogits, fn);
    fn->save(0, dlogits, true);
  }
  return {loss, dlogits, count};
}

// The loss whose gradient replaces the logits in their buffer: one read and one write of the same addresses and no second
// logits-sized tensor.  For callers that own the logits and never look at them again; not an operator, because one that
// overwrites an argument it is differentiated by has no functional form to register.
Tensor cross_entropy_over_logits(const Tensor& logits, const Tensor& labels, int64_t ignore_index) {
  refuse_tangents("ce_fwd_bwd", logits);
  std::shared_ptr<CrossEntropyBackward> fn;
  if (compute_requires_grad(logits)) {
    fn = make_formula<CrossEntropyBackward>();
    fn->set_next_edges(collect_next_edges(logits));
    fn->twice = "cross_entropy(overwrite_logits=True): backward ran twice through the same loss; its logits gradient is scaled in place by the "
                "first pass, so recompute the loss instead";
  }
  at::AutoDispatchBelowADInplaceOrView below_autograd;
  Tensor loss = std::get<0>(ce_fwd_bwd(logits, labels, ignore_index, true));
  // the kernel wrote through a raw pointer: tell autograd, so that another node that saved these logits for its own
  // backward raises instead of differentiating through the gradient that now stands in their place
  logits.unsafeGetTensorImpl()->bump_version();
  if (fn) {
    set_history(loss, fn);
    fn->save(0, logits.detach());
  }
  return loss;
}

TORCH_LIBRARY_IMPL(maltos, CUDA, m) {
  m.impl("attn_fwd", TORCH_FN(attention_forward));
  m.impl("attn_bwd", TORCH_FN(attention_backward));
  m.impl("rmsnorm_fwd", TORCH_FN(rmsnorm_fwd));
  m.impl("rmsnorm_bwd", TORCH_FN(rmsnorm_bwd));
  m.impl("add_rmsnorm_fwd", TORCH_FN(add_rmsnorm_fwd));
  m.impl("add_rmsnorm_bwd", TORCH_FN(add_rmsnorm_bwd));
  m.impl("rope", TORCH_FN(rope));
  m.impl("rope_pair", TORCH_FN(rope_pair_op));
  m.impl("swiglu_fwd", TORCH_FN(swiglu_fwd));
  m.impl("swiglu_bwd", TORCH_FN(swiglu_bwd));
  m.impl("ce_fwd_bwd", TORCH_FN(ce_fwd_bwd_op));
  m.impl("scale_by_scalar", TORCH_FN(scale_by_scalar));
  m.impl("scale_by_scalar_", TORCH_FN(scale_by_scalar_));
}

TORCH_LIBRARY_IMPL(maltos, Autograd, m) {
  m.impl("attn_fwd", TORCH_FN(attn_fwd_autograd));
  m.impl("rmsnorm_fwd", TORCH_FN(rmsnorm_fwd_autograd));
  m.impl("add_rmsnorm_fwd", TORCH_FN(add_rmsnorm_fwd_autograd));
  m.impl("rope", TORCH_FN(rope_autograd));
  m.impl("rope_pair", TORCH_FN(rope_pair_autograd));
  m.impl("swiglu_fwd", TORCH_FN(swiglu_fwd_autograd));
  m.impl("ce_fwd_bwd", TORCH_FN(ce_fwd_bwd_autograd));
}

// ---- the functions behind maltos_amd.ops ------------------------------------------------------------------------------
std::tuple<Tensor, Tensor> py_attention(const Tensor& q, const Tensor& k, const Tensor& v, int64_t mask_mode, std::optional<double> scale,
                                        const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  check_attn_inputs(q, k, v);
  return op::attn_fwd().call(q, k, v, mask_mode, resolve_scale(scale, q), q_pos, k_pos, q_seq, k_seq);
}
std::tuple<Tensor, Tensor> py_attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, int64_t mask_mode, std::optional<double> scale,
                                                const OptTensor& q_pos, const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  check_attn_inputs(q, k, v);
  at::AutoDispatchBelowADInplaceOrView below_autograd;
  return attention_forward(q, k, v, mask_mode, resolve_scale(scale, q), q_pos, k_pos, q_seq, k_seq);
}
std::tuple<Tensor, Tensor, Tensor> py_attention_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                         const Tensor& lse, int64_t mask_mode, std::optional<double> scale, const OptTensor& q_pos,
                                                         const OptTensor& k_pos, const OptTensor& q_seq, const OptTensor& k_seq) {
  check_attn_inputs(q, k, v);
  at::AutoDispatchBelowADInplaceOrView below_autograd;
  return attention_backward(dout, q, k, v, o, lse, mask_mode, resolve_scale(scale, q), q_pos, k_pos, q_seq, k_seq);
}
Tensor py_rope(const Tensor& x, const Tensor& cos, const Tensor& sin, const OptTensor& positions, int64_t offset) {
  return op::rope().call(x, cos, sin, positions, offset, false);
}
std::tuple<Tensor, Tensor> py_rope_pair(const Tensor& xa, const Tensor& xb, const Tensor& cos, const Tensor& sin, const OptTensor& positions,
                                        int64_t offset) {
  return op::rope_pair().call(xa, xb, cos, sin, positions, offset, false);
}
Tensor py_swiglu(const Tensor& gate, const Tensor& up) { return op::swiglu_fwd().call(gate, up); }
Tensor py_cross_entropy(const Tensor& logits, const Tensor& labels, int64_t ignore_index) {
  return std::get<0>(op::ce_fwd_bwd().call(logits, labels, ignore_index));
}

size_t set_doc_plan_cache_entries(int64_t n) {
  TORCH_CHECK_VALUE(n >= 0, "the number of cached plans is >= 0");
  PlanList gone;
  std::lock_guard<std::mutex> lock(plan_mutex);
  const size_t previous = plan_cache_entries;
  plan_cache_entries = static_cast<size_t>(n);
  evict_plans(gone);
  return previous;
}
void clear_doc_plan_cache() {
  PlanList gone;
  std::lock_guard<std::mutex> lock(plan_mutex);
  gone.swap(plan_cache);
}
size_t doc_plan_cache_size() {
  std::lock_guard<std::mutex> lock(plan_mutex);
  return std::count_if(plan_cache.begin(), plan_cache.end(), [](const auto& e) { return e->plan.defined(); });
}

}  // namespace

Tensor rms_norm(const Tensor& x, const Tensor& w, double eps, bool into_grad) {
  return std::get<0>(into_grad && at::GradMode::is_enabled() ? rmsnorm_recorded(x, w, eps, true) : op::rmsnorm_fwd().call(x, w, eps));
}
std::tuple<Tensor, Tensor> add_rms_norm(const Tensor& x, const Tensor& res, const Tensor& w, double eps, bool into_grad) {
  auto [h, y, rstd] = into_grad && at::GradMode::is_enabled() ? add_rmsnorm_recorded(x, res, w, eps, true) : op::add_rmsnorm_fwd().call(x, res, w, eps);
  return {h, y};
}

void bind_ops(pybind11::module& m) {
  using torch::wrap_pybind_function;
  m.def("attention", wrap_pybind_function(py_attention));
  m.def("attention_forward", wrap_pybind_function(py_attention_forward));
  m.def("attention_backward", wrap_pybind_function(py_attention_backward));
  m.def("attention_backward_accumulate", wrap_pybind_function(attention_backward_accumulate));
  m.def("attention_backward_ring_block", wrap_pybind_function(attention_backward_ring_block));
  m.def("attention_merge_", wrap_pybind_function(attention_merge_));
  namespace py = pybind11;
  m.def("rms_norm", wrap_pybind_function(rms_norm), py::arg("x"), py::arg("w"), py::arg("eps"), py::arg("into_grad") = false);
  m.def("add_rms_norm", wrap_pybind_function(add_rms_norm), py::arg("x"), py::arg("res"), py::arg("w"), py::arg("eps"), py::arg("into_grad") = false);
  m.def("rope", wrap_pybind_function(py_rope));
  m.def("rope_pair", wrap_pybind_function(py_rope_pair));
  m.def("rope_pair_", wrap_pybind_function(rope_pair_));
  m.def("swiglu", wrap_pybind_function(py_swiglu));
  m.def("swiglu_rows", wrap_pybind_function(swiglu_rows));
  m.def("swiglu_rows_backward", wrap_pybind_function(swiglu_rows_backward));
  m.def("cross_entropy", wrap_pybind_function(py_cross_entropy));
  m.def("cross_entropy_over_logits", wrap_pybind_function(cross_entropy_over_logits));
  m.def("ce_fwd_bwd", wrap_pybind_function(ce_fwd_bwd));
  m.def("adamw_step_", wrap_pybind_function(adamw_step_));
  m.def("sq_norm", wrap_pybind_function(sq_norm));
  m.def("scale_", wrap_pybind_function(scale_));
  m.def("list_sq_norm", wrap_pybind_function(list_sq_norm));
  m.def("list_scale_", wrap_pybind_function(list_scale_));
  m.def("list_adamw_step_", wrap_pybind_function(list_adamw_step_));
  m.def("grad_to_f32_", wrap_pybind_function(grad_to_f32_));
  m.def("grad_sum_slices", wrap_pybind_function(grad_sum_slices));
  m.def("set_doc_plan_cache_entries", wrap_pybind_function(set_doc_plan_cache_entries));
  m.def("clear_doc_plan_cache", wrap_pybind_function(clear_doc_plan_cache));
  m.def("doc_plan_cache_size", wrap_pybind_function(doc_plan_cache_size));
}

}  // namespace maltos
