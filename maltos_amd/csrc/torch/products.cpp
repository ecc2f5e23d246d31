// Matrix products of the linear layers: the kernels of csrc/gemm.hip up to a size, the vendor library through torch above it.
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "common.hpp"

namespace maltos {
namespace {

// M * N * K up to which the own kernels run.  A product through torch costs 18 us of host time, a call here 5, and that is what
// small steps wait for: up to a few thousand rows of a 512-wide model the host is behind the GPU.  There the own kernels are
// the faster ones on the GPU as well (1023 x 512 x 32000, dx: 45 us against the library's 145; 512-wide: 9 against 12).  From
// 16384 x 512 x 512 on a step fills the GPU for longer than the host needs, and the library's kernels, with the shipped
// per-shape selection, are ahead: a training step of that size took 90 us more of 9500 with its 512-wide products done here.
constexpr double kOwnLimit = 4.0e9;

// Above it they still run for dx = dy W with so long a contraction that it is split over workgroups (dx of an lm_head): the
// library does not split those (us, 512 wide, 32000 terms: 1024 rows 47 against 160, 8192 rows 270 against 346).
bool within_own_range(int form, int dtype, int64_t M, int64_t N, int64_t K) {
  return static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(K) <= kOwnLimit ||
         (form == MLTS_GEMM_NN && mlts_gemm_workspace_bytes(form, dtype, M, N, K) > 0);
}

struct Sizes {
  int64_t M, N, K;  // (K as the first operand has it)
  Sizes(int form, const Tensor& a, const Tensor& b)
      : M(form == MLTS_GEMM_TN ? a.size(1) : a.size(0)), N(form == MLTS_GEMM_NT ? b.size(0) : b.size(1)), K(form == MLTS_GEMM_TN ? a.size(0) : a.size(1)) {}
};

bool plain(const Tensor& t) { return t.is_cuda() && t.dim() == 2 && (t.stride(1) == 1 || t.size(1) == 1) && !at::isTensorSubclassLike(t); }

bool same_contraction(int form, const Tensor& a, const Tensor& b) { return a.size(form == MLTS_GEMM_TN ? 0 : 1) == b.size(form == MLTS_GEMM_NT ? 1 : 0); }

int64_t row_stride(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }  // (a single row's stride means nothing)

Tensor library_product(int form, const Tensor& a, const Tensor& b, const Tensor& out, bool accumulate) {
  const Tensor x = form == MLTS_GEMM_TN ? a.t() : a, y = form == MLTS_GEMM_NT ? b.t() : b;
  if (!out.defined()) return at::mm(x, y);
  Tensor o = out;
  return accumulate ? o.addmm_(x, y) : at::mm_out(o, x, y);
}

}  // namespace

bool own_product(int form, const Tensor& a, const Tensor& b) {
  if (!plain(a) || !plain(b) || !same_contraction(form, a, b)) return false;  // (operands that do not match: torch says so)
  const Sizes z(form, a, b);
  return z.M > 0 && z.N > 0 && z.K > 0 && a.scalar_type() == b.scalar_type() &&
         (a.scalar_type() == at::kBFloat16 || a.scalar_type() == at::kFloat) && within_own_range(form, dtype_code(a), z.M, z.N, z.K) &&
         mlts_gemm_supports(form, dtype_code(a), z.M, z.N, z.K, a.stride(0), b.stride(0), z.N) == nullptr && aligned(a) && aligned(b) &&
         !c10::impl::dispatch_mode_enabled() && !at::autocast::is_autocast_enabled(at::kCUDA);
}

Tensor product(int form, const Tensor& a, const Tensor& b, const Tensor& out, bool accumulate) {
  TORCH_CHECK_VALUE(a.dim() == 2 && b.dim() == 2, "a product takes two matrices, got ", a.sizes(), " and ", b.sizes());
  const Sizes z(form, a, b);
  TORCH_CHECK_VALUE(!out.defined() || (out.dim() == 2 && out.size(0) == z.M && out.size(1) == z.N), "a product of shape [", z.M, ", ", z.N,
                    "] cannot be written to a tensor of shape ", out.sizes());
  if (!own_product(form, a, b) || (out.defined() && !own_output(out, a))) return library_product(form, a, b, out, accumulate);
  Tensor c = out.defined() ? out : at::empty({z.M, z.N}, a.options());
  const int dtype = dtype_code(a);
  const int64_t ws_bytes = mlts_gemm_workspace_bytes(form, dtype, z.M, z.N, z.K);
  Tensor ws = workspace(ws_bytes, a);
  check(mlts_gemm(form, dtype, z.M, z.N, z.K, ptr(a), a.stride(0), ptr(b), b.stride(0), mptr(c), row_stride(c), accumulate,
                  ws.defined() ? mptr(ws) : nullptr, ws_bytes, current_stream()));
  return c;
}

bool own_output(const Tensor& out, const Tensor& a) {
  return plain(out) && aligned(out) && out.scalar_type() == a.scalar_type() && row_stride(out) >= out.size(1);
}

void ProductList::add(int form, const Tensor& a, const Tensor& b, const Tensor& out, bool accumulate) {
  const Sizes z(form, a, b);
  mlts_gemm_product& p = items[count++];
  p = {};
  p.form = form, p.accumulate = accumulate;
  p.M = z.M, p.N = z.N, p.c = mptr(out), p.ldc = row_stride(out);
  add_segment(a, b);
  like = a;
}

void ProductList::add_segment(const Tensor& a, const Tensor& b) {
  mlts_gemm_product& p = items[count - 1];
  const int i = p.segments++;
  p.k[i] = Sizes(p.form, a, b).K;
  p.a[i] = ptr(a), p.lda[i] = a.stride(0), p.b[i] = ptr(b), p.ldb[i] = b.stride(0);
}

void ProductList::run() const {
  const int dtype = dtype_code(like);
  const int64_t ws_bytes = mlts_gemm_multi_workspace_bytes(items, count, dtype);
  Tensor ws = workspace(ws_bytes, like);
  check(mlts_gemm_multi(items, count, dtype, ws.defined() ? mptr(ws) : nullptr, ws_bytes, current_stream()));
}

}  // namespace maltos
