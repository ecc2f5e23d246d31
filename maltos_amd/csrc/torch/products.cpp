// Matrix products of the linear layers: the kernels of csrc/gemm.hip up to a size, the vendor library through torch above it.
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "common.hpp"

namespace maltos {
namespace {

// Where the own kernels run, by M * N * K.  A product through torch costs 18 us of host time, a call here 5, and that is what
// small steps wait for.  On the GPU alone (both sides timed with the weights out of HBM; rows from 100 to 16384; the library's choice
// untuned, or with the shipped per-shape selection where that has the shape) they are ahead of the library
//   fp32  0.5 to 1e9  0.86 of its time (y), 0.86 (dx), 0.82 (dW)    2.5 to 3e9  0.90, 0.92, 0.87    3 to 4e9  1.13, 1.15, 1.17
//   bf16  up to 4e9   0.4 to 0.95
//         above it, y and dx of 256 or 512 terms: 8192 x 2752 x 512 34.3 us against 61.7, 12000 x 2752 x 512 50 against 80, 16384 x 2752 x 512
//         61 against 78, 16384 x 1376 x 512 36 against 50; but 16384 x 1536 x 512 38 against 32 with the shipped selection (rotated on
//         its way out 39 against 32 + 15)
//         1024 to 1536 terms: 12000 x 512 x 1376 31 against 36, 16384 x 512 x 1376 34 against 40, 16384 x 512 x 1536 32 against 35; but 6000 and
//         12000 x 1024 x 1024 20.9 and 33.6 against 19.6 and 30.0
//         2752 terms: 3000 x 512 21 against 26, 6000 x 512 31 against 33, 12000 x 512 50 against 46
//         dW against a batch of row slices: 6000 rows 1536 x 512 27 against 44, 8192 rows 2752 x 512 46 against 52, 12000 rows 39 against 52
//         and 58 against 95; but 16384 rows 47 against 41 and 73 against 63
//         columns of a vocabulary (32000 x 512): 1023 rows 54 against 49, 3000 rows 136 against 131
constexpr double kOwnLimitBf16 = 4.0e9, kOwnLimitF32 = 3.0e9;
double larger_limit_bf16(int form, int64_t M, int64_t N, int64_t K) {
  if (N >= 16384 || N % 8) return 0;
  if (form == MLTS_GEMM_TN) return M < 16384 && K < 16384 ? 3.0e10 : 0;
  return K <= 768 ? 3.0e10 : K <= 1536 ? 1.3e10 : K <= 2816 ? 8.5e9 : 0;
}

// In bf16 they also run for dx = dy W with so long a contraction that it is split over workgroups (dx of an lm_head, of a wide
// MLP): the library does not split those.  Own over library's time, 256 to 8192 rows, 512 to 4096 wide: 32000 terms 0.17 to 0.79, 11008
// terms 0.54 to 0.83, 8192 terms 0.42 to 0.98; with 4096 or 5504 terms 0.76 to 1.04 where fewer than 128 tiles of 256 x 128 leave more
// than half of the CUs idle unsplit, but 1.05 and 1.12 for 128 tiles (2048 x 2048 x 5504 56.6 us against 53.8, 1024 x 4096 x 4096 46.1
// against 41.1).
bool within_own_range(int form, int dtype, int64_t M, int64_t N, int64_t K) {
  const double size = static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(K);
  if (dtype == MLTS_F32) return size <= kOwnLimitF32;
  if (size <= std::max(kOwnLimitBf16, larger_limit_bf16(form, M, N, K))) return true;
  return form == MLTS_GEMM_NN && (K >= 8192 || M * N < 128 * 256 * 128) && mlts_gemm_workspace_bytes(form, dtype, M, N, K) > 0;
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
