// Matrix products of the linear layers: the kernels of csrc/gemm.hip up to a size, the vendor library through torch above it.
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "common.hpp"

namespace maltos {

// Number of K-splits for dW = dY^T X.  The product has only out * in outputs but `rows` (= tokens) terms each: for the
// LLaMA-50M projections (512..1536 wide, 16384 tokens) a single GEMM fills a quarter of the 256 CUs and runs at ~85
// TFLOP/s, the same work as a batch of 8-16 row slices reaches 300-600 TFLOP/s on MI355X.
int64_t weight_grad_splits(int64_t rows, int64_t out_features, int64_t in_features) {
  const int64_t tiles = ((out_features + 255) / 256) * ((in_features + 255) / 256);
  int64_t splits = 1;
  while (splits < 16 && tiles * splits < 128 && rows % (splits * 2) == 0 && rows / (splits * 2) >= 1024) splits *= 2;
  return splits;
}

namespace {

// Where the own kernels run, by M * N * K.  A product through torch costs 18 us of host time, a call here 5, and that is what
// small steps wait for.  On the GPU alone (both sides timed with the weights out of HBM; rows from 100 to 16384; the library's choice
// untuned) they are ahead of the library in bf16 up to 4e9 (0.4 to 0.95), and in fp32 without a limit: 0.6 to 1.09 of its time from 5e8 to 2.5e10, 0.75 on the mean, and 0.73 to 0.82 from there
// to 3.2e11 (logits of 16384 x 32000 x 512 3165 us for 3843, their dx 2695 / 3493, dW 2842 / 3578), with smaller errors
constexpr double kOwnLimitBf16 = 4.0e9;

// Larger bf16 products, by what running one of them on the own kernels adds to a layer's training step in which the library has the others (us; 145
// layers of 21 shapes, 256 to 2048 wide, of 3000 to 32768 rows; two runs differ by 4 us).  These lines take 7 % off a layer's step on the mean, and the
// one that is slower than with the library alone by more than half a percent is by 1.7 % (dW of 1024 x 1024, 10000 rows).
//   terms of y and dx, either side of the lines
//     up to 768, 3e10      y of 3 x 768 rotated, 16384 rows -33, 20020 +7; gate and up of 2 x 1376 x 512, 16384 rows -23; of 2 x 2048 x 768, 6000 rows -7, 24576 +91
//     up to 1536, 1.3e10   y of 512 x 1376, 16384 rows -18; of 512 x 1536, 8192 rows -5, 16384 0, 20020 +10, 24576 +17
//     up to 2816, 8.5e9    y of 512 x 2048, 4096 rows -15, 8192 +8, 20020 +27; of 896 x 2392, 4096 rows -3, 10000 +26
//   1024 and more columns and terms, both whole tiles of 256 (the library's): y of 1024 x 1024, 6000 rows +2 to +27, 12000 -2 to +11 (alone, 6000 and 12000 rows:
//     22 us against 18, 34 against 26).  With their dW in one launch up to 8.5e9: 3000 x 1280 x 1280 -22, 6000 x 1024 x 1024 -15 to +4, but 10000 rows +54 to +76.
//   gate and up in one launch, kept for a backward pass, 257 to 512 terms, whole tiles whose 256 x 256 fill their rounds over the CUs: 2 x 2048 x 512, 8192 rows +13 and 10000
//     +25, beside -15 and -17 for the product and the pass apart; but 12000 rows of 2 x 1536 x 512 (a quarter idle) -11.
//   dW, which the library forms as a batch of row slices (weight_grad_splits).  Slices too few for 64 of its tiles: 1024 x 1024 of 20001 rows, alone, 56 us against 162.  Slices of
//     whole 1024 rows, from 16384 rows on: 512 to 768 wide 16384 rows -14 to +20, 24576 -32 to +32, but 20020 rows -2 to -57; below, up to 2e10: 5456 x 1024 x 4096 +13 to +15,
//     3072 x 1024 x 8192 +4 to +21; 64 tiles without slices: 6912 x 1280 x 3000 +21, 5456 x 1024 x 3000 -4 to -9; others up to 3e10: 1024 x 2728 x 10000 -55, 1280 x 1792 x 12000 -27.
//   dW of 8192 rows and more (of a vocabulary), own over library's time, alone, added onto a gradient, 640 to 20001 terms, by tiles of 256 x 256
//     up to 64                       0.45 to 1.07, 8192 x 512 0.64 to 0.94, 16384 x 256 0.59 to 0.99
//     65 to 95 (20000 x 256)         from 2048 terms on 0.40 to 1.08; 1536 terms 0.87 to 1.20; 96, whole ones (8192 x 768, 24576 x 256) 0.84 to 1.31
//     up to 128 wide                 up to 128 tiles 0.40 to 1.14; 157 and 197 tiles (40000 x 128, 50264 x 64 and x 128) 0.79 to 1.40
//     whole ones, 10000 terms on     up to 128 tiles 0.65 to 1.07; 129 to 192 (16384 x 768, 40000 x 256: part of the CUs idle in the last round) 0.73 to 1.11; more 0.73 to 0.98
//     others                         16384 x 384 and x 512 below 10000 terms 0.91 to 1.22; 20000 x 512, 24576 x 384, 40000 x 256, 50264 x 256 0.82 to 1.57; 32000 x 512 0.93 to 1.06
//     In one launch with dh = dy W and the activation -2 to -107 at all row counts up to 32768; that dh without its dW up to +74.
// These were measured on tiles of 128 x 128 where 256 x 128 is taken since (y of 512 x 1376, 16384 rows, 39 us, now 34), and dW of fewer than 8192 rows before its 256 x 256 had a ring of stages.
// (With the shipped per-shape selection, 16384 rows, alone: y 512 x 512 17 us against 16, 1536 x 512 42 / 32, in a step rotated on its way out 48 / 32 + 15,
// 512 x 1376 34 / 40, 2752 x 512 65 / 73; dW 512 x 1376 41 / 45, 1536 x 512 41 / 37, 2752 x 512 63 / 58.)  Products with the columns of a vocabulary (32000 x 512): 1023 rows
// 54 / 49, 3000 rows 136 / 131.
bool larger_own_range_bf16(int form, int64_t M, int64_t N, int64_t K, Use use) {
  const double size = static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(K);
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
  if (N >= 16384 || N % 8) return false;
  if (form == MLTS_GEMM_TN) {
    if (M >= 8192 && (tiles <= 64 || (tiles < 96 && K >= 2048) || (N <= 128 && tiles <= 128))) return true;
    if (M >= 8192 && N % 256 == 0 && K >= 10000 && (tiles <= 128 || (M >= 16384 && tiles > 192))) return true;
    if (M >= 16384) return false;
    if (use == Use::ACTIVATION) return true;
    const bool few = tiles * weight_grad_splits(K, M, N) < 64, whole = !few && K % 1024 == 0;
    return !(whole && K >= 16384) && size <= (whole || tiles >= 64 ? 2.0e10 : 3.0e10);
  }
  if (size > (K <= 768 ? 3.0e10 : K <= 1536 ? 1.3e10 : K <= 2816 ? 8.5e9 : 0)) return false;
  if (K >= 1024 && N >= 1024 && N % 256 == 0 && K % 256 == 0) {
    if (use == Use::ALONE) return false;
    if (use == Use::WITH_WEIGHT_GRAD) return size <= 8.5e9;
  }
  return use != Use::GATE_AND_UP || N % 256 || K % 64 || K <= 256 || K > 512 || tiles <= 256 || 10 * tiles < 8 * ((tiles + 255) / 256 * 256);
}

// In bf16 they also run for dx = dy W with a long contraction over few outputs (dx of an lm_head, of a wide MLP), which is split over
// workgroups where the tiles leave CUs idle: the library does not split those.  Own over library's time, 605 products of 64 to 20001 rows,
// 256 to 4096 columns, 4e9 to 3e11 terms, by tiles of 256 x 128 (geometric mean, largest):
//   2816 to 6144 terms    up to 32 0.71, 0.99    33 to 64 0.74, 0.91    65 to 128 0.87, 0.99    129 to 160 0.97, 1.22    161 to 256 1.03, 1.15    more 1.07, 1.33
//   8192 to 50264 terms   up to 32 0.38, 0.63    33 to 64 0.52, 0.73    65 to 128 0.71, 0.91    129 to 160 0.94, 1.21    161 to 255 1.04, 1.18    256 1.00, 1.05    more 1.09, 1.33
bool long_contraction_bf16(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 127) / 128);
  return K >= 2816 && (tiles <= 128 || (K >= 8192 && tiles == 256));
}

bool within_own_range(int form, int dtype, int64_t M, int64_t N, int64_t K, Use use) {
  const double size = static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(K);
  return dtype == MLTS_F32 || size <= kOwnLimitBf16 || larger_own_range_bf16(form, M, N, K, use) || (form == MLTS_GEMM_NN && long_contraction_bf16(M, N, K));
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

bool own_product(int form, const Tensor& a, const Tensor& b, Use use) {
  if (!plain(a) || !plain(b) || !same_contraction(form, a, b)) return false;  // (operands that do not match: torch says so)
  const Sizes z(form, a, b);
  return z.M > 0 && z.N > 0 && z.K > 0 && a.scalar_type() == b.scalar_type() &&
         (a.scalar_type() == at::kBFloat16 || a.scalar_type() == at::kFloat) && within_own_range(form, dtype_code(a), z.M, z.N, z.K, use) &&
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
