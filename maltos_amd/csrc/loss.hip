// Causal cross-entropy: loss and d(logits) from ONE read of the logits.  A block owns one row, keeps it in registers,
// reduces max and sum-exp with 64-lane shuffles, then streams the gradient out.  Rows whose label is the ignore
// index are never read: their gradient is zero.
//
// A vocabulary that the vector width does not divide (50257) leaves rows that start anywhere within 16 bytes: a row is
// then walked as a short head, aligned 16-byte vectors, and a short tail, whose at most 2 * (vector - 1) single elements go to
// one lane each.
#include "common.hpp"

namespace {

constexpr int kCeThreads = 512;
constexpr int kCeWaves = kCeThreads / MLTS_WAVE;
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float block_max(float x, float* red) {
  x = wave_max(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < kCeWaves; ++w) r = fmaxf(r, red[w]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ float block_sum(float x, float* red) {
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float r = 0.f;
#pragma unroll
  for (int w = 0; w < kCeWaves; ++w) r += red[w];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(1024) void ce_count_kernel(const int64_t* __restrict__ labels, int64_t rows,
                                                        int64_t ignore_index, int32_t* __restrict__ count_out) {
  __shared__ int part[16];
  int c = 0;
  for (int64_t i = threadIdx.x; i < rows; i += 1024) c += labels[i] != ignore_index ? 1 : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, MLTS_WAVE);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int w = 0; w < 16; ++w) s += part[w];
    *count_out = s;
  }
}

// A row as a head of single elements, whole aligned vectors and a tail of single elements.  Logits and gradient rows have the
// same split because both buffers start 16-byte aligned (checked by the launcher).
template <typename T>
struct CeRow {
  static constexpr int N = Vec16<T>::N;
  int head, nvec, singles, vocab;
  __device__ __forceinline__ CeRow(int64_t row, int vocab_) : vocab(vocab_) {
    const int off = static_cast<int>((row * vocab) & (N - 1));
    head = min(vocab, off ? N - off : 0);
    nvec = (vocab - head) / N;
    singles = vocab - nvec * N;
  }
  // column of single element t < singles (head first, then tail)
  __device__ __forceinline__ int single(int t) const { return t < head ? t : t + nvec * N; }
};

template <typename T>
__device__ __forceinline__ void ce_zero_row(T* dr, const CeRow<T>& r) {
  Vec16<T> z;
#pragma unroll
  for (int j = 0; j < CeRow<T>::N; ++j) z.set(j, 0.f);
  for (int c = threadIdx.x; c < r.nvec; c += kCeThreads) __builtin_nontemporal_store(z.v, reinterpret_cast<decltype(z.v)*>(dr + r.head) + c);
  if (static_cast<int>(threadIdx.x) < r.singles) dr[r.single(threadIdx.x)] = from_f32<T>(0.f);
}

// Row kept in registers: NV 16-byte vectors per lane (a 32000-entry bf16 row is 8 per lane of a 512-lane block), all loads of a
// row issued before the first use.  No LDS beyond the reduction scratch: three blocks per CU up to eight vectors per lane (the
// register budget that still compiles without spills), two with sixteen.
// bf16 1021 x 50257: 180 us with one 2-byte access per lane, 50 us (4.1 TB/s) in this form.
template <typename T, int NV>
__global__ __launch_bounds__(kCeThreads, NV > 8 ? 4 : 6) void ce_row_reg_kernel(const T* logits,  // may be dlogits (gradient in place)
                                                                const int64_t* __restrict__ labels, T* dlogits,
                                                                float* __restrict__ row_loss,
                                                                const int32_t* __restrict__ count, int vocab,
                                                                int64_t ignore_index) {
  constexpr int N = Vec16<T>::N;
  __shared__ float red[kCeWaves];
  const int64_t row = blockIdx.x;
  const int64_t label = labels[row];
  const CeRow<T> r(row, vocab);
  const T* zr = logits + row * vocab;
  T* dr = dlogits + row * vocab;
  const int tid = threadIdx.x;
  if (label == ignore_index) {
    if (tid == 0) row_loss[row] = 0.f;
    ce_zero_row<T>(dr, r);
    return;
  }
  const bool label_ok = label >= 0 && label < vocab;
  const bool has_single = tid < r.singles;
  const int single_col = has_single ? r.single(tid) : 0;
  Vec16<T> t[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = tid + i * kCeThreads;
    if (c < r.nvec) t[i].v = __builtin_nontemporal_load(reinterpret_cast<const decltype(t[i].v)*>(zr + r.head) + c);
  }
  const float single = has_single ? to_f32<T>(zr[single_col]) : -INFINITY;
  float label_logit = 0.f;
  if (tid == 0 && label_ok) label_logit = to_f32<T>(zr[label]);
  float mx = single;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (tid + i * kCeThreads < r.nvec) {
#pragma unroll
      for (int j = 0; j < N; ++j) mx = fmaxf(mx, t[i].get(j));
    }
  }
  mx = block_max(mx, red);
  const float mxs = mx * kLog2e;
  float se = has_single ? exp2f(single * kLog2e - mxs) : 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (tid + i * kCeThreads < r.nvec) {
#pragma unroll
      for (int j = 0; j < N; ++j) se += exp2f(t[i].get(j) * kLog2e - mxs);
    }
  }
  se = block_sum(se, red);
  const float lse = mx + logf(se);
  if (tid == 0) row_loss[row] = label_ok ? lse - label_logit : NAN;
  const int cnt = *count;
  const float inv = 1.0f / static_cast<float>(cnt > 0 ? cnt : 1);
  const float lses = lse * kLog2e;
  const int lcol = label_ok ? static_cast<int>(label) - r.head : -1;  // negative: the label is in the head (or nowhere)
  const int lvec = lcol >= 0 ? lcol / N : -1;
  const int lsub = lcol >= 0 ? lcol % N : 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = tid + i * kCeThreads;
    if (c < r.nvec) {
      Vec16<T> o;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        float p = exp2f(t[i].get(j) * kLog2e - lses);
        if (c == lvec && j == lsub) p -= 1.0f;
        o.set(j, p * inv);
      }
      __builtin_nontemporal_store(o.v, reinterpret_cast<decltype(o.v)*>(dr + r.head) + c);
    }
  }
  if (has_single) {
    float p = exp2f(single * kLog2e - lses);
    if (single_col == label) p -= 1.0f;
    dr[single_col] = from_f32<T>(p * inv);
  }
}

// Rows that do not fit the registers of a block (more than 65536 bf16 or 32768 fp32 entries), and buffers that are not 16-byte
// aligned (VEC = false: single elements throughout): max and sum in one pass (a running maximum per lane), the gradient in a
// second one that reads the row again.
template <typename T, bool VEC>
__global__ __launch_bounds__(kCeThreads) void ce_row_stream_kernel(const T* logits,  // may be dlogits (gradient in place)
                                                                   const int64_t* __restrict__ labels, T* dlogits,
                                                                   float* __restrict__ row_loss,
                                                                   const int32_t* __restrict__ count, int vocab,
                                                                   int64_t ignore_index) {
  constexpr int N = Vec16<T>::N;
  __shared__ float red[kCeWaves];
  const int64_t row = blockIdx.x;
  const int64_t label = labels[row];
  CeRow<T> r(row, vocab);
  if (!VEC) r.head = 0, r.nvec = 0, r.singles = vocab;
  const T* zr = logits + row * vocab;
  T* dr = dlogits + row * vocab;
  if (label == ignore_index) {
    if (threadIdx.x == 0) row_loss[row] = 0.f;
    if (VEC) {
      ce_zero_row<T>(dr, r);
    } else {
      for (int c = threadIdx.x; c < vocab; c += kCeThreads) dr[c] = from_f32<T>(0.f);
    }
    return;
  }
  const bool label_ok = label >= 0 && label < vocab;
  float m = -INFINITY, se = 0.f;
  auto take = [&](const float* x, int n) {
    float top = m;
    for (int j = 0; j < n; ++j) top = fmaxf(top, x[j]);
    const float base = top == -INFINITY ? 0.f : top;
    if (top > m) se *= exp2f((m - base) * kLog2e), m = top;
    for (int j = 0; j < n; ++j) se += exp2f((x[j] - base) * kLog2e);
  };
  for (int c = threadIdx.x; c < r.nvec; c += kCeThreads) {
    const Vec16<T> t = reinterpret_cast<const Vec16<T>*>(zr + r.head)[c];
    float x[N];
#pragma unroll
    for (int j = 0; j < N; ++j) x[j] = t.get(j);
    take(x, N);
  }
  for (int c = threadIdx.x; c < r.singles; c += kCeThreads) {
    const float x = to_f32<T>(zr[r.single(c)]);
    take(&x, 1);
  }
  // read before the barriers: behind the last one other threads may already be storing gradients over the row
  float label_logit = 0.f;
  if (threadIdx.x == 0 && label_ok) label_logit = to_f32<T>(zr[label]);
  const float mx = block_max(m, red);
  // (a lane without a maximum has seen nothing, only -inf, which add 0, or NaN, which is its sum and has to reach the loss)
  se = block_sum(m == -INFINITY ? se : se * exp2f((m - mx) * kLog2e), red);
  const float lse = mx + logf(se);
  if (threadIdx.x == 0) row_loss[row] = label_ok ? lse - label_logit : NAN;
  const int cnt = *count;
  const float inv = 1.0f / static_cast<float>(cnt > 0 ? cnt : 1);
  const float lses = lse * kLog2e;
  const int lcol = label_ok ? static_cast<int>(label) - r.head : -1;
  const int lvec = lcol >= 0 ? lcol / N : -1;
  const int lsub = lcol >= 0 ? lcol % N : 0;
  for (int c = threadIdx.x; c < r.nvec; c += kCeThreads) {
    const Vec16<T> t = reinterpret_cast<const Vec16<T>*>(zr + r.head)[c];
    Vec16<T> o;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      float p = exp2f(t.get(j) * kLog2e - lses);
      if (c == lvec && j == lsub) p -= 1.0f;
      o.set(j, p * inv);
    }
    __builtin_nontemporal_store(o.v, reinterpret_cast<decltype(o.v)*>(dr + r.head) + c);
  }
  for (int s = threadIdx.x; s < r.singles; s += kCeThreads) {
    const int c = r.single(s);
    float p = exp2f(to_f32<T>(zr[c]) * kLog2e - lses);
    if (c == label) p -= 1.0f;
    dr[c] = from_f32<T>(p * inv);
  }
}

__global__ __launch_bounds__(kCeThreads) void ce_loss_reduce_kernel(const float* __restrict__ row_loss, int64_t rows,
                                                                    const int32_t* __restrict__ count,
                                                                    float* __restrict__ loss_out) {
  __shared__ double part[kCeWaves];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < rows; i += kCeThreads) acc += static_cast<double>(row_loss[i]);
  acc = wave_sum_f64(acc);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < kCeWaves; ++w) s += part[w];
    const int c = *count;
    *loss_out = static_cast<float>(s / static_cast<double>(c > 0 ? c : 1));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void scale_by_scalar_kernel(T* x, const float* scale, int64_t n) {
  const float s = *scale;
  if (s == 1.0f) return;  // the usual case: loss is the root of the graph
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride)
    x[i] = from_f32<T>(to_f32<T>(x[i]) * s);
}

// 16-byte form for an aligned buffer: n_vec whole vectors, the tail (< one vector) by the first lanes of block 0.
template <typename T>
__global__ __launch_bounds__(256) void scale_by_scalar_vec_kernel(T* x, const float* scale, int64_t n_vec, int64_t n) {
  using V = Vec16<T>;
  const float s = *scale;
  if (s == 1.0f) return;
  V* xv = reinterpret_cast<V*>(x);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n_vec; i += stride) {
    V v = xv[i];
#pragma unroll
    for (int j = 0; j < V::N; ++j) v.set(j, v.get(j) * s);
    xv[i] = v;
  }
  const int64_t tail = n_vec * V::N + static_cast<int64_t>(threadIdx.x);
  if (blockIdx.x == 0 && tail < n) x[tail] = from_f32<T>(to_f32<T>(x[tail]) * s);
}

template <typename T>
void ce_launch(const void* logits, const int64_t* labels, void* dlogits, float* row_loss, const int32_t* count,
               int64_t rows, int vocab, int64_t ignore_index, hipStream_t st) {
  constexpr int N = Vec16<T>::N;
  const bool aligned = mlts_aligned16(logits) && mlts_aligned16(dlogits);
  const T* lg = static_cast<const T*>(logits);
  T* dl = static_cast<T*>(dlogits);
  const int per_lane = (vocab / N + kCeThreads - 1) / kCeThreads;  // whole vectors of a row per lane
#define MLTS_CE(KERN) \
  hipLaunchKernelGGL((KERN), dim3((unsigned)rows), dim3(kCeThreads), 0, st, lg, labels, dl, row_loss, count, vocab, ignore_index)
#define MLTS_CE_REG(NV) MLTS_CE((ce_row_reg_kernel<T, NV>))
  if (!aligned) MLTS_CE((ce_row_stream_kernel<T, false>));
  else if (per_lane <= 1) MLTS_CE_REG(1);
  else if (per_lane <= 2) MLTS_CE_REG(2);
  else if (per_lane <= 4) MLTS_CE_REG(4);
  else if (per_lane <= 8) MLTS_CE_REG(8);
  else if (per_lane <= 16) MLTS_CE_REG(16);
  else MLTS_CE((ce_row_stream_kernel<T, true>));
#undef MLTS_CE_REG
#undef MLTS_CE
}

}  // namespace

extern "C" int64_t mlts_ce_workspace_bytes(int64_t rows) { return (rows < 0 ? 0 : rows) * 4 + 64; }

extern "C" int mlts_ce_fwd_bwd(const void* logits, const int64_t* labels, void* dlogits, float* loss_out,
                               int32_t* count_out, void* workspace, int64_t workspace_bytes, int64_t rows,
                               int32_t vocab, int64_t ignore_index, int32_t dtype, mlts_stream_t stream) {
  MLTS_REQUIRE(dtype == MLTS_BF16 || dtype == MLTS_F32, "mlts_ce_fwd_bwd: unknown dtype %d", dtype);
  MLTS_REQUIRE(rows >= 0 && vocab > 0, "mlts_ce_fwd_bwd: bad shape rows=%lld vocab=%d", (long long)rows, vocab);
  MLTS_REQUIRE(rows <= 0x7fffffffLL, "mlts_ce_fwd_bwd: too many rows");
  MLTS_REQUIRE(loss_out && count_out && workspace, "mlts_ce_fwd_bwd: null output pointer");
  MLTS_REQUIRE(workspace_bytes >= mlts_ce_workspace_bytes(rows), "mlts_ce_fwd_bwd: workspace too small");
  MLTS_REQUIRE(rows == 0 || (logits && labels && dlogits), "mlts_ce_fwd_bwd: null input pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* row_loss = static_cast<float*>(workspace);
  hipLaunchKernelGGL(ce_count_kernel, dim3(1), dim3(1024), 0, st, labels, rows, ignore_index, count_out);
  if (rows > 0) {
    MltsKernelTimer timer("ce", st);
    if (dtype == MLTS_BF16) ce_launch<bf16_t>(logits, labels, dlogits, row_loss, count_out, rows, vocab, ignore_index, st);
    else ce_launch<float>(logits, labels, dlogits, row_loss, count_out, rows, vocab, ignore_index, st);
  }
  hipLaunchKernelGGL(ce_loss_reduce_kernel, dim3(1), dim3(kCeThreads), 0, st, row_loss, rows, count_out, loss_out);
  return mlts_check_launch("mlts_ce_fwd_bwd");
}

extern "C" int mlts_scale_by_device_scalar(void* x, const float* scale, int64_t n, int32_t dtype,
                                           mlts_stream_t stream) {
  MLTS_REQUIRE(dtype == MLTS_BF16 || dtype == MLTS_F32, "mlts_scale_by_device_scalar: unknown dtype %d", dtype);
  MLTS_REQUIRE(n >= 0, "mlts_scale_by_device_scalar: n must be >= 0");
  if (n == 0) return MLTS_OK;
  MLTS_REQUIRE(x && scale, "mlts_scale_by_device_scalar: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (mlts_aligned16(x)) {
    const int64_t per = dtype == MLTS_BF16 ? 8 : 4;
    const int64_t n_vec = n / per;
    int64_t blocks = (n_vec + 255) / 256;
    blocks = blocks < 1 ? 1 : (blocks > 1024 ? 1024 : blocks);  // four per CU stream as fast, and leave early in the usual case
    if (dtype == MLTS_BF16)
      hipLaunchKernelGGL(scale_by_scalar_vec_kernel<bf16_t>, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<bf16_t*>(x), scale, n_vec, n);
    else
      hipLaunchKernelGGL(scale_by_scalar_vec_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<float*>(x), scale, n_vec, n);
    return mlts_check_launch("mlts_scale_by_device_scalar");
  }
  int64_t blocks = (n + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  if (dtype == MLTS_BF16)
    hipLaunchKernelGGL(scale_by_scalar_kernel<bf16_t>, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<bf16_t*>(x), scale, n);
  else
    hipLaunchKernelGGL(scale_by_scalar_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<float*>(x), scale, n);
  return mlts_check_launch("mlts_scale_by_device_scalar");
}
