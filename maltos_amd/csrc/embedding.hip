// Gradient of the token embedding: dw[ids[t]] += dy[t] over all tokens t, equal ids summed in fp32 in a fixed order, added onto dw
// and rounded once.  Rows no token names are not touched.
//
// The work is one read of dy; what costs is finding the tokens of a row without atomics.  A sort of the ids takes seven launches
// and 90 us at 16384 tokens, and a gradient of the whole table (32 MB for 32000 x 512) written and added afterwards another 50.
// Here each of 256 workgroups (one per CU) owns the rows whose id leaves its remainder mod 256, reads ALL ids (128 KB at 16384
// tokens, from L2), keeps the matching tokens in order as a list in LDS, and then a wavefront takes one distinct id at a time and
// sums its rows.  An id with more than kHeavy tokens (padding) is summed by the whole workgroup instead, its wavefronts' sums
// joined in LDS.  50M model, per step: 16384 tokens 190 -> 22 us, 1024 tokens 95 -> 6 us (sort or scan, clear and add included).
#include "common.hpp"

namespace {

constexpr int kBuckets = 256;
constexpr int kWaves = 16, kThreads = kWaves * MLTS_WAVE;
constexpr int kMaxTokens = 28 * 1024;  // the list: 4 bytes a token, 112 KB, beside 32 KB of sums
constexpr int kHeavy = 64;

// sum of the listed rows with this key among entries first, first + 64 * step, ..., columns col .. col + N - 1 (lane's own)
template <typename T>
__device__ __forceinline__ void sum_rows(const uint32_t* list, int total, int first, int step, uint32_t key, const T* dy, int64_t hidden, int64_t col,
                                         bool inside, float* acc) {
  constexpr int N = Vec16<T>::N;
  const int lane = threadIdx.x & 63;
  for (int base = first; base < total; base += 64 * step) {
    const uint32_t e = base + lane < total ? list[base + lane] : 0xffffffffu;
    uint64_t hits = __ballot(base + lane < total && (e >> 16) == key);
    while (hits) {
      Vec16<T> v[4];
      int count = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (hits) {
          const int src = __ffsll(static_cast<unsigned long long>(hits)) - 1;
          hits &= hits - 1;
          const int64_t t = __builtin_amdgcn_readlane(e, src) & 0xffffu;
          if (inside) v[u] = *reinterpret_cast<const Vec16<T>*>(dy + t * hidden + col);
          count = u + 1;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (u < count)
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += v[u].get(j);
    }
  }
}

template <typename T>
__device__ __forceinline__ void add_row(T* p, const float* acc) {
  constexpr int N = Vec16<T>::N;
  Vec16<T> old = *reinterpret_cast<const Vec16<T>*>(p), out;
#pragma unroll
  for (int j = 0; j < N; ++j) out.set(j, old.get(j) + acc[j]);
  *reinterpret_cast<Vec16<T>*>(p) = out;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void embedding_bwd_kernel(const int64_t* __restrict__ ids, const T* __restrict__ dy, T* __restrict__ dw, int n,
                                                                 int64_t hidden, int64_t vocab) {
  constexpr int N = Vec16<T>::N;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  float* sums = reinterpret_cast<float*>(lds);                            // [kWaves][64 * N]
  uint32_t* heavy = reinterpret_cast<uint32_t*>(sums + kWaves * 64 * N);  // keys of the ids left to the whole workgroup
  uint32_t* list = heavy + kMaxTokens / kHeavy;                           // (id / 256) << 16 | token, in token order
  __shared__ int counts[kWaves];
  __shared__ int heavy_count;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t bucket = blockIdx.x;
  if (threadIdx.x == 0) heavy_count = 0;

  // the wavefront's own run of tokens: which of them are this bucket's (step j: bit j), how many
  const int steps = (n + kThreads - 1) / kThreads, begin = wave * steps * 64;
  uint32_t mine = 0;
  int found = 0;
  for (int j0 = 0; j0 < steps; j0 += 8) {
    int64_t id[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = begin + (j0 + u) * 64 + lane;
      id[u] = j0 + u < steps && t < n ? ids[t] : -1;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool hit = id[u] >= 0 && id[u] < vocab && (id[u] & (kBuckets - 1)) == bucket;
      if (hit) mine |= 1u << (j0 + u);
      found += __popcll(__ballot(hit));
    }
  }
  if (lane == 0) counts[wave] = found;
  __syncthreads();
  int at = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) at += counts[w];
    total += counts[w];
  }
  if (found)
    for (int j = 0; j < steps; ++j) {
      const bool hit = (mine >> j) & 1;
      const uint64_t hits = __ballot(hit);
      if (hit) {
        const int t = begin + j * 64 + lane;
        list[at + __popcll(hits & ((uint64_t{1} << lane) - 1))] = static_cast<uint32_t>(ids[t] >> 8) << 16 | static_cast<uint32_t>(t);
      }
      at += __popcll(hits);
    }
  __syncthreads();

  for (int i = wave; i < total; i += kWaves) {
    const uint32_t key = __builtin_amdgcn_readfirstlane(list[i] >> 16);
    bool first = true;
    int count = 0;
    for (int base = 0; base < total && first; base += 64) {
      const uint64_t hits = __ballot(base + lane < total && (list[min(base + lane, total - 1)] >> 16) == key);
      if (base + 64 <= i) first = hits == 0;
      else if (base <= i) first = (hits & ((uint64_t{1} << (i - base)) - 1)) == 0;
      count += __popcll(hits);
    }
    if (!first) continue;  // another wavefront has this id
    if (count > kHeavy) {
      if (lane == 0) heavy[atomicAdd(&heavy_count, 1)] = key;
      continue;
    }
    T* row = dw + (static_cast<int64_t>(key) * kBuckets + bucket) * hidden;
    for (int64_t c0 = 0; c0 < hidden; c0 += 64 * N) {
      const int64_t col = c0 + lane * N;
      float acc[N] = {};
      sum_rows<T>(list, total, i & ~63, 1, key, dy, hidden, col, col < hidden, acc);
      if (col < hidden) add_row<T>(row + col, acc);
    }
  }
  __syncthreads();
  for (int h = 0; h < heavy_count; ++h) {
    const uint32_t key = __builtin_amdgcn_readfirstlane(heavy[h]);
    T* row = dw + (static_cast<int64_t>(key) * kBuckets + bucket) * hidden;
    for (int64_t c0 = 0; c0 < hidden; c0 += 64 * N) {
      const int64_t col = c0 + lane * N;
      float acc[N] = {};
      sum_rows<T>(list, total, wave * 64, kWaves, key, dy, hidden, col, col < hidden, acc);
#pragma unroll
      for (int j = 0; j < N; ++j) sums[(wave * 64 + lane) * N + j] = acc[j];
      __syncthreads();
      if (wave == 0) {
        for (int w = 1; w < kWaves; ++w)
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += sums[(w * 64 + lane) * N + j];
        if (col < hidden) add_row<T>(row + col, acc);
      }
      __syncthreads();
    }
  }
}

template <typename T>
int launch(const int64_t* ids, const void* dy, void* dw, int n, int64_t hidden, int64_t vocab, hipStream_t st) {
  const int fixed = kWaves * 64 * Vec16<T>::N * 4 + kMaxTokens / kHeavy * 4, bytes = fixed + n * 4;
  static_assert(kWaves * 64 * 8 * 4 + kMaxTokens / kHeavy * 4 + kMaxTokens * 4 + 256 <= 160 * 1024, "LDS");
  auto kern = embedding_bwd_kernel<T>;
  static MltsLdsOptIn opt_in;
  if (hipError_t e = opt_in.reserve(reinterpret_cast<const void*>(kern), fixed + kMaxTokens * 4); e != hipSuccess) {
    mlts_set_error("mlts_embedding_bwd: cannot reserve %d bytes of LDS: %s", fixed + kMaxTokens * 4, hipGetErrorString(e));
    return MLTS_ERR_LAUNCH;
  }
  MltsKernelTimer timer("embedding_bwd", st);
  hipLaunchKernelGGL(kern, dim3(kBuckets), dim3(kThreads), bytes, st, ids, static_cast<const T*>(dy), static_cast<T*>(dw), n, hidden, vocab);
  return mlts_check_launch("mlts_embedding_bwd");
}

}  // namespace

extern "C" const char* mlts_embedding_bwd_supports(int64_t n, int64_t hidden, int64_t vocab, int32_t dtype) {
  if (dtype != MLTS_BF16 && dtype != MLTS_F32) return "dtype must be MLTS_F32 or MLTS_BF16";
  if (n < 0 || n > kMaxTokens) return "too many tokens for one list";
  if (vocab < 0 || vocab > (int64_t{1} << 24)) return "more than 2^24 rows";
  if (hidden <= 0 || hidden % (dtype == MLTS_BF16 ? 8 : 4)) return "rows must be whole 16-byte vectors";
  return nullptr;
}

extern "C" int mlts_embedding_bwd(const int64_t* ids, const void* dy, void* dw, int64_t n, int64_t hidden, int64_t vocab, int32_t dtype,
                                  mlts_stream_t stream) {
  const char* why = mlts_embedding_bwd_supports(n, hidden, vocab, dtype);
  MLTS_REQUIRE(why == nullptr, "mlts_embedding_bwd: %s", why);
  if (n == 0) return MLTS_OK;
  MLTS_REQUIRE(ids && dy && dw, "mlts_embedding_bwd: null pointer");
  MLTS_REQUIRE(mlts_aligned16(dy) && mlts_aligned16(dw), "mlts_embedding_bwd: pointers must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == MLTS_BF16 ? launch<bf16_t>(ids, dy, dw, static_cast<int>(n), hidden, vocab, st)
                            : launch<float>(ids, dy, dw, static_cast<int>(n), hidden, vocab, st);
}
