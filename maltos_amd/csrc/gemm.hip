// Matrix products of the linear layers: C = A B for row-major operands in the three forms a layer needs,
//   NT  y  = x W^T      A [M, K], B [N, K]     both contiguous along the contraction
//   NN  dx = dy W       A [M, K], B [K, N]
//   TN  dW = dy^T x     A [K, M], B [K, N]     optionally added onto C, the contraction split over workgroups
// in bf16 (v_mfma_f32_32x32x16_bf16) and fp32 (v_mfma_f32_32x32x2_f32: true fp32 products and sums).  fp32 accumulation, one
// rounding at the end.
//
// Why not the vendor library for these: through torch a product costs 18 us of host time whatever its size (a launch is 4), and
// for 1000-token micro-batches of 512-wide layers the library's kernels take 9-20 us where the work is 0.5-3 GFLOP.
//
// A workgroup computes a BM x BN tile of C.  A [BM][128 bytes] slab of A and of B travels global -> registers -> LDS, two LDS
// stages: while a slab is multiplied the next one is written to the other stage and the one after that is on its way from
// memory, with one barrier per slab.  Loads go through buffer descriptors, whose bounds check supplies the zeros past the end
// of an operand.  Rows along the contraction are padded by 16 bytes in LDS (16-byte fragment reads conflict free); rows along
// M or N by 64 (transpose reads, bf16) or 32 bytes (4-byte reads, fp32).  The product is computed with the operands swapped, so
// that a lane holds four neighbouring columns of one row of C, and leaves through LDS in whole row segments.
#include "common.hpp"

namespace {

constexpr int FORM_NT = MLTS_GEMM_NT, FORM_NN = MLTS_GEMM_NN, FORM_TN = MLTS_GEMM_TN;

typedef short i16x4 __attribute__((ext_vector_type(4)));
#define MLTS_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr uint32_t kOutside = 0x80000000u;  // an offset past every operand (operands are smaller than 2 GiB)

template <typename T>
struct Elem;
template <>
struct Elem<bf16_t> {
  static constexpr int BK = 64;    // contraction elements per slab: 128 bytes
  static constexpr int STEP = 16;  // ... per fragment
  static constexpr int PAD = 64;   // bytes behind a row along M / N
  typedef bf16x8 frag;
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Elem<float> {
  static constexpr int BK = 32;
  static constexpr int STEP = 8;
  static constexpr int PAD = 32;
  typedef f32x4 frag;
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], c, 0, 0, 0);
    return c;
  }
};

// One operand's slab: ROWS rows (of C's rows or columns), KC: the contraction is its contiguous dimension.
template <typename T, int ROWS, bool KC, int THREADS, int SETS>
struct Slab {
  static constexpr int ES = static_cast<int>(sizeof(T));
  static constexpr int BK = Elem<T>::BK;
  static constexpr int LINES = KC ? ROWS : BK;                 // lines in memory order
  static constexpr int LINE_BYTES = KC ? 128 : ROWS * ES;
  static constexpr int STRIDE = LINE_BYTES + (KC ? 16 : Elem<T>::PAD);
  static constexpr int BYTES = LINES * STRIDE;
  static constexpr int CHUNKS = LINE_BYTES / 16;               // 16-byte chunks per line
  static constexpr int PER = LINES * CHUNKS / THREADS;         // chunks per lane
  static_assert(LINES * CHUNKS % THREADS == 0, "whole chunks per lane");

  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t offset[PER];
  uint32_t advance;
  u32x4 reg[SETS][PER];

  // base: first element of the slab's first row (KC) or column; ld: elements between lines; lines / line_elems: what exists
  __device__ __forceinline__ void init(const T* base, int64_t ld, int64_t lines, int64_t line_elems, int64_t k_begin) {
    const int64_t bytes = lines > 0 ? ((lines - 1) * ld + line_elems) * ES : 0;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, static_cast<int>(bytes), 0x00020000);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = i * THREADS + threadIdx.x;
      const int64_t line = idx / CHUNKS + (KC ? 0 : k_begin);
      offset[i] = static_cast<uint32_t>((line * ld + (KC ? k_begin : 0)) * ES + (idx % CHUNKS) * 16);
    }
    advance = static_cast<uint32_t>(KC ? 128 : BK * ld * ES);
  }
  // chunk i of the slab at the current offsets; k_left: contraction elements from there to the end
  __device__ __forceinline__ void fetch(int set, int i, int k_left) {
    const int idx = i * THREADS + threadIdx.x;
    const int k = KC ? (idx % CHUNKS) * (16 / ES) : idx / CHUNKS;
    reg[set][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, k < k_left ? offset[i] : kOutside, 0, 0);
    offset[i] += advance;
  }
  __device__ __forceinline__ void store(int set, int i, unsigned char* lds) const {
    const int idx = i * THREADS + threadIdx.x;
    *reinterpret_cast<u32x4*>(lds + (idx / CHUNKS) * STRIDE + (idx % CHUNKS) * 16) = reg[set][i];
  }
  // fragment of rows row0 .. row0 + 31, contraction step ks; lane: row l % 32, contraction STEP * ks + (STEP / 2) * (l / 32) ..
  static __device__ __forceinline__ typename Elem<T>::frag fragment(const unsigned char* lds, int row0, int ks, int lane) {
    const int l32 = lane & 31, hh = lane >> 5;
    if constexpr (KC) {
      return *reinterpret_cast<const typename Elem<T>::frag*>(lds + (row0 + l32) * STRIDE + (2 * ks + hh) * 16);
    } else if constexpr (ES == 2) {
      const int l16 = lane & 15;
      const unsigned char* src = lds + (16 * ks + 8 * hh + (l16 >> 2)) * STRIDE + (row0 + (l32 >> 4) * 16 + (l16 & 3) * 4) * 2;
      const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src));
      const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src + 4 * STRIDE));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      const unsigned char* src = lds + (8 * ks + 4 * hh) * STRIDE + (row0 + l32) * 4;
      f32x4 f;
#pragma unroll
      for (int i = 0; i < 4; ++i) f[i] = *reinterpret_cast<const float*>(src + i * STRIDE);
      return f;
    }
  }
};

struct GemmArgs {
  const void *a, *b;
  void* c;
  float* partial;   // split contraction: [slices][M][N] fp32 in place of c
  int64_t lda, ldb, ldc;
  int M, N;
  int64_t K, k_slice;  // contraction elements per slice (a multiple of the slab)
  int tiles_m, tiles_n, slices;
  int accumulate;
};

template <typename T, int FORM, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_kernel(const GemmArgs g) {
  constexpr int WAVES_N = BN / WN, WAVES = (BM / WM) * WAVES_N, THREADS = WAVES * 64;
  constexpr int MB = WM / 32, NB = WN / 32;
  constexpr int SETS = MB * NB >= 8 ? 1 : 2;  // (eight accumulator blocks leave no registers for a second set)
  typedef Slab<T, BM, FORM != FORM_TN, THREADS, SETS> SA;
  typedef Slab<T, BN, FORM == FORM_NT, THREADS, SETS> SB;
  constexpr int STAGE = SA::BYTES + SB::BYTES;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave / WAVES_N) * WM, wn = (wave % WAVES_N) * WN;

  // Consecutive workgroups go to the eight XCDs in turn; each XCD gets a contiguous run of tiles, walked along N, so that the
  // workgroups that share rows of A share an L2.
  const int tiles = g.tiles_m * g.tiles_n * g.slices;
  int tile = static_cast<int>(blockIdx.x);
  {
    const int per = tiles >> 3, rest = tiles & 7, xcd = tile & 7, pos = tile >> 3;
    tile = xcd * per + min(xcd, rest) + pos;
  }
  const int slice = tile / (g.tiles_m * g.tiles_n);
  tile -= slice * (g.tiles_m * g.tiles_n);
  const int m0 = (tile / g.tiles_n) * BM, n0 = (tile % g.tiles_n) * BN;
  const int64_t k_begin = slice * g.k_slice, k_end = min(g.K, k_begin + g.k_slice);

  SA sa;
  SB sb;
  if (FORM == FORM_TN) sa.init(static_cast<const T*>(g.a) + m0, g.lda, g.K, g.M - m0, k_begin);
  else sa.init(static_cast<const T*>(g.a) + static_cast<int64_t>(m0) * g.lda, g.lda, g.M - m0, g.K, k_begin);
  if (FORM == FORM_NT) sb.init(static_cast<const T*>(g.b) + static_cast<int64_t>(n0) * g.ldb, g.ldb, g.N - n0, g.K, k_begin);
  else sb.init(static_cast<const T*>(g.b) + n0, g.ldb, g.K, g.N - n0, k_begin);

  f32x16 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // One slab ahead in LDS, the next SETS in registers: chunk c of slab s + 1 goes to the other stage and its registers fetch
  // chunk c of slab s + 1 + SETS, a quarter of the chunks behind the products of each fragment step.  (Past the end: zeros, never
  // multiplied.)  With one set a load has the time of one slab to arrive, which short contractions out of HBM exceed.
  constexpr int CHUNKS = SA::PER + SB::PER;
  auto store = [&](int set, int c, unsigned char* stage) {
    if (c < SA::PER) sa.store(set, c, stage);
    else sb.store(set, c - SA::PER, stage + SA::BYTES);
  };
  auto fetch = [&](int set, int c, int k_left) {
    if (c < SA::PER) sa.fetch(set, c, k_left);
    else sb.fetch(set, c - SA::PER, k_left);
  };
  const int slabs = static_cast<int>((k_end - k_begin + Elem<T>::BK - 1) / Elem<T>::BK);
  int k_left = static_cast<int>(k_end - k_begin);
#pragma unroll
  for (int f = 0; f < SETS; ++f) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) fetch(f, c, k_left);
    k_left -= Elem<T>::BK;
  }
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) store(0, c, lds);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) fetch(0, c, k_left);
  auto slab = [&](int s, int set) {  // set: registers of slab s + 1
    k_left -= Elem<T>::BK;
    __syncthreads();  // stage s & 1 is written everywhere, and nobody reads the other one any more
    const unsigned char* la = lds + (s & 1) * STAGE;
    const unsigned char* lb = la + SA::BYTES;
    unsigned char* next = lds + (~s & 1) * STAGE;
    typename Elem<T>::frag fa[2][MB], fb[2][NB];
    auto read = [&](int ks) {
#pragma unroll
      for (int j = 0; j < NB; ++j) fb[ks & 1][j] = SB::fragment(lb, wn + 32 * j, ks, lane);
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[ks & 1][i] = SA::fragment(la, wm + 32 * i, ks, lane);
    };
    read(0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) read(ks + 1);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = Elem<T>::mma(fb[ks & 1][j], fa[ks & 1][i], acc[i][j]);
#pragma unroll
      for (int c = ks * CHUNKS / 4; c < (ks + 1) * CHUNKS / 4; ++c) {
        store(set, c, next);
        fetch(set, c, k_left);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (SETS == 1) {
    for (int s = 0; s < slabs; ++s) slab(s, 0);
  } else {
    for (int s = 0; s < slabs; s += 2) {
      slab(s, 1);
      if (s + 1 < slabs) slab(s + 1, 0);
    }
  }

  // acc[i][j][4 q + r]: row wm + 32 i + l % 32 of C, column wn + 32 j + 8 q + 4 hh + r.  Out through LDS, 32 rows at a time.
  __syncthreads();
  constexpr int ROW = WN + 4;  // floats
  float* stage = reinterpret_cast<float*>(lds) + wave * 32 * ROW;
  constexpr int LPR = WN / 4;         // lanes per row, four columns each
  constexpr int RPP = 64 / LPR;       // rows per pass
  const int c4 = (lane % LPR) * 4, col = n0 + wn + c4;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        *reinterpret_cast<f32x4*>(stage + l32 * ROW + 32 * j + 8 * q + 4 * hh) = v;
      }
    // (a wavefront reads only what it wrote: LDS operations of a wavefront complete in order)
#pragma unroll
    for (int r = 0; r < 32 / RPP; ++r) {
      const int rr = r * RPP + lane / LPR, row = m0 + wm + 32 * i + rr;
      f32x4 v = *reinterpret_cast<const f32x4*>(stage + rr * ROW + c4);
      if (row >= g.M || col >= g.N) continue;
      if (g.partial) {
        float* p = g.partial + (static_cast<int64_t>(slice) * g.M + row) * g.N + col;
        if (col + 4 <= g.N && (g.N & 3) == 0) {
          *reinterpret_cast<f32x4*>(p) = v;
        } else {
          for (int e = 0; e < 4 && col + e < g.N; ++e) p[e] = v[e];
        }
        continue;
      }
      T* p = static_cast<T*>(g.c) + static_cast<int64_t>(row) * g.ldc + col;
      typedef T t4 __attribute__((ext_vector_type(4)));
      if (col + 4 <= g.N && (g.ldc & 3) == 0) {
        if (g.accumulate) {
          const t4 old = *reinterpret_cast<const t4*>(p);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += to_f32<T>(old[e]);
        }
        t4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(v[e]);
        *reinterpret_cast<t4*>(p) = w;
      } else {
        for (int e = 0; e < 4 && col + e < g.N; ++e) p[e] = from_f32<T>(v[e] + (g.accumulate ? to_f32<T>(p[e]) : 0.f));
      }
    }
  }
}

// C (+)= sum of the slices' fp32 partial products, one rounding
template <typename T, bool ACC>
__global__ __launch_bounds__(256) void gemm_join_kernel(T* __restrict__ c, const float* __restrict__ partial, int slices, int64_t n4) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n4) return;
  typedef T t4 __attribute__((ext_vector_type(4)));
  const f32x4* p = reinterpret_cast<const f32x4*>(partial) + i;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  int k = 0;
  for (; k + 4 <= slices; k += 4) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = p[static_cast<int64_t>(k + u) * n4];
#pragma unroll
    for (int u = 0; u < 4; ++u) s += v[u];
  }
  for (; k < slices; ++k) s += p[static_cast<int64_t>(k) * n4];
  t4 o;
  if (ACC) o = reinterpret_cast<const t4*>(c)[i];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = from_f32<T>(ACC ? s[e] + to_f32<T>(o[e]) : s[e]);
  reinterpret_cast<t4*>(c)[i] = o;
}

struct Plan {
  int tile;    // 0: 64 x 64, 1: 128 x 128, 2: 256 x 128, 3: 256 x 256
  int slices;
  int64_t k_slice;
};
constexpr int kTileM[4] = {64, 128, 256, 256}, kTileN[4] = {64, 128, 128, 256};

// The largest tile that still gives every CU a workgroup; a product with fewer tiles than CUs is split along its contraction
// where that is long.  Best of all tiles and splits (us): NT 16384 x 512 x 512 256x128 15.6 (128x128 16.7, 64x64 19.2, 256x256
// 21.6); NT 16384 x 2752 x 512 256x256 66 (76, 96, 77); NN 1023 x 512 x 32000 256x128 in 16 parts 45 (unsplit 210); TN 512 x
// 512 x 16384 in 32 parts 24 (128x128 in 16: 23); TN 2752 x 512 x 16384 in 4 parts 70 (256x256 in 8: 68); TN 512 x 512 x 1023
// 64x64 unsplit 10.1 (in 4: 12.7).
Plan make_plan(int64_t M, int64_t N, int64_t K, int bk, bool dense) {
  auto tiles = [&](int t) { return ((M + kTileM[t] - 1) / kTileM[t]) * ((N + kTileN[t] - 1) / kTileN[t]); };
  const int64_t slabs = (K + bk - 1) / bk;
  Plan p{0, 1, 0};
  auto split = [&](int64_t least_slabs) {
    while (tiles(p.tile) * p.slices * 2 <= 256 && slabs / (p.slices * 2) >= least_slabs) p.slices *= 2;
  };
  if (tiles(3) >= 240) {
    p.tile = 3;
  } else if (tiles(2) >= 256) {
    p.tile = 2;
  } else if (slabs >= 64 && tiles(2) * (slabs / 8) >= 192) {
    p.tile = 2;
    split(8);
  } else if (tiles(1) >= 256) {
    p.tile = 1;
  } else {
    split(bk == 64 ? 16 : 8);
  }
  if (N % 4 || !dense) p.slices = 1;
  p.k_slice = (slabs + p.slices - 1) / p.slices * bk;
  p.slices = p.k_slice > 0 ? static_cast<int>((K + p.k_slice - 1) / p.k_slice) : 1;
  if (p.slices < 1) p.slices = 1;
  return p;
}

template <typename T, int FORM, int BM, int BN, int WM, int WN>
int launch_tile(const GemmArgs& g, hipStream_t st) {
  constexpr int WAVES = (BM / WM) * (BN / WN), THREADS = WAVES * 64;
  constexpr int stages = 2 * (Slab<T, BM, FORM != FORM_TN, THREADS, 1>::BYTES + Slab<T, BN, FORM == FORM_NT, THREADS, 1>::BYTES);
  constexpr int out = WAVES * 32 * (WN + 4) * 4;
  constexpr int bytes = stages > out ? stages : out;
  static_assert(bytes <= 160 * 1024, "LDS");
  auto kern = gemm_kernel<T, FORM, BM, BN, WM, WN>;
  static MltsLdsOptIn opt_in;
  if (bytes > 48 * 1024) {
    if (hipError_t e = opt_in.reserve(reinterpret_cast<const void*>(kern), bytes); e != hipSuccess) {
      mlts_set_error("mlts_gemm: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
      return MLTS_ERR_LAUNCH;
    }
  }
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(g.tiles_m * g.tiles_n * g.slices)), dim3(THREADS), bytes, st, g);
  return MLTS_OK;
}

template <typename T, int FORM>
int launch_form(int tile, const GemmArgs& g, hipStream_t st) {
  if (tile == 0) return launch_tile<T, FORM, 64, 64, 32, 32>(g, st);
  if (tile == 1) return launch_tile<T, FORM, 128, 128, 64, 64>(g, st);
  if (tile == 2) return launch_tile<T, FORM, 256, 128, 64, 64>(g, st);
  return launch_tile<T, FORM, 256, 256, 128, 64>(g, st);
}

bool small_enough(int64_t lines, int64_t ld, int es) { return lines * ld * es < (int64_t{1} << 31) - 4096; }

}  // namespace

extern "C" const char* mlts_gemm_supports(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc) {
  if (dtype != MLTS_BF16 && dtype != MLTS_F32) return "dtype must be MLTS_F32 or MLTS_BF16";
  if (form < FORM_NT || form > FORM_TN) return "unknown form";
  if (M < 0 || N < 0 || K < 0 || M > 0x7fffffff || N > 0x7fffffff) return "bad shape";
  const int es = dtype == MLTS_BF16 ? 2 : 4, v = 16 / es;
  if (lda % v || ldb % v) return "operand rows must be 16-byte aligned";
  const bool a_kc = form != FORM_TN, b_kc = form == FORM_NT;
  if ((a_kc || b_kc) && K % v) return "the contraction must be a multiple of 16 bytes";
  if (lda < (a_kc ? K : M) || ldb < (b_kc ? K : N) || ldc < N) return "row strides must be at least the row length";
  if (!small_enough(a_kc ? M : K, lda, es) || !small_enough(b_kc ? N : K, ldb, es)) return "operands of 2 GiB or more";
  return nullptr;
}

extern "C" int64_t mlts_gemm_workspace_bytes(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0) return 0;
  const Plan p = make_plan(M, N, K, dtype == MLTS_BF16 ? 64 : 32, true);
  return p.slices > 1 ? M * N * 4 * p.slices : 0;
}

extern "C" int mlts_gemm(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K, const void* a, int64_t lda, const void* b, int64_t ldb,
                         void* c, int64_t ldc, int32_t accumulate, void* workspace, int64_t workspace_bytes, mlts_stream_t stream) {
  const char* why = mlts_gemm_supports(form, dtype, M, N, K, lda, ldb, ldc);
  MLTS_REQUIRE(why == nullptr, "mlts_gemm: %s", why);
  if (M == 0 || N == 0) return MLTS_OK;
  MLTS_REQUIRE(c && (K == 0 || (a && b)), "mlts_gemm: null pointer");
  MLTS_REQUIRE(mlts_aligned16(a) && mlts_aligned16(b) && mlts_aligned16(c), "mlts_gemm: pointers must be 16-byte aligned");
  const Plan p = make_plan(M, N, K, dtype == MLTS_BF16 ? 64 : 32, ldc == N);
  GemmArgs g{};
  g.a = a;
  g.b = b;
  g.c = c;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.M = static_cast<int>(M);
  g.N = static_cast<int>(N);
  g.K = K;
  g.k_slice = p.k_slice;
  g.slices = p.slices;
  g.accumulate = accumulate != 0;
  g.tiles_m = static_cast<int>((M + kTileM[p.tile] - 1) / kTileM[p.tile]);
  g.tiles_n = static_cast<int>((N + kTileN[p.tile] - 1) / kTileN[p.tile]);
  MLTS_REQUIRE(static_cast<int64_t>(g.tiles_m) * g.tiles_n * g.slices < (int64_t{1} << 31), "mlts_gemm: too many tiles");
  if (p.slices > 1) {
    MLTS_REQUIRE(workspace && workspace_bytes >= M * N * 4 * p.slices && mlts_aligned16(workspace), "mlts_gemm: workspace too small or unaligned");
    g.partial = static_cast<float*>(workspace);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  MltsKernelTimer timer("gemm", st);
  int rc;
  if (dtype == MLTS_BF16)
    rc = form == FORM_NT ? launch_form<bf16_t, FORM_NT>(p.tile, g, st)
         : form == FORM_NN ? launch_form<bf16_t, FORM_NN>(p.tile, g, st) : launch_form<bf16_t, FORM_TN>(p.tile, g, st);
  else
    rc = form == FORM_NT ? launch_form<float, FORM_NT>(p.tile, g, st)
         : form == FORM_NN ? launch_form<float, FORM_NN>(p.tile, g, st) : launch_form<float, FORM_TN>(p.tile, g, st);
  if (rc != MLTS_OK) return rc;
  if (p.slices > 1) {
    const int64_t n4 = M * N / 4;
    const dim3 grid(static_cast<unsigned>((n4 + 255) / 256));
    if (dtype == MLTS_BF16) {
      if (accumulate) hipLaunchKernelGGL((gemm_join_kernel<bf16_t, true>), grid, dim3(256), 0, st, static_cast<bf16_t*>(c), g.partial, p.slices, n4);
      else hipLaunchKernelGGL((gemm_join_kernel<bf16_t, false>), grid, dim3(256), 0, st, static_cast<bf16_t*>(c), g.partial, p.slices, n4);
    } else {
      if (accumulate) hipLaunchKernelGGL((gemm_join_kernel<float, true>), grid, dim3(256), 0, st, static_cast<float*>(c), g.partial, p.slices, n4);
      else hipLaunchKernelGGL((gemm_join_kernel<float, false>), grid, dim3(256), 0, st, static_cast<float*>(c), g.partial, p.slices, n4);
    }
  }
  return mlts_check_launch("mlts_gemm");
}
