// fp32 attention without tiles that wavefronts share in LDS: pieces of attn_f32_fwd.hip and attn_f32_bwd.hip.
//
// A wavefront owns 16 or 32 rows (queries in the forward and dQ kernels, keys in the dK/dV kernel) and walks the other side in
// units of 16 or 32 rows.  Everything is computed transposed, S^T = K Q^T and O^T = V^T P^T (dK/dV: S = Q K^T, dV^T = dO^T P), on
// v_mfma_f32_16x16x4_f32 (true fp32 products and sums), so that a lane holds scores of one own row and the second product takes
// them from the registers they were computed in: the 16 x 16 result layout (lane l: column l % 16, rows 4 (l / 16) ..+3) is the
// operand layout of the next product once the contraction index is renumbered, which both operands agree on.
//
// The wavefronts of a workgroup share their own rows and take every `splits`-th unit, so that no two of them read the same walked
// rows: staging those for all of them in LDS would share nothing and cost two barriers a tile.  Each fetches its own straight from memory,
// all as 16-byte loads at head dims 64, 128 and 192, and a product needs them in one of two forms.  The forward kernel fetches K in the
// first and V in the second; the backward kernels, which need K, or Q and dO, in both, fetch the first and turn it into the second through
// LDS of the wavefront's own (Turn below), without a barrier:
//   dot          lane l: row l % 16, columns 16 j + 4 (l / 16) ..+3           (contraction over the columns)
//   accumulate   lane l: row 4 (l / 16) + i, columns NC (l % 16) .. + NC - 1  (contraction over the rows; NC = head_dim / 16: column
//                block db of a product is column NC (l % 16) + db, so that one load feeds NC products)
// The unit behind the one that is multiplied is on its way meanwhile.  The splits' sums meet in LDS at the end.
//
// What bounds it: MFMA (32 cycles per 16x16x4) with the vector work between, by counters 0.63 to 0.77 of the pipe where the chip is full
// (8 x 8 x 1024 and 4 x 8 x 1024; 0.47 at 2 x 8 x 777); below that the fixed 5 us of a launch, a chain of first loads and the join.  Before, four wavefronts staged whole 64-row tiles in LDS, which all of
// them waited for.  Before / now (us; forward, dQ, dK/dV): 2 x 8 heads (4 KV) x 777 causal, head_dim 64: 41 48 90 / 24 36 45;
// 8 x 4 x 256: 15.5 18.8 19.4 / 9.6 13.4 14.6; 1 x 4 x 100: 8.8 10.5 10.2 / 6.0 7.2 8.3; 8 x 8 x 1024: 120 165 216 / 114 132 222;
// 4 x 8 x 1024 unmasked: 132 175 220 / 92 120 192; 2 x 8 x 700, head_dim 96: 48 54 61 / 31 47 54; 4 x 8 x 500 x 1000, head_dim 128:
// 191 352 277 / 81 115 165; packed, 1 x 8 (4) x 2048: 78 83 165 / 52 71 106.
//
// Two blocks of 16 rows to a wavefront in the backward kernels (head dims up to 64) share what is fetched and its way through LDS, for longer
// and fewer chains (us, one / two; blocks of 16 own rows; head_dim 64, causal).  dQ: 8 x 8 heads x 1024, 4096 blocks, 161 / 122, 4 x 8 x 1024, 2048
// blocks, 70 / 69, unmasked 126 / 116, 2 x 8 x 1024 42 / 43.  dK/dV, which fetches most for a row: 4096 blocks 207 / 174, 2048 119 / 93, 1024 63 / 53,
// 704 (4 x 4 x 700) 40 / 36.5, 912 of short walks (6 x 8 x 300) 27.6 / 26, but 8 x 8 x 256 23.4 / 24.1 and 512 blocks (8 x 1024) 36 / 49; head_dim 32, two of
// whose eight-wavefront workgroups share a CU while others are idle, from 1024 blocks on (4 x 4 x 700 23.0 / 27.5).
//
// dK/dV takes the statistics of a unit's queries through LDS, a lane one of them, in place of eight loads a lane and their addresses (before / now):
// 2 x 8 (4) x 777 46 / 42, 8 x 8 x 1024 174 / 159, 2 x 8 (2) x 1024 92 / 81, unmasked 8 x 1024 54.5 / 48.4.  (With registers for four wavefronts a SIMD, 16
// of them spilled, 62, 159, 107, 61.)
#pragma once
#include "attn_rows.hpp"

namespace {

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// How the rows of an operand lie in memory: anywhere; 16-byte aligned and D a multiple of 4; the same, D = DP, rows and row strides (in
// bytes) below 2^24 and every offset below 2^32.
enum { ROWS_ANY, ROWS_VEC, ROWS_WHOLE };

// Wavefronts of a workgroup at most: eight where a wavefront gets by with 256 registers.
constexpr int max_splits(int DP, int LAYOUT) { return DP <= 64 || (DP <= 128 && LAYOUT == ROWS_WHOLE) ? 8 : 4; }

// (a 64-bit product per row takes as many cycles as three MFMAs, and vector work does not hide behind another wavefront's MFMAs)
template <int ROWS>
__device__ __forceinline__ const float* row_of(const float* base, int row, int64_t stride) {
  if (ROWS != ROWS_WHOLE) return base + static_cast<uint32_t>(row) * stride;
  const uint32_t offset = __umul24(static_cast<uint32_t>(row), static_cast<uint32_t>(stride) * 4u);
  return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + offset);
}

// Columns d .. d + 3 of a row, with anything past D: `inside` takes that out where the fragment is used (a select behind the load would
// wait for it).
template <int ROWS>
__device__ __forceinline__ f32x4 load_dot(const float* row, int d, int D) {
  if (ROWS == ROWS_WHOLE) return *reinterpret_cast<const f32x4*>(row + d);
  if (ROWS == ROWS_VEC) return *reinterpret_cast<const f32x4*>(row + (d < D ? d : 0));
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = row[d + e < D ? d + e : 0];
  return v;
}
template <int ROWS>
__device__ __forceinline__ f32x4 inside(f32x4 v, int d, int D) {
  if (ROWS == ROWS_WHOLE) return v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = d + e < D ? v[e] : 0.f;
  return v;
}

// columns c .. c + NC - 1 of a row.  (Past D: anything finite or not; such columns of the result are not stored.)
template <int NC>
struct Columns {
  float v[NC];
  template <int ROWS>
  __device__ __forceinline__ void load(const float* row, int c, int D) {
    constexpr int W = ROWS == ROWS_ANY ? 1 : NC % 4 == 0 ? 4 : 2;
    typedef float vec __attribute__((ext_vector_type(W)));
#pragma unroll
    for (int i = 0; i < NC / W; ++i) {
      const vec x = *reinterpret_cast<const vec*>(row + (ROWS == ROWS_WHOLE || c + W * i < D ? c + W * i : 0));
#pragma unroll
      for (int e = 0; e < W; ++e) v[W * i + e] = x[e];
    }
  }
};
// The same out of a unit's dot fragments, through LDS that belongs to the wavefront alone (its LDS operations complete in order): fetching
// the rows a second time would take as long on their way through the L1 as half of the products they feed.
template <int DP>
struct Turn {
  static constexpr int NC = DP / 16, STRIDE = DP + 4, FLOATS = 16 * STRIDE;  // (16-byte accesses of 16 rows and of 4 are conflict free)
  static __device__ __forceinline__ void put(float* lds, int j, const f32x4 v, int l16, int g) {
    *reinterpret_cast<f32x4*>(lds + l16 * STRIDE + 16 * j + 4 * g) = v;
  }
  static __device__ __forceinline__ void get(Columns<NC> (&rows)[4], const float* lds, int l16, int g) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[i].template load<ROWS_WHOLE>(lds + (4 * g + i) * STRIDE, NC * l16, DP);
  }
};

// acc[db] += walked columns x own rows, for the 16 walked rows of which `rows[i]` are this lane's (row 4 g + i)
template <int NC>
__device__ __forceinline__ void accumulate(f32x4 (&acc)[NC], const Columns<NC> (&rows)[4], const f32x4 x) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int db = 0; db < NC; ++db) acc[db] = mfma4(rows[i].v[db], x[i], acc[db]);
}

// What a row's result becomes before it is stored: nothing else, or rotated back (columns d ..+1 or ..+3; D is then a multiple of 4)
struct AsIs {
  __device__ __forceinline__ void operator()(int, int, float&, float&) const {}
  __device__ __forceinline__ f32x4 operator()(int, int, f32x4 v) const { return v; }
};
template <int N>
struct Back {
  const RotateBack& rot;
  int64_t table[N];  // negative: not rotated
  __device__ __forceinline__ void operator()(int n, int d, float& even, float& odd) const {
    if (table[n] < 0 || d >= 2 * rot.half) return;
    const auto a = rot.angles<float, 1>(table[n], d / 2);
    RotateBack::back<float>(even, odd, a.c[0], a.s[0]);
  }
  __device__ __forceinline__ f32x4 operator()(int n, int d, f32x4 v) const {
    return table[n] < 0 || d >= 2 * rot.half ? v : RotateBack::back<float>(v, rot.angles<float, 2>(table[n], d / 2));
  }
};

// A row's result as it lies in the accumulators: acc[db][r] is column NC (4 g + r) + db.  Times scale, overwritten or added to.
template <int NC, typename F>
__device__ __forceinline__ void store_row(float* row, const f32x4 (&acc)[NC], float scale, int g, int D, bool vec, bool add, int n, const F& finish) {
  f32x4 w[NC];
#pragma unroll
  for (int t = 0; t < NC; ++t) {  // (what is loaded, in front of the first store)
#pragma unroll
    for (int e = 0; e < 4; ++e) w[t][e] = acc[(4 * t + e) % NC][(4 * t + e) / NC] * scale;
    w[t] = finish(n, 4 * NC * g + 4 * t, w[t]);
  }
#pragma unroll
  for (int t = 0; t < NC; ++t) {
    const int d = 4 * NC * g + 4 * t;
    if (vec) {
      if (d >= D) continue;
      f32x4* at = reinterpret_cast<f32x4*>(row + d);
      *at = add ? *at + w[t] : w[t];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d + e < D) row[d + e] = add ? row[d + e] + w[t][e] : w[t][e];
    }
  }
}

// N results of 16 rows each, spread over the splits: summed through LDS (N * DP / 16 KiB a split) and stored, every wavefront a part of
// the columns.  lds: of these splits.  scale, row: as for store_row; row null: not stored.
template <int NC, int N, typename F>
__device__ __forceinline__ void join_and_store(const f32x4 (&acc)[N][NC], float* lds, int split, int splits, float* const (&row)[N], const float (&scale)[N],
                                               int lane, int D, bool vec, bool add, const F& finish) {
  const int g = lane >> 4;
  if (splits == 1) {
#pragma unroll
    for (int n = 0; n < N; ++n)
      if (row[n]) store_row(row[n], acc[n], scale[n], g, D, vec, add, n, finish);
    return;
  }
  __syncthreads();  // nobody needs what the LDS holds any more
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int db = 0; db < NC; ++db) lds[(((split * N + n) * 4 + e) * NC + db) * 64 + lane] = acc[n][db][e];
  __syncthreads();
#pragma unroll
  for (int n = 0; n < N; ++n) {
    for (int e = (split - 4 * n) & (splits - 1); e < 4; e += splits) {
      float v[NC];
#pragma unroll
      for (int db = 0; db < NC; ++db) v[db] = 0.f;
      for (int s = 0; s < splits; ++s)
#pragma unroll
        for (int db = 0; db < NC; ++db) v[db] += lds[(((s * N + n) * 4 + e) * NC + db) * 64 + lane];
      if (!row[n]) continue;
      const int d = NC * (4 * g + e);
#pragma unroll
      for (int db = 0; db < NC; ++db) v[db] *= scale[n];
      if constexpr (NC % 4 == 0) {
#pragma unroll
        for (int t = 0; t < NC; t += 4) {
          const f32x4 w = finish(n, d + t, f32x4{v[t], v[t + 1], v[t + 2], v[t + 3]});
#pragma unroll
          for (int e = 0; e < 4; ++e) v[t + e] = w[e];
        }
      } else {
#pragma unroll
        for (int db = 0; db < NC; db += 2) finish(n, d + db, v[db], v[db + 1]);
      }
      if (vec && NC % 4 == 0) {
#pragma unroll
        for (int t = 0; t < NC / 4; ++t) {
          if (d + 4 * t >= D) continue;
          f32x4* at = reinterpret_cast<f32x4*>(row[n] + d + 4 * t);
          const f32x4 w = {v[4 * t], v[4 * t + 1], v[4 * t + 2], v[4 * t + 3]};
          *at = add ? *at + w : w;
        }
      } else {
#pragma unroll
        for (int db = 0; db < NC; ++db)
          if (d + db < D) row[n][d + db] = add ? row[n][d + db] + v[db] : v[db];
      }
    }
  }
}

// Document masks: ids of the own rows, as ranges, and which of the walked rows they concern.
struct IdRange {
  int pos_min, pos_max, seq_min, seq_max;
};
__device__ __forceinline__ IdRange id_range(const int32_t* pos, const int32_t* seq, int row0, int rows, int limit, int lane) {
  IdRange r{0x7fffffff, -0x7fffffff - 1, 0x7fffffff, -0x7fffffff - 1};
  const int i = row0 + lane;
  if (lane < rows && i < limit) {
    r.pos_min = r.pos_max = pos[i];
    r.seq_min = r.seq_max = seq[i];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    r.pos_min = min(r.pos_min, __shfl_xor(r.pos_min, o, 64));
    r.pos_max = max(r.pos_max, __shfl_xor(r.pos_max, o, 64));
    r.seq_min = min(r.seq_min, __shfl_xor(r.seq_min, o, 64));
    r.seq_max = max(r.seq_max, __shfl_xor(r.seq_max, o, 64));
  }
  return r;
}

// The units (16 rows) of the walked side that a split works on, in order: every splits-th; under a document mask those of them
// that hold a row some own row may see (KEYS: the walked rows are keys; else queries), found 256 rows at a time, four a lane.
template <bool DOC, bool KEYS>
struct Units {
  const int32_t *pos, *seq;
  IdRange own;
  int split, splits, end, lane;  // end: rows walked
  int base;                      // DOC: rows of the current look
  unsigned long long left;       // DOC: its units that are left, one bit each (the unit's lowest)

  __device__ __forceinline__ void look() {
    bool some = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = base + 4 * lane + e;
      if (r < end) {
        const int p = pos[r], s = seq[r];
        some |= (KEYS ? p <= own.pos_max : p >= own.pos_min) && s >= own.seq_min && s <= own.seq_max && s >= 0;
      }
    }
    unsigned long long m = __builtin_amdgcn_ballot_w64(some);
    m |= m >> 1;
    m |= m >> 2;
    unsigned long long mine = 0;  // the lowest of the four bits of each unit of this split
#pragma unroll
    for (int u = 0; u < 16; ++u) mine |= static_cast<unsigned long long>((u & (splits - 1)) == split) << (4 * u);
    left = m & mine;
  }
  // first: the walked row to start from (DOC: 0)
  __device__ __forceinline__ int first(int start) {
    if (!DOC) return start + 16 * split;
    base = -256, left = 0;
    return next(0);
  }
  __device__ __forceinline__ int next(int row) {
    if (!DOC) return row + 16 * splits;
    while (left == 0) {
      base += 256;
      if (base >= end) return end;
      look();
    }
    const int bit = __builtin_ctzll(left);
    left &= left - 1;
    return base + 4 * bit;
  }
};

inline bool rows_vec(const int64_t* s, const void* ptr) { return ((s[0] | s[1] | s[2]) & 3) == 0 && mlts_aligned16(ptr); }

inline bool rows_near(int64_t rows, int64_t stride, int D) {
  return rows < (1 << 24) && stride < (1 << 22) && ((rows - 1) * stride + D) * 4 < (int64_t{1} << 32);
}

}  // namespace

#define MLTS_F32_DISPATCH_DP(FN, DOC, ROWS, ...)         \
  do {                                                   \
    if (D <= 32) return FN<32, DOC, ROWS>(__VA_ARGS__);  \
    if (D <= 64) return FN<64, DOC, ROWS>(__VA_ARGS__);  \
    if (D <= 96) return FN<96, DOC, ROWS>(__VA_ARGS__);  \
    if (D <= 128) return FN<128, DOC, ROWS>(__VA_ARGS__); \
    if (D <= 160) return FN<160, DOC, ROWS>(__VA_ARGS__); \
    return FN<192, DOC, ROWS>(__VA_ARGS__);              \
  } while (0)
#define MLTS_F32_DISPATCH_ROWS(FN, DOC, ...)                                         \
  do {                                                                               \
    if (whole) MLTS_F32_DISPATCH_DP(FN, DOC, ROWS_WHOLE, __VA_ARGS__);  \
    if (vec) MLTS_F32_DISPATCH_DP(FN, DOC, ROWS_VEC, __VA_ARGS__);                   \
    MLTS_F32_DISPATCH_DP(FN, DOC, ROWS_ANY, __VA_ARGS__);                            \
  } while (0)
#define MLTS_F32_DISPATCH(FN, ...)                                         \
  do {                                                                     \
    if (mode == MLTS_MASK_DOC) MLTS_F32_DISPATCH_ROWS(FN, true, __VA_ARGS__); \
    MLTS_F32_DISPATCH_ROWS(FN, false, __VA_ARGS__);                        \
  } while (0)
