// Attention on 16-row wavefront tiles: bf16 at head dims <= 192 that neither the 32-row kernels nor attn_small.hip cover (documents, rows at
// any alignment, head dims other than 32, 64, 96 and 128).
//
// A wavefront owns 16 rows (queries in the forward and dQ kernels, keys in the dK/dV kernel) and walks the other side in
// units of 32, staged in LDS 64 at a time.  Everything is computed transposed, S^T = K Q^T and O^T = V^T P^T (dK/dV: S = Q K^T,
// dV^T = dO^T P), so that a lane holds the scores of ONE of its wavefront's rows and the second product takes them from the
// registers they were computed in: the 16 x 16 result layout (lane l: column l % 16, rows 4 (l / 16) ..+3) is the operand
// layout of the next product once the contraction index is renumbered, which both operands agree on.
//
// Products run on v_mfma_f32_16x16x32_bf16.  Probabilities and dS enter their second product as the sum of three bf16 values of 8
// bits each, which is all of an fp32 number: products and sums as with fp32 probabilities.  (Two of them are enough for a bf16
// output, but not for gradients added in fp32: 2.5e-6 off the exact ones at S = 777, with three 0.3 to 0.5e-6.  The third
// costs a few percent where a kernel is short, 9 to 15 where it fills the chip: 8 x 8 heads x 1024, head_dim 32, forward and
// backward 27 + 68 us with two, 30 + 77 with three.)
//
// What bounds it: the matrix pipe for long rows, the chain of tiles of one workgroup for short ones.  A workgroup is four
// wavefronts: 64 rows, or, when the grid would leave compute units idle, 32 rows with the two halves of every tile on different
// wavefronts (joined in LDS at the end).
#include "attn_common.hpp"

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kTile = 64;  // rows of the walked side per LDS stage: two units of 32
constexpr int kVec = 8;    // elements of a 16-byte vector: a fragment

typedef short i16x4 __attribute__((ext_vector_type(4)));

#define MLTS_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

// DP: head_dim rounded up to a multiple of 32 (the padding is zero in every operand)
template <int DP>
struct Tile16 {
  static constexpr int STEP = 32;
  static constexpr int FRAGS = DP / STEP;
  static constexpr int LS = DP + 8;
  static __device__ __forceinline__ f32x4 dot(bf16x8 a, bf16x8 b, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  }
  static __device__ __forceinline__ void accumulate(f32x4 (&acc)[DP / 16], const bf16_t* unit, const f32x4 (&x)[2], int l16, int g) {
    bf16x8 part[3];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float rest = x[b][i];
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          part[n][4 * b + i] = static_cast<bf16_t>(rest);
          rest -= static_cast<float>(part[n][4 * b + i]);
        }
      }
    const bf16_t* src = unit + (4 * g + (l16 >> 2)) * LS + (l16 & 3) * 4;
#pragma unroll
    for (int db = 0; db < DP / 16; ++db) {
      const i16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src + 16 * db));
      const i16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src + 16 * LS + 16 * db));
      const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(r0, r1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
      for (int n = 0; n < 3; ++n) acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, part[n], acc[db], 0, 0, 0);
    }
  }
};

// columns d0 .. d0 + kVec - 1 of a row, zero past D (and everywhere if the row does not exist)
__device__ __forceinline__ bf16x8 load_frag(const bf16_t* row, bool exists, int d0, int D, bool vec) {
  bf16x8 f;
#pragma unroll
  for (int e = 0; e < kVec; ++e) f[e] = static_cast<bf16_t>(0.f);
  if (!exists) return f;
  if (vec) {
    if (d0 < D) f = *reinterpret_cast<const bf16x8*>(row + d0);
  } else {
#pragma unroll
    for (int e = 0; e < kVec; ++e)
      if (d0 + e < D) f[e] = row[d0 + e];
  }
  return f;
}

// A [64][DP] tile on its way from global memory to LDS through registers: fetched while the tile before it is worked on.
template <int DP>
struct Stage {
  static constexpr int CHUNKS = DP / kVec;                       // 16-byte chunks per row
  static constexpr int N = kTile * CHUNKS / kThreads;            // chunks per lane
  static_assert(kTile * CHUNKS % kThreads == 0, "whole chunks per lane");
  bf16x8 r[N];
  __device__ __forceinline__ void fetch(const bf16_t* base, int64_t row_stride, int row0, int limit, int D, bool vec) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int idx = n * kThreads + threadIdx.x;
      const int row = row0 + idx / CHUNKS;
      r[n] = load_frag(base + static_cast<int64_t>(row) * row_stride, row < limit, (idx % CHUNKS) * kVec, D, vec);
    }
  }
  __device__ __forceinline__ void store(bf16_t* lds) const {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int idx = n * kThreads + threadIdx.x;
      *reinterpret_cast<bf16x8*>(lds + (idx / CHUNKS) * Tile16<DP>::LS + (idx % CHUNKS) * kVec) = r[n];
    }
  }
};

// e^x.  Scores, maxima and log-sum-exps stay in natural units and are subtracted first: what is rounded on the way into the hardware's
// 2^x is then a difference that is near 0 wherever the probability counts, and not a score (with the scores multiplied by log2 e
// before the subtraction the errors were up to 1.25 times as large).  expf would take up to 60 % of the kernels' time.
__device__ __forceinline__ float exponential(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

struct Tile16Args {
  int D;
  int row_waves;  // wavefronts over the owned rows: 4, or 2 (the others work on the other of a tile's two units)
  bool vec;       // every row of every tensor is 16-byte aligned and D a multiple of the 16-byte vector
};

__device__ __forceinline__ float sum_groups(float x) {  // over the four 16-lane groups: the lanes that share an own row
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}
__device__ __forceinline__ float max_groups(float x) {
  x = fmaxf(x, __shfl_xor(x, 16, 64));
  return fmaxf(x, __shfl_xor(x, 32, 64));
}

// One row's columns 16 db + 4 g ..+3 as they lie in the accumulators.  mode 0: bf16, overwritten; 1: fp32, added to; 2: fp32, overwritten.
template <int DP>
__device__ __forceinline__ void store_row(void* base, int64_t off, const f32x4 (&acc)[DP / 16], float scale, int g, int D, bool vec, int mode) {
#pragma unroll
  for (int db = 0; db < DP / 16; ++db) {
    const int d = 16 * db + 4 * g;
    if (mode == 0 && vec) {
      bf16x4 w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = from_f32<bf16_t>(acc[db][i] * scale);
      if (d < D) *reinterpret_cast<bf16x4*>(static_cast<bf16_t*>(base) + off + d) = w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (d + i >= D) continue;
        const float x = acc[db][i] * scale;
        float* f = static_cast<float*>(base) + off + d + i;
        if (mode == 0) static_cast<bf16_t*>(base)[off + d + i] = from_f32<bf16_t>(x);
        else if (mode == 1) *f += x;
        else *f = x;
      }
    }
  }
}

// Document masks: can any of the 64 walked rows at t0 be seen by / see the block?  Evaluated by every wavefront on the same
// rows, so the answer is uniform over the workgroup.
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

// Joins the accumulators of the wavefronts that split the tiles of the same rows: all add onto the one with split 0, through LDS.
template <int N>
__device__ __forceinline__ void join_splits(f32x4 (&acc)[N], float* lds, int row_wave, int row_waves, int split, int splits, int lane) {
  __syncthreads();
  f32x4* base = reinterpret_cast<f32x4*>(lds) + lane;
  if (split > 0) {
#pragma unroll
    for (int n = 0; n < N; ++n) base[(((split - 1) * row_waves + row_wave) * N + n) * 64] = acc[n];
  }
  __syncthreads();
  if (split == 0) {
    for (int s = 1; s < splits; ++s)
#pragma unroll
      for (int n = 0; n < N; ++n) acc[n] += base[(((s - 1) * row_waves + row_wave) * N + n) * 64];
  }
}

template <int DP, bool DOC>
__global__ __launch_bounds__(kThreads) void attn_tile16_fwd(const AttnParams p, const Tile16Args a) {
  typedef Tile16<DP> C;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  bf16_t* sK = reinterpret_cast<bf16_t*>(lds_raw);
  bf16_t* sV = sK + kTile * C::LS;
  int2* sIds = reinterpret_cast<int2*>(sV + kTile * C::LS);
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row_wave = wave & (a.row_waves - 1), split = wave / a.row_waves, splits = kWaves / a.row_waves;
  const int unit0 = split, unit_step = splits;
  const int rows = a.row_waves * 16;
  // last blocks first: with a causal mask they are the long ones
  const int nbh = p.B * p.Hq, qt = p.nqt - 1 - static_cast<int>(blockIdx.x) / nbh, bh = static_cast<int>(blockIdx.x) % nbh;
  const int b = bh / p.Hq, hq = bh % p.Hq, hkv = hq / (p.Hq / p.Hkv);
  const int q0 = qt * rows, qrow = q0 + row_wave * 16 + l16;
  const bf16_t* Q = static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1];
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1];

  bf16x8 qf[C::FRAGS];
#pragma unroll
  for (int j = 0; j < C::FRAGS; ++j)
    qf[j] = load_frag(Q + static_cast<int64_t>(min(qrow, p.Sq - 1)) * p.qs[2], true, C::STEP * j + kVec * g, a.D, a.vec);
  // keys this lane's query sees: up to klim (p.causal_off is Sk without a causal mask); documents also by their ids
  const int klim = qrow < p.Sq ? min(p.Sk - 1, qrow + p.causal_off) : -1;
  int kend = p.Sk, qpos = 0, qseq = -1;
  const int32_t *kpos = nullptr, *kseq = nullptr;
  IdRange blk{};
  if (DOC) {
    kpos = p.k_pos + static_cast<int64_t>(b) * p.Sk;
    kseq = p.k_seq + static_cast<int64_t>(b) * p.Sk;
    const int32_t *qp = p.q_pos + static_cast<int64_t>(b) * p.Sq, *qs = p.q_seq + static_cast<int64_t>(b) * p.Sq;
    if (qrow < p.Sq) qpos = qp[qrow], qseq = qs[qrow];
    blk = id_range(qp, qs, q0, rows, p.Sq, lane);
  } else {
    kend = max(0, min(p.Sk, min(q0 + rows, p.Sq) + p.causal_off));
  }
  const int wave_klim = DOC ? 0 : min(p.Sk - 1, min(q0 + row_wave * 16, p.Sq - 1) + p.causal_off);        // seen by every row of the wavefront
  const int wave_kmax = DOC ? p.Sk : min(q0 + row_wave * 16 + 15, p.Sq - 1) + p.causal_off;               // last key any of its rows sees
  auto next_tile = [&](int k) {
    if (DOC) {
      for (; k < kend; k += kTile) {
        const int kj = k + lane;
        bool some = false;
        if (kj < p.Sk) {
          const int kp = kpos[kj], ks = kseq[kj];
          some = kp <= blk.pos_max && ks >= blk.seq_min && ks <= blk.seq_max && ks >= 0;
        }
        if (__builtin_amdgcn_ballot_w64(some) != 0) break;
      }
    }
    return k;
  };

  float m = -INFINITY, l = 0.f;
  f32x4 o[DP / 16];
#pragma unroll
  for (int db = 0; db < DP / 16; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  Stage<DP> stK, stV;
  int2 ids = make_int2(0, -2);
  int k0 = next_tile(0);
  auto fetch = [&](int k) {
    stK.fetch(K, p.ks[2], k, p.Sk, a.D, a.vec);
    stV.fetch(V, p.vs[2], k, p.Sk, a.D, a.vec);
    if (DOC && tid < kTile) ids = k + tid < p.Sk ? make_int2(kpos[k + tid], kseq[k + tid]) : make_int2(0, -2);
  };
  if (k0 < kend) fetch(k0);
  while (k0 < kend) {
    __syncthreads();
    stK.store(sK);
    stV.store(sV);
    if (DOC && tid < kTile) sIds[tid] = ids;
    __syncthreads();
    const int kn = next_tile(k0 + kTile);
    if (kn < kend) fetch(kn);
    for (int u = unit0; u < 2; u += unit_step) {
      const int ku = k0 + 32 * u;
      if (ku >= p.Sk || ku > wave_kmax) continue;
      const bf16_t* ku_rows = sK + (32 * u + l16) * C::LS + kVec * g;
      f32x4 s[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < C::FRAGS; ++j)
          s[kb] = C::dot(*reinterpret_cast<const bf16x8*>(ku_rows + 16 * kb * C::LS + C::STEP * j), qf[j], s[kb]);
      }
      if (DOC) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int2 id = sIds[32 * u + 16 * kb + 4 * g + i];
            if (!(id.x <= qpos && id.y == qseq && qseq >= 0)) s[kb][i] = -INFINITY;
          }
      } else if (ku + 31 > wave_klim) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (ku + 16 * kb + 4 * g + i > klim) s[kb][i] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kb][i]);
      mx = max_groups(mx) * p.scale;
      if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
        const float m_new = fmaxf(m, mx);
        const float alpha = exponential(m - (m_new == -INFINITY ? 0.f : m_new));  // 1 for rows that do not rise, 0 from -inf
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int db = 0; db < DP / 16; ++db) o[db] *= alpha;
      }
      const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[kb][i] = exponential(s[kb][i] * p.scale - m_use);
          l += s[kb][i];
        }
      C::accumulate(o, sV + 32 * u * C::LS, s, l16, g);
    }
    k0 = kn;
  }
  l = sum_groups(l);
  if (splits > 1) {  // several wavefronts hold parts of every tile for the same rows: bring all to the largest maximum
    float* ml = reinterpret_cast<float*>(lds_raw);
    __syncthreads();
    if (g == 0) ml[wave * 32 + l16] = m, ml[wave * 32 + 16 + l16] = l;
    __syncthreads();
    float m_new = -INFINITY;
    for (int s = 0; s < splits; ++s) m_new = fmaxf(m_new, ml[(s * a.row_waves + row_wave) * 32 + l16]);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exponential(m - m_use);
    l = 0.f;
    for (int s = 0; s < splits; ++s) {
      const float* other = ml + (s * a.row_waves + row_wave) * 32 + l16;
      l += other[16] * exponential(other[0] - m_use);
    }
    m = m_new;
#pragma unroll
    for (int db = 0; db < DP / 16; ++db) o[db] *= alpha;
    join_splits(o, reinterpret_cast<float*>(lds_raw), row_wave, a.row_waves, split, splits, lane);
    if (split > 0) return;
  }
  if (qrow >= p.Sq) return;
  store_row<DP>(p.o, b * p.os[0] + hq * p.os[1] + static_cast<int64_t>(qrow) * p.os[2], o, l > 0.f ? 1.0f / l : 0.f, g, a.D, a.vec, 0);
  if (g == 0)
    p.lse[(static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + qrow] = l > 0.f ? m + logf(l) : -INFINITY;
}

// dQ of 64 (32) query rows: dq = scale * sum_j ds_ij k_j, ds = p (dp - delta), p = exp(scale s - lse).  Runs first in a backward
// pass and writes delta = rowsum(dO * O) for the dK/dV kernel.  bp.dq_f32: dq is fp32 and added to (1) or overwritten (2); 0: bf16.
template <int DP, bool DOC>
__global__ __launch_bounds__(kThreads) void attn_tile16_bwd_dq(const AttnBwdParams bp, const Tile16Args a) {
  typedef Tile16<DP> C;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  bf16_t* sK = reinterpret_cast<bf16_t*>(lds_raw);
  bf16_t* sV = sK + kTile * C::LS;
  int2* sIds = reinterpret_cast<int2*>(sV + kTile * C::LS);
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row_wave = wave & (a.row_waves - 1), split = wave / a.row_waves, splits = kWaves / a.row_waves;
  const int unit0 = split, unit_step = splits;
  const int rows = a.row_waves * 16;
  const int nbh = p.B * p.Hq, qt = p.nqt - 1 - static_cast<int>(blockIdx.x) / nbh, bh = static_cast<int>(blockIdx.x) % nbh;
  const int b = bh / p.Hq, hq = bh % p.Hq, hkv = hq / (p.Hq / p.Hkv);
  const int q0 = qt * rows, qrow = q0 + row_wave * 16 + l16, qsafe = min(qrow, p.Sq - 1);
  const bf16_t* Q = static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1] + static_cast<int64_t>(qsafe) * p.qs[2];
  const bf16_t* dO = static_cast<const bf16_t*>(bp.dout) + b * bp.dos[0] + hq * bp.dos[1] + static_cast<int64_t>(qsafe) * bp.dos[2];
  const bf16_t* O = static_cast<const bf16_t*>(p.o) + b * p.os[0] + hq * p.os[1] + static_cast<int64_t>(qsafe) * p.os[2];
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1];

  bf16x8 qf[C::FRAGS], dof[C::FRAGS];
  float delta = 0.f;
#pragma unroll
  for (int j = 0; j < C::FRAGS; ++j) {
    const int d0 = C::STEP * j + kVec * g;
    qf[j] = load_frag(Q, true, d0, a.D, a.vec);
    dof[j] = load_frag(dO, true, d0, a.D, a.vec);
    const bf16x8 of = load_frag(O, true, d0, a.D, a.vec);
#pragma unroll
    for (int e = 0; e < kVec; ++e) delta += static_cast<float>(dof[j][e]) * static_cast<float>(of[e]);
  }
  delta = sum_groups(delta);
  const int64_t stat = (static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + qsafe;
  float lse = p.lse[stat];
  lse = (qrow < p.Sq && lse != -INFINITY) ? lse : INFINITY;  // rows that saw no key: every probability 0
  if (g == 0 && split == 0 && qrow < p.Sq) bp.delta_out[stat] = delta;

  const int klim = qrow < p.Sq ? min(p.Sk - 1, qrow + p.causal_off) : -1;
  int kend = p.Sk, qpos = 0, qseq = -1;
  const int32_t *kpos = nullptr, *kseq = nullptr;
  IdRange blk{};
  if (DOC) {
    kpos = p.k_pos + static_cast<int64_t>(b) * p.Sk;
    kseq = p.k_seq + static_cast<int64_t>(b) * p.Sk;
    const int32_t *qp = p.q_pos + static_cast<int64_t>(b) * p.Sq, *qs = p.q_seq + static_cast<int64_t>(b) * p.Sq;
    if (qrow < p.Sq) qpos = qp[qrow], qseq = qs[qrow];
    blk = id_range(qp, qs, q0, rows, p.Sq, lane);
  } else {
    kend = max(0, min(p.Sk, min(q0 + rows, p.Sq) + p.causal_off));
  }
  const int wave_klim = DOC ? 0 : min(p.Sk - 1, min(q0 + row_wave * 16, p.Sq - 1) + p.causal_off);
  const int wave_kmax = DOC ? p.Sk : min(q0 + row_wave * 16 + 15, p.Sq - 1) + p.causal_off;
  auto next_tile = [&](int k) {
    if (DOC) {
      for (; k < kend; k += kTile) {
        const int kj = k + lane;
        bool some = false;
        if (kj < p.Sk) {
          const int kp = kpos[kj], ks = kseq[kj];
          some = kp <= blk.pos_max && ks >= blk.seq_min && ks <= blk.seq_max && ks >= 0;
        }
        if (__builtin_amdgcn_ballot_w64(some) != 0) break;
      }
    }
    return k;
  };

  f32x4 dq[DP / 16];
#pragma unroll
  for (int db = 0; db < DP / 16; ++db) dq[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  Stage<DP> stK, stV;
  int2 ids = make_int2(0, -2);
  int k0 = next_tile(0);
  auto fetch = [&](int k) {
    stK.fetch(K, p.ks[2], k, p.Sk, a.D, a.vec);
    stV.fetch(V, p.vs[2], k, p.Sk, a.D, a.vec);
    if (DOC && tid < kTile) ids = k + tid < p.Sk ? make_int2(kpos[k + tid], kseq[k + tid]) : make_int2(0, -2);
  };
  if (k0 < kend) fetch(k0);
  while (k0 < kend) {
    __syncthreads();
    stK.store(sK);
    stV.store(sV);
    if (DOC && tid < kTile) sIds[tid] = ids;
    __syncthreads();
    const int kn = next_tile(k0 + kTile);
    if (kn < kend) fetch(kn);
    for (int u = unit0; u < 2; u += unit_step) {
      const int ku = k0 + 32 * u;
      if (ku >= p.Sk || ku > wave_kmax) continue;
      const int frag0 = (32 * u + l16) * C::LS + kVec * g;
      f32x4 s[2], dp[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        s[kb] = dp[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < C::FRAGS; ++j) {
          const int at = frag0 + 16 * kb * C::LS + C::STEP * j;
          s[kb] = C::dot(*reinterpret_cast<const bf16x8*>(sK + at), qf[j], s[kb]);
          dp[kb] = C::dot(*reinterpret_cast<const bf16x8*>(sV + at), dof[j], dp[kb]);
        }
      }
      const bool masked = !DOC && ku + 31 > wave_klim;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float pv = exponential(s[kb][i] * p.scale - lse);
          if (DOC) {
            const int2 id = sIds[32 * u + 16 * kb + 4 * g + i];
            if (!(id.x <= qpos && id.y == qseq && qseq >= 0)) pv = 0.f;
          } else if (masked && ku + 16 * kb + 4 * g + i > klim) {
            pv = 0.f;
          }
          s[kb][i] = pv * (dp[kb][i] - delta);
        }
      C::accumulate(dq, sK + 32 * u * C::LS, s, l16, g);
    }
    k0 = kn;
  }
  if (splits > 1) {
    join_splits(dq, reinterpret_cast<float*>(lds_raw), row_wave, a.row_waves, split, splits, lane);
    if (split > 0) return;
  }
  if (qrow < p.Sq)
    store_row<DP>(bp.dq_acc, b * bp.dqs[0] + hq * bp.dqs[1] + static_cast<int64_t>(qrow) * bp.dqs[2], dq, p.scale, g, a.D, a.vec, bp.dq_f32);
}

// dK, dV of 64 (32) key rows of one KV head, summed over the query heads of its group.
template <int DP, bool DOC>
__global__ __launch_bounds__(kThreads) void attn_tile16_bwd_dkv(const AttnBwdParams bp, const Tile16Args a) {
  typedef Tile16<DP> C;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  bf16_t* sQ = reinterpret_cast<bf16_t*>(lds_raw);
  bf16_t* sdO = sQ + kTile * C::LS;
  float2* sStat = reinterpret_cast<float2*>(sdO + kTile * C::LS);  // (lse, delta) of the tile's queries
  int2* sIds = reinterpret_cast<int2*>(sStat + kTile);
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row_wave = wave & (a.row_waves - 1), split = wave / a.row_waves, splits = kWaves / a.row_waves;
  const int unit0 = split, unit_step = splits;
  const int rows = a.row_waves * 16;
  // first blocks first: with a causal mask they are the long ones
  const int nbh = p.B * p.Hkv, kt = static_cast<int>(blockIdx.x) / nbh, bh = static_cast<int>(blockIdx.x) % nbh;
  const int b = bh / p.Hkv, hkv = bh % p.Hkv, group = p.Hq / p.Hkv;
  const int kb0 = kt * rows, krow = kb0 + row_wave * 16 + l16, ksafe = min(krow, p.Sk - 1);
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1] + static_cast<int64_t>(ksafe) * p.ks[2];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1] + static_cast<int64_t>(ksafe) * p.vs[2];
  bf16x8 kf[C::FRAGS], vf[C::FRAGS];
#pragma unroll
  for (int j = 0; j < C::FRAGS; ++j) {
    const int d0 = C::STEP * j + kVec * g;
    kf[j] = load_frag(K, true, d0, a.D, a.vec);
    vf[j] = load_frag(V, true, d0, a.D, a.vec);
  }
  const int qlim = krow < p.Sk ? krow - p.causal_off : 0x7fffffff;          // first query that sees this lane's key
  const int wave_qall = min(kb0 + row_wave * 16 + 15, p.Sk - 1) - p.causal_off;  // from here on every row of the wavefront is seen
  const int wave_qmin = kb0 + row_wave * 16 - p.causal_off;                  // before it none is
  const bool ragged = kb0 + row_wave * 16 + 16 > p.Sk;
  int kpos = 0, kseq = -2, qstart = 0;
  const int32_t *qpos = nullptr, *qseq = nullptr;
  IdRange blk{};
  if (DOC) {
    const int32_t *kp = p.k_pos + static_cast<int64_t>(b) * p.Sk, *ks = p.k_seq + static_cast<int64_t>(b) * p.Sk;
    qpos = p.q_pos + static_cast<int64_t>(b) * p.Sq;
    qseq = p.q_seq + static_cast<int64_t>(b) * p.Sq;
    if (krow < p.Sk) kpos = kp[krow], kseq = ks[krow];
    blk = id_range(kp, ks, kb0, rows, p.Sk, lane);
  } else {
    qstart = max(0, kb0 - p.causal_off) / kTile * kTile;
  }
  auto next_tile = [&](int q) {
    if (DOC) {
      for (; q < p.Sq; q += kTile) {
        const int qi = q + lane;
        bool some = false;
        if (qi < p.Sq) {
          const int qp = qpos[qi], qs = qseq[qi];
          some = qp >= blk.pos_min && qs >= blk.seq_min && qs <= blk.seq_max && qs >= 0;
        }
        if (__builtin_amdgcn_ballot_w64(some) != 0) break;
      }
    }
    return q;
  };

  f32x4 dk[DP / 16], dv[DP / 16];
#pragma unroll
  for (int db = 0; db < DP / 16; ++db) dk[db] = dv[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  Stage<DP> stQ, stdO;
  float2 stat = make_float2(INFINITY, 0.f);
  int2 ids = make_int2(0, -1);
  auto fetch = [&](int hq, int q) {
    stQ.fetch(static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1], p.qs[2], q, p.Sq, a.D, a.vec);
    stdO.fetch(static_cast<const bf16_t*>(bp.dout) + b * bp.dos[0] + hq * bp.dos[1], bp.dos[2], q, p.Sq, a.D, a.vec);
    if (tid < kTile) {
      stat = make_float2(INFINITY, 0.f);  // probability 0: rows past the end, rows that saw no key
      if (DOC) ids = make_int2(0, -1);
      if (q + tid < p.Sq) {
        const int64_t at = (static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + q + tid;
        const float lse = p.lse[at];
        stat = make_float2(lse == -INFINITY ? INFINITY : lse, bp.delta[at]);
        if (DOC) ids = make_int2(qpos[q + tid], qseq[q + tid]);
      }
    }
  };
  const int qfirst = next_tile(qstart);
  int hg = 0, q0 = qfirst;
  if (q0 < p.Sq) fetch(hkv * group, q0);
  while (hg < group && qfirst < p.Sq) {
    __syncthreads();
    stQ.store(sQ);
    stdO.store(sdO);
    if (tid < kTile) {
      sStat[tid] = stat;
      if (DOC) sIds[tid] = ids;
    }
    __syncthreads();
    int hn = hg, qn = next_tile(q0 + kTile);
    if (qn >= p.Sq) ++hn, qn = qfirst;
    if (hn < group) fetch(hkv * group + hn, qn);
    for (int u = unit0; u < 2; u += unit_step) {
      const int qu = q0 + 32 * u;
      if (qu >= p.Sq || (!DOC && qu + 31 < wave_qmin)) continue;
      const int frag0 = (32 * u + l16) * C::LS + kVec * g;
      f32x4 s[2], dp[2];
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        s[qb] = dp[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < C::FRAGS; ++j) {
          const int at = frag0 + 16 * qb * C::LS + C::STEP * j;
          s[qb] = C::dot(*reinterpret_cast<const bf16x8*>(sQ + at), kf[j], s[qb]);
          dp[qb] = C::dot(*reinterpret_cast<const bf16x8*>(sdO + at), vf[j], dp[qb]);
        }
      }
      const bool masked = !DOC && (qu < wave_qall || ragged);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 32 * u + 16 * qb + 4 * g + i;
          const float2 st = sStat[r];
          float pv = exponential(s[qb][i] * p.scale - st.x);
          if (DOC) {
            const int2 id = sIds[r];
            if (!(kpos <= id.x && kseq == id.y && id.y >= 0)) pv = 0.f;
          } else if (masked && q0 + r < qlim) {
            pv = 0.f;
          }
          s[qb][i] = pv;
          dp[qb][i] = pv * (dp[qb][i] - st.y);
        }
      C::accumulate(dv, sdO + 32 * u * C::LS, s, l16, g);
      C::accumulate(dk, sQ + 32 * u * C::LS, dp, l16, g);
    }
    hg = hn, q0 = qn;
  }
  if (splits > 1) {
    join_splits(dv, reinterpret_cast<float*>(lds_raw), row_wave, a.row_waves, split, splits, lane);
    join_splits(dk, reinterpret_cast<float*>(lds_raw), row_wave, a.row_waves, split, splits, lane);
    if (split > 0) return;
  }
  if (krow >= p.Sk) return;
  store_row<DP>(bp.dk, b * bp.dks[0] + hkv * bp.dks[1] + static_cast<int64_t>(krow) * bp.dks[2], dk, p.scale, g, a.D, a.vec, bp.accumulate_f32);
  store_row<DP>(bp.dv, b * bp.dvs[0] + hkv * bp.dvs[1] + static_cast<int64_t>(krow) * bp.dvs[2], dv, 1.f, g, a.D, a.vec, bp.accumulate_f32);
}

template <int DP>
constexpr int lds_bytes() {
  const int tiles = 2 * kTile * Tile16<DP>::LS * static_cast<int>(sizeof(bf16_t)) + kTile * 16;
  const int join = 3 * (DP / 16) * 64 * 16;
  return tiles > join ? tiles : join;
}

// Wavefronts over the owned rows (each 16 of them); the others of a workgroup's four take the other half of every tile.  64 rows
// per workgroup stage a tile for twice as many products as 32 rows do, but short rows then leave compute units idle and
// the kernel lasts as long as one workgroup's chain of tiles.  The line, from forward + backward at 4 and 2 (us), D=64:
//   S=1024   16 heads (256 workgroups of 64 rows) 118 / 88   32 heads (512) 123 / 95      S=2048, 32 heads (1024) 248 / 267
int row_waves_for(int64_t rows, int64_t heads) {
  const int64_t blocks = (rows + 63) / 64 * heads;
  return blocks >= 768 ? 4 : 2;
}

template <auto KERN, typename P>
int launch(int lds, int64_t blocks, hipStream_t st, const P& params, const Tile16Args& a, const char* what) {
  static MltsLdsOptIn opt_in;
  if (lds > 48 * 1024) {
    if (hipError_t e = opt_in.reserve(reinterpret_cast<const void*>(KERN), lds); e != hipSuccess) {
      mlts_set_error("%s: cannot reserve %d bytes of LDS: %s", what, lds, hipGetErrorString(e));
      return MLTS_ERR_LAUNCH;
    }
  }
  MLTS_REQUIRE(blocks <= 0x7fffffffLL, "%s: too many workgroups", what);
  hipLaunchKernelGGL(KERN, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), lds, st, params, a);
  return mlts_check_launch(what);
}

bool rows_vec(const int64_t* s, const void* ptr) {
  return ((s[0] | s[1] | s[2]) & (kVec - 1)) == 0 && mlts_aligned16(ptr);
}

template <int DP, bool DOC>
int fwd(AttnParams p, int D, hipStream_t st) {
  Tile16Args a{D, row_waves_for(p.Sq, static_cast<int64_t>(p.B) * p.Hq),
               D % kVec == 0 && rows_vec(p.qs, p.q) && rows_vec(p.ks, p.k) && rows_vec(p.vs, p.v) && rows_vec(p.os, p.o)};
  p.nqt = (p.Sq + a.row_waves * 16 - 1) / (a.row_waves * 16);
  MltsKernelTimer timer("attn_fwd", st);
  return launch<attn_tile16_fwd<DP, DOC>>(lds_bytes<DP>(), static_cast<int64_t>(p.nqt) * p.B * p.Hq, st, p, a, "mlts_attn_fwd");
}

template <int DP, bool DOC>
int bwd(AttnBwdParams bp, int D, hipStream_t st) {
  AttnParams& p = bp.a;
  const bool in_vec = D % kVec == 0 && rows_vec(p.qs, p.q) && rows_vec(p.ks, p.k) && rows_vec(p.vs, p.v) &&
                      rows_vec(bp.dos, bp.dout) && rows_vec(p.os, p.o);
  if (p.Sq > 0) {
    Tile16Args a{D, row_waves_for(p.Sq, static_cast<int64_t>(p.B) * p.Hq), in_vec && (bp.dq_f32 || rows_vec(bp.dqs, bp.dq_acc))};
    p.nqt = (p.Sq + a.row_waves * 16 - 1) / (a.row_waves * 16);
    MltsKernelTimer timer("attn_bwd_dq", st);
    if (int rc = launch<attn_tile16_bwd_dq<DP, DOC>>(lds_bytes<DP>(), static_cast<int64_t>(p.nqt) * p.B * p.Hq, st, bp, a, "mlts_attn_bwd"); rc != MLTS_OK)
      return rc;
  }
  if (p.Sk == 0) return MLTS_OK;
  Tile16Args a{D, row_waves_for(p.Sk, static_cast<int64_t>(p.B) * p.Hkv),
               in_vec && (bp.accumulate_f32 || (rows_vec(bp.dks, bp.dk) && rows_vec(bp.dvs, bp.dv)))};
  const int64_t nkt = (p.Sk + a.row_waves * 16 - 1) / (a.row_waves * 16);
  MltsKernelTimer timer("attn_bwd_dkdv", st);
  return launch<attn_tile16_bwd_dkv<DP, DOC>>(lds_bytes<DP>(), nkt * p.B * p.Hkv, st, bp, a, "mlts_attn_bwd");
}

// p.causal_off: the last key query i sees is i + causal_off; without a causal mask it is past every key
void set_causal_off(AttnParams& p, int mode) {
  if (mode != MLTS_MASK_CAUSAL) p.causal_off = p.Sk > p.Sq ? p.Sk : p.Sq;
}

#define MLTS_TILE16_DP(FN, DOC, ...)                \
  do {                                              \
    if (D <= 32) return FN<32, DOC>(__VA_ARGS__);   \
    if (D <= 64) return FN<64, DOC>(__VA_ARGS__);   \
    if (D <= 96) return FN<96, DOC>(__VA_ARGS__);   \
    if (D <= 128) return FN<128, DOC>(__VA_ARGS__); \
    if (D <= 160) return FN<160, DOC>(__VA_ARGS__); \
    return FN<192, DOC>(__VA_ARGS__);               \
  } while (0)
#define MLTS_TILE16(FN, ...)                                          \
  do {                                                                \
    if (mode == MLTS_MASK_DOC) MLTS_TILE16_DP(FN, true, __VA_ARGS__); \
    MLTS_TILE16_DP(FN, false, __VA_ARGS__);                           \
  } while (0)

}  // namespace

int mlts_attn_tile16_fwd(AttnParams p, int D, int mode, hipStream_t st) {
  set_causal_off(p, mode);
  MLTS_TILE16(fwd, p, D, st);
}

// bp.delta_out receives rowsum(dO * O); bp.delta must point at the same buffer
int mlts_attn_tile16_bwd(AttnBwdParams bp, int D, int mode, hipStream_t st) {
  set_causal_off(bp.a, mode);
  MLTS_TILE16(bwd, bp, D, st);
}
