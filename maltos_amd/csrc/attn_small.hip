// bf16 attention at head_dim 64 and 128 on grids that leave most of the chip to few workgroups of the 32-row kernels (attn_fwd_dma.hip,
// attn_bwd_dq_tr.hip, attn_bwd_split.hip), and at head_dim 32 and 96 without documents (mlts_attn_small_serves_parts()).
//
// Those give a workgroup 128 or 256 rows and walk the other side 64 rows at a time, one tile behind the other at about a microsecond each:
// with few rows and heads the kernel lasts as long as one workgroup's chain.  Here a wavefront owns R blocks of 16 rows (queries in the forward
// and dQ kernels, keys in the dK/dV kernel) and takes every `splits`-th unit of 32 rows of the other side, so that there are up to 64 times as
// many wavefronts, with chains of a few units.  Two blocks share what a wavefront fetches, puts to LDS and reads from there: on grids that fill the
// chip that is most of a unit's time besides the softmax arithmetic (two_blocks()).  A unit arrives in whole lines, one unit ahead, and goes through LDS of its own wavefront to
// the fragments of v_mfma_f32_16x16x32_bf16 (rows: 16-byte reads; contraction over the rows: transposing reads), without a barrier before
// the splits' sums meet at the end.  Scores are computed transposed, as in the fp32 kernels, so that a lane holds the probabilities of one
// own row and the next product takes them, rounded to bf16 once, from the registers they are in.
//
// Documents: the plan's tile classes and visibility bits, as in the 32-row kernels.
#include "attn_bf16.hpp"

namespace {

constexpr int kUnit = 32;      // walked rows
constexpr int kMaxSplits = 8;  // wavefronts to a row block

__device__ __forceinline__ const bf16_t* row_of(const bf16_t* base, int row, int64_t stride) {  // (near(): offsets fit 32 bits)
  const uint32_t offset = __umul24(static_cast<uint32_t>(row), static_cast<uint32_t>(stride) * 2u);
  return reinterpret_cast<const bf16_t*>(reinterpret_cast<const char*>(base) + offset);
}

// A unit of one operand: fetched, put to LDS, read as fragments.  A wavefront's 64 chunks of 16 bytes are whole rows, or those of three fetches are.
template <int D>
struct Unit : Rows<D> {
  static constexpr int CHUNKS = D / 8, N = kUnit * CHUNKS / 64, BYTES = kUnit * Rows<D>::BYTES;
  static constexpr int PERIOD = 64 % CHUNKS == 0 ? 1 : 3, ROWS = 64 * PERIOD / CHUNKS;  // of that many fetches
  static_assert(64 * PERIOD % CHUNKS == 0 && N % PERIOD == 0, "whole rows");
  bf16x8 raw[N];
  uint32_t stride, offset[PERIOD];  // bytes: between rows, of this lane's chunks in the first rows
  __device__ __forceinline__ void init(int64_t elements, int lane) {
    stride = static_cast<uint32_t>(elements) * 2u;
#pragma unroll
    for (int i = 0; i < PERIOD; ++i) offset[i] = static_cast<uint32_t>((64 * i + lane) / CHUNKS) * stride + 16u * static_cast<uint32_t>((64 * i + lane) % CHUNKS);
  }
  // rows row0 ..; rows past the last one are zeros, from the bounds check of the descriptor (near(): no offset wraps).  One addition a chunk:
  // the row's part of the address is the same in all lanes.
  __device__ __forceinline__ void fetch(const bf16_t* base, int row0, int last) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), 0, static_cast<uint32_t>(last) * stride + 2u * D, 0x00020000);
    const uint32_t at = static_cast<uint32_t>(min(row0, last)) * stride;
#pragma unroll
    for (int i = 0; i < N; ++i)
      raw[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset[i % PERIOD] + (at + static_cast<uint32_t>(i / PERIOD * ROWS) * stride), 0, 0));
  }
  __device__ __forceinline__ void put(unsigned char* lds, int lane) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int chunk = 64 * (i % PERIOD) + lane;
      *reinterpret_cast<bf16x8*>(lds + Rows<D>::at(i / PERIOD * ROWS + chunk / CHUNKS, chunk % CHUNKS)) = raw[i];
    }
  }
};

// What a probability or dS goes into its second product as: at head_dim 64 and 128 rounded to bf16, as in the 32-row kernels; else the sum of three bf16
// values of 8 bits each, which is all of an fp32 number, as in attn_tile16.hip.
template <int D>
constexpr int kParts = D == 64 || D == 128 ? 1 : 3;
template <int PARTS>
__device__ __forceinline__ void split(bf16x8 (&part)[PARTS], const f32x4 (&x)[2]) {
  if constexpr (PARTS == 1) {
    part[0] = pack(x);
  } else {
    f32x4 rest[2] = {x[0], x[1]};
#pragma unroll
    for (int n = 0; n < PARTS; ++n) {
      part[n] = pack(rest);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) rest[b][i] -= static_cast<float>(part[n][4 * b + i]);
    }
  }
}
// acc[r][db] += columns x own rows; column(db): of the walked rows
template <int R, int NC, int PARTS, typename F>
__device__ __forceinline__ void add_products(f32x4 (&acc)[R][NC], const bf16x8 (&x)[R][PARTS], F column) {
  if constexpr (PARTS == 1) {
#pragma unroll
    for (int db = 0; db < NC; ++db) {
      const bf16x8 c = column(db);
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r][db] = mfma32(c, x[r][0], acc[r][db]);
    }
  } else {
    bf16x8 c[NC];
#pragma unroll
    for (int db = 0; db < NC; ++db) c[db] = column(db);
#pragma unroll
    for (int n = 0; n < PARTS; ++n)
#pragma unroll
      for (int db = 0; db < NC; ++db)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][db] = mfma32(c[db], x[r][n], acc[r][db]);
  }
}

// The units a split works on, in order: every `splits`-th.  Documents: those of them whose tile of 64 rows the plan's statistics do not
// rule out for the own rows' group of 64, 32 tiles at a time, a lane for each unit.
template <bool DOC, bool KEYS>
struct Walk {
  int split, splits, end, lane;   // end: rows walked
  const int4* stats;              // DOC: of the walked side's tiles
  int4 own;
  int base;                       // first row of the current look
  unsigned long long left, full;  // of the current look: units that are left, units that every own row sees
  bool masked;                    // of the unit that was returned last: what is seen is in the plan's bits

  __device__ __forceinline__ void look() {
    const int row = base + kUnit * lane;
    int c = TILE_SKIP;
    if (row < end) {
      const int4 tile = stats[row >> 6];
      c = KEYS ? classify_doc_tile(own, tile) : classify_doc_tile(tile, own);
    }
    const unsigned long long every = splits == 8 ? 0x0101010101010101ull : splits == 4 ? 0x1111111111111111ull : splits == 2 ? 0x5555555555555555ull : ~0ull;
    left = __builtin_amdgcn_ballot_w64(c != TILE_SKIP) & (every << split);
    full = __builtin_amdgcn_ballot_w64(c == TILE_FULL);
  }
  __device__ __forceinline__ int first(int start) {
    if (!DOC) return start + kUnit * split;
    base = -64 * kUnit, left = 0;
    return next(0);
  }
  __device__ __forceinline__ int next(int row) {
    if (!DOC) return row + kUnit * splits;
    while (left == 0) {
      base += 64 * kUnit;
      if (base >= end) return end;
      look();
    }
    const int bit = __builtin_ctzll(left);
    left &= left - 1;
    masked = ((full >> bit) & 1) == 0;
    return base + kUnit * bit;
  }
};

// The splits' sums of N results of 16 rows, and what becomes of them: acc[n][db] are columns 16 db + 4 g ..+3 of this lane's row.  finish: what a sum
// becomes before it is stored, which may load (ahead of the first store)
template <int NC, int N, typename F, typename G>
__device__ __forceinline__ void join_and_store(f32x4 (&acc)[N][NC], f32x4* lds, const Place& at, G finish, F store) {
  if (at.splits == 1) {
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int db = 0; db < NC; ++db) acc[n][db] = finish(n, db, acc[n][db]);
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int db = 0; db < NC; ++db) store(n, db, acc[n][db]);
    return;
  }
  lds += at.slot * at.splits * N * NC * 64 + at.lane;
  __syncthreads();  // nobody needs what the LDS holds any more
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int db = 0; db < NC; ++db) lds[((at.split * N + n) * NC + db) * 64] = acc[n][db];
  __syncthreads();
#pragma unroll
  for (int n = 0; n < N; ++n)
    for (int db = (at.split - n * NC) & (at.splits - 1); db < NC; db += at.splits) {
      f32x4 v = lds[(n * NC + db) * 64];
      for (int s = 1; s < at.splits; ++s) v += lds[((s * N + n) * NC + db) * 64];
      store(n, db, finish(n, db, v));
    }
}

// O and LSE of R * 16 query rows
template <int D, bool DOC, int R>
__global__ __launch_bounds__(kMaxSplits * 64) void attn_small_fwd(const AttnParams p, const RowArgs a) {
  typedef Unit<D> U;
  static_assert(!DOC || R == 1, "documents: one block of 16 rows to a wavefront");
  constexpr int FRAGS = D / 32, NC = D / 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g;
  // with a causal mask the last blocks are the long ones
  int bh, hq, member;
  const int qt = p.nqt - 1 - a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hq), hkv = a.group.over(hq, &member);
  const int q0 = 16 * R * qt;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1];
  bf16x8 qf[R][FRAGS];
  int klim[R];  // keys this lane's queries see: up to klim (causal_off is Sk without a causal mask); documents also by the plan's bits
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int qrow = q0 + 16 * r + l16;
    const bf16_t* q_row = row_of(static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1], min(qrow, p.Sq - 1), p.qs[2]);
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) qf[r][j] = *reinterpret_cast<const bf16x8*>(q_row + 32 * j + 8 * g);
    klim[r] = DOC || qrow < p.Sq ? min(p.Sk - 1, DOC ? p.Sk : qrow + p.causal_off) : -1;
  }
  Walk<DOC, true> walk;
  walk.split = at.split, walk.splits = at.splits, walk.lane = lane;
  const unsigned long long* bits = nullptr;
  if (DOC) {
    const int group = q0 >> 6;
    walk.stats = p.k_stats + b * p.nk_stats;
    walk.own = p.q_stats[b * p.nq_stats + group];
    bits = p.doc_bits + (static_cast<int64_t>(b) * p.nq_stats + group) * p.nk_stats * 64 + ((q0 + l16) & 63);
    walk.end = p.Sk;
  } else {
    walk.end = max(0, min(p.Sk, min(q0 + 16 * R, p.Sq) + p.causal_off));
  }
  const int kend = at.there ? walk.end : 0;
  const int all_klim = DOC ? p.Sk - 1 : min(p.Sk - 1, min(q0, p.Sq - 1) + p.causal_off);  // seen by every row (that exists)

  float m[R], l[R];
  f32x4 o[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    m[r] = -INFINITY, l[r] = 0.f;
#pragma unroll
    for (int db = 0; db < NC; ++db) o[r][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  U keys, values;
  keys.init(p.ks[2], lane), values.init(p.vs[2], lane);
  unsigned char *lk = lds_raw + at.wave * 2 * U::BYTES, *lv = lk + U::BYTES;
  // (past the end some key is fetched again: a branch around the loads would wait for all of them)
  unsigned long long word = 0, word_now = 0;
  bool masked = false, masked_now = false;
  auto fetch_keys = [&](int k) {
    keys.fetch(K, k, p.Sk - 1);
    if (DOC) word = bits[static_cast<int64_t>(min(k, p.Sk - 1) >> 6) * 64], masked = walk.masked;
  };
  int k0 = walk.first(0), kn = k0;
  if (k0 < kend) {
    fetch_keys(k0);
    values.fetch(V, k0, p.Sk - 1);
    keys.put(lk, lane), values.put(lv, lane);
    word_now = word, masked_now = masked;
    kn = walk.next(k0);
    fetch_keys(kn);
    values.fetch(V, kn, p.Sk - 1);
  }
  while (k0 < kend) {
    f32x4 s[R][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < R; ++r) s[r][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) {
        const bf16x8 key = U::dot(lk, u, j, l16, g);
#pragma unroll
        for (int r = 0; r < R; ++r) s[r][u] = mfma32(key, qf[r][j], s[r][u]);
      }
    }
    if (k0 + kUnit - 1 > all_klim) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (k0 + 16 * u + 4 * g + i > klim[r]) s[r][u][i] = -INFINITY;
    }
    if (DOC && masked_now) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t w = static_cast<uint32_t>(word_now >> (k0 & 32));
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!((w >> (16 * u + 4 * g + i)) & 1)) s[r][u][i] = -INFINITY;
      }
    }
    const int kn2 = kn < kend ? walk.next(kn) : kn;
    const unsigned long long word_next = word;
    const bool masked_next = masked;
    keys.put(lk, lane);  // the next unit's, which have had one unit's time to arrive
    fetch_keys(kn2);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 pr[R][kParts<D>];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float mx = -INFINITY;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[r][u][i]);
      mx = max_groups(mx) * p.scale;
      if (__builtin_amdgcn_ballot_w64(mx > m[r]) != 0) {
        const float m_new = fmaxf(m[r], mx);
        const float alpha = exponential(m[r] - (m_new == -INFINITY ? 0.f : m_new));  // 1 for rows that do not rise, 0 from -inf
        m[r] = m_new;
        l[r] *= alpha;
#pragma unroll
        for (int db = 0; db < NC; ++db) o[r][db] *= alpha;
      }
      const float m_use = m[r] == -INFINITY ? 0.f : m[r];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[r][u][i] = exponential(s[r][u][i] * p.scale - m_use);
          l[r] += s[r][u][i];
        }
      split(pr[r], s[r]);
    }
    add_products(o, pr, [&](int db) { return U::columns(lv, db, l16, g); });
    values.put(lv, lane);
    values.fetch(V, kn2, p.Sk - 1);
    k0 = kn, kn = kn2, word_now = word_next, masked_now = masked_next;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) l[r] = sum_groups(l[r]);
  if (at.splits > 1) {  // every split holds some of the keys: all to the largest maximum
    __syncthreads();    // the units' LDS is free
    float* ml = reinterpret_cast<float*>(lds_raw) + at.slot * at.splits * 32 * R;
    if (g == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) ml[(at.split * R + r) * 32 + l16] = m[r], ml[(at.split * R + r) * 32 + 16 + l16] = l[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float* of = ml + r * 32 + l16;
      float m_new = -INFINITY;
      for (int s = 0; s < at.splits; ++s) m_new = fmaxf(m_new, of[s * R * 32]);
      const float m_use = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = exponential(m[r] - m_use);
      l[r] = 0.f;
      for (int s = 0; s < at.splits; ++s) l[r] += of[s * R * 32 + 16] * exponential(of[s * R * 32] - m_use);
      m[r] = m_new;
#pragma unroll
      for (int db = 0; db < NC; ++db) o[r][db] *= alpha;
    }
  }
  const int64_t row = b * p.os[0] + hq * p.os[1] + 4 * g;
  float scale[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int qrow = q0 + 16 * r + l16;
    if (at.there && qrow < p.Sq && g == 0 && at.split == 0)
      p.lse[(static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + qrow] = l[r] > 0.f ? m[r] + logf(l[r]) : -INFINITY;
    scale[r] = l[r] > 0.f ? 1.0f / l[r] : 0.f;
  }
  join_and_store(o, reinterpret_cast<f32x4*>(lds_raw), at, [&](int r, int, f32x4 v) { return v * scale[r]; }, [&](int r, int db, f32x4 v) {
    const int qrow = q0 + 16 * r + l16;
    if (at.there && qrow < p.Sq) store4(p.o, row + qrow * p.os[2] + 16 * db, v, 0);
  });
}

// dQ of R * 16 query rows: dq = scale * sum_j ds_ij k_j, ds = p (dp - delta), p = exp(scale s - lse).  Runs first in a backward pass and writes
// delta = rowsum(dO * O) for the dK/dV kernel.  bp.dq_f32: dq is fp32 and added to (1) or overwritten (2); 0: bf16.
template <int D, bool DOC, int R>
__global__ __launch_bounds__(kMaxSplits * 64) void attn_small_bwd_dq(const AttnBwdParams bp, const RowArgs a) {
  typedef Unit<D> U;
  static_assert(!DOC || R == 1, "documents: one block of 16 rows to a wavefront");
  constexpr int FRAGS = D / 32, NC = D / 16;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g;
  // with a causal mask the last blocks are the long ones
  int bh, hq, member;
  const int qt = p.nqt - 1 - a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hq), hkv = a.group.over(hq, &member);
  const int q0 = 16 * R * qt;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1];
  bf16x8 qf[R][FRAGS], dof[R][FRAGS];
  float delta[R], lse[R];
  int klim[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int qrow = q0 + 16 * r + l16, safe = min(qrow, p.Sq - 1);
    const bf16_t* q_row = row_of(static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1], safe, p.qs[2]);
    const bf16_t* do_row = row_of(static_cast<const bf16_t*>(bp.dout) + b * bp.dos[0] + hq * bp.dos[1], safe, bp.dos[2]);
    const bf16_t* o_row = row_of(static_cast<const bf16_t*>(p.o) + b * p.os[0] + hq * p.os[1], safe, p.os[2]);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      qf[r][j] = *reinterpret_cast<const bf16x8*>(q_row + 32 * j + 8 * g);
      dof[r][j] = *reinterpret_cast<const bf16x8*>(do_row + 32 * j + 8 * g);
      const bf16x8 of = *reinterpret_cast<const bf16x8*>(o_row + 32 * j + 8 * g);
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += static_cast<float>(dof[r][j][e]) * static_cast<float>(of[e]);
    }
    delta[r] = sum_groups(sum);
    const int64_t stat = (static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + safe;
    lse[r] = p.lse[stat];
    lse[r] = qrow < p.Sq && lse[r] != -INFINITY ? lse[r] : INFINITY;  // rows that saw no key: every probability 0
    if (at.there && qrow < p.Sq && g == 0 && at.split == 0) {  // the statistics of the backward pass, for whichever dK/dV kernel comes next
      bp.delta_out[stat] = delta[r];
      if (kParts<D> == 1) bp.lse2_out[stat] = lse[r] * 1.44269504088896340736f;
    }
    klim[r] = DOC || qrow < p.Sq ? min(p.Sk - 1, DOC ? p.Sk : qrow + p.causal_off) : -1;
  }
  if (kParts<D> == 1 && blockIdx.x == 0 && threadIdx.x == 0) bp.lse2_out[static_cast<int64_t>(p.B) * p.Hq * p.Sq] = INFINITY;
  Walk<DOC, true> walk;
  walk.split = at.split, walk.splits = at.splits, walk.lane = lane;
  const unsigned long long* bits = nullptr;
  if (DOC) {
    const int group = q0 >> 6;
    walk.stats = p.k_stats + b * p.nk_stats;
    walk.own = p.q_stats[b * p.nq_stats + group];
    bits = p.doc_bits + (static_cast<int64_t>(b) * p.nq_stats + group) * p.nk_stats * 64 + ((q0 + l16) & 63);
    walk.end = p.Sk;
  } else {
    walk.end = max(0, min(p.Sk, min(q0 + 16 * R, p.Sq) + p.causal_off));
  }
  const int kend = at.there ? walk.end : 0;
  const int all_klim = DOC ? p.Sk - 1 : min(p.Sk - 1, min(q0, p.Sq - 1) + p.causal_off);

  f32x4 dq[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int db = 0; db < NC; ++db) dq[r][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  U keys, values;
  keys.init(p.ks[2], lane), values.init(p.vs[2], lane);
  unsigned char *lk = lds_raw + at.wave * 2 * U::BYTES, *lv = lk + U::BYTES;
  unsigned long long word = 0, word_now = 0;
  bool masked = false, masked_now = false;
  auto fetch = [&](int k) {  // (past the end the last key again: a branch around the loads would wait for all of them)
    keys.fetch(K, k, p.Sk - 1);
    values.fetch(V, k, p.Sk - 1);
    if (DOC) word = bits[static_cast<int64_t>(min(k, p.Sk - 1) >> 6) * 64], masked = walk.masked;
  };
  auto put = [&] {
    keys.put(lk, lane), values.put(lv, lane);
    word_now = word, masked_now = masked;
  };
  int k0 = walk.first(0), kn = k0;
  if (k0 < kend) {
    fetch(k0);
    put();
    kn = walk.next(k0);
    fetch(kn);
  }
  while (k0 < kend) {
    f32x4 s[R][2], dp[R][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < R; ++r) s[r][u] = dp[r][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) {
        const bf16x8 key = U::dot(lk, u, j, l16, g), value = U::dot(lv, u, j, l16, g);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          s[r][u] = mfma32(key, qf[r][j], s[r][u]);
          dp[r][u] = mfma32(value, dof[r][j], dp[r][u]);
        }
      }
    }
    const bool edge = k0 + kUnit - 1 > all_klim;
    bf16x8 ds[R][kParts<D>];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[r][u][i] = exponential(s[r][u][i] * p.scale - lse[r]);
      if (edge) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (k0 + 16 * u + 4 * g + i > klim[r]) s[r][u][i] = 0.f;
      }
      if (DOC && masked_now) {
        const uint32_t w = static_cast<uint32_t>(word_now >> (k0 & 32));
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!((w >> (16 * u + 4 * g + i)) & 1)) s[r][u][i] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[r][u][i] *= dp[r][u][i] - delta[r];
      split(ds[r], s[r]);
    }
    bf16x8 kc[NC];
#pragma unroll
    for (int db = 0; db < NC; ++db) kc[db] = U::columns(lk, db, l16, g);
    const int kn2 = kn < kend ? walk.next(kn) : kn;
    put();  // the next unit's, which have had one unit's time to arrive
    fetch(kn2);
    __builtin_amdgcn_sched_barrier(0);
    add_products(dq, ds, [&](int db) { return kc[db]; });
    k0 = kn, kn = kn2;
  }
  const int64_t row = b * bp.dqs[0] + hq * bp.dqs[1] + 4 * g;
  const RotateBack rot = rotation_of_kernel<decltype(attn_small_bwd_dq<D, DOC, R>)>();
  int64_t table[R];
  if (rot.cos) {
#pragma unroll
    for (int r = 0; r < R; ++r) table[r] = rot.row(b, q0 + 16 * r + l16);
  }
  const auto finish = [&](int r, int db, f32x4 v) {
    return rot.cos ? RotateBack::back<bf16_t>(v * p.scale, rot.angles<bf16_t, 2>(table[r], 8 * db + 2 * g)) : v * p.scale;
  };
  join_and_store(dq, reinterpret_cast<f32x4*>(lds_raw), at, finish, [&](int r, int db, f32x4 v) {
    const int qrow = q0 + 16 * r + l16;
    if (at.there && qrow < p.Sq) store4(bp.dq_acc, row + qrow * bp.dqs[2] + 16 * db, v, bp.dq_f32);
  });
}

// dK, dV of R * 16 key rows of one KV head, summed over the query heads of its group.
template <int D, bool DOC, int R>
__global__ __launch_bounds__(kMaxSplits * 64) void attn_small_bwd_dkv(const AttnBwdParams bp, const RowArgs a) {
  typedef Unit<D> U;
  static_assert(!DOC || R == 1, "documents: one block of 16 rows to a wavefront");
  constexpr int FRAGS = D / 32, NC = D / 16;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g;
  // with a causal mask the first blocks are the long ones
  int bh, hkv;
  const int kt = a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hkv), group = static_cast<int>(a.group.d);
  const int kb0 = kt * 16 * R;
  bf16x8 kf[R][FRAGS], vf[R][FRAGS];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int ksafe = min(kb0 + 16 * r + l16, p.Sk - 1);
    const bf16_t* k_row = row_of(static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1], ksafe, p.ks[2]);
    const bf16_t* v_row = row_of(static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1], ksafe, p.vs[2]);
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      kf[r][j] = *reinterpret_cast<const bf16x8*>(k_row + 32 * j + 8 * g);
      vf[r][j] = *reinterpret_cast<const bf16x8*>(v_row + 32 * j + 8 * g);
    }
  }
  const int qlim = DOC ? 0 : kb0 + l16 - p.causal_off;                              // first query that sees this lane's first key
  const int all_qmin = DOC ? 0 : min(kb0 + 16 * R - 1, p.Sk - 1) - p.causal_off;    // from here on every key that exists is seen
  Walk<DOC, false> walk;
  walk.split = at.split, walk.splits = at.splits, walk.lane = lane, walk.end = p.Sq;
  const unsigned long long* bits = nullptr;
  int qstart = 0;
  if (DOC) {
    const int tile = kb0 >> 6;
    walk.stats = p.q_stats + b * p.nq_stats;
    walk.own = p.k_stats[b * p.nk_stats + tile];
    bits = p.doc_bits_k + (static_cast<int64_t>(b) * p.nk_stats + tile) * p.nq_stats * 64 + ((kb0 + l16) & 63);
  } else {
    qstart = max(0, kb0 - p.causal_off) / kUnit * kUnit;
  }

  f32x4 dk[R][NC], dv[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int db = 0; db < NC; ++db) dk[r][db] = dv[r][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  U queries, grads;
  queries.init(p.qs[2], lane), grads.init(bp.dos[2], lane);
  unsigned char* own = lds_raw + at.wave * (2 * U::BYTES + 256);
  unsigned char *lq = own, *ld = own + U::BYTES;
  float* lstat = reinterpret_cast<float*>(own + 2 * U::BYTES);  // (lse, delta) of the unit's queries: a lane fetches one, and reads eight of each
  float stat = 0.f;
  unsigned long long word = 0, word_now = 0;
  bool masked = false, masked_now = false;
  const bf16_t* Q0 = static_cast<const bf16_t*>(p.q) + b * p.qs[0];
  const bf16_t* dO0 = static_cast<const bf16_t*>(bp.dout) + b * bp.dos[0];
  int row_fetched = 0;
  auto fetch = [&](int hg, int q) {  // (past the end the last query again: a branch around the loads would wait for all of them)
    const int head = hkv * group + hg;
    queries.fetch(Q0 + head * p.qs[1], q, p.Sq - 1);
    grads.fetch(dO0 + head * bp.dos[1], q, p.Sq - 1);
    row_fetched = q + (lane & 31);
    stat = (lane < 32 ? p.lse : bp.delta)[(static_cast<int64_t>(b) * p.Hq + head) * p.Sq + min(row_fetched, p.Sq - 1)];
    if (DOC) word = bits[static_cast<int64_t>(min(q, p.Sq - 1) >> 6) * 64], masked = walk.masked;
  };
  auto put = [&] {
    queries.put(lq, lane), grads.put(ld, lane);
    // probability 0: rows past the end, rows that saw no key
    lstat[lane] = lane < 32 && (row_fetched >= p.Sq || stat == -INFINITY) ? INFINITY : stat;
    word_now = word, masked_now = masked;
  };
  // the units of all heads of the group, one after the other
  int hg = at.there ? 0 : group, q0 = walk.first(qstart);
  auto skip = [&](int& h, int& q) {
    while (q >= p.Sq && ++h < group) q = walk.first(qstart);
  };
  skip(hg, q0);
  int hn = hg, qn = q0;
  if (hg < group) {
    fetch(hg, q0);
    put();
    qn = walk.next(q0);
    skip(hn, qn);
    fetch(min(hn, group - 1), qn);
  }
  while (hg < group) {
    f32x4 s[R][2], dp[R][2], lse[2], delta[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < R; ++r) s[r][u] = dp[r][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) {
        const bf16x8 query = U::dot(lq, u, j, l16, g), grad = U::dot(ld, u, j, l16, g);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          s[r][u] = mfma32(query, kf[r][j], s[r][u]);
          dp[r][u] = mfma32(grad, vf[r][j], dp[r][u]);
        }
      }
      lse[u] = *reinterpret_cast<const f32x4*>(lstat + 16 * u + 4 * g);
      delta[u] = *reinterpret_cast<const f32x4*>(lstat + 32 + 16 * u + 4 * g);
    }
    const bool edge = !DOC && q0 < all_qmin;
    bf16x8 pr[R][kParts<D>], ds[R][kParts<D>];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[r][u][i] = exponential(s[r][u][i] * p.scale - lse[u][i]);
      if (edge) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (q0 + 16 * u + 4 * g + i < qlim + 16 * r) s[r][u][i] = 0.f;
      }
      if (DOC && masked_now) {
        const uint32_t w = static_cast<uint32_t>(word_now >> (q0 & 32));
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!((w >> (16 * u + 4 * g + i)) & 1)) s[r][u][i] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) dp[r][u][i] = s[r][u][i] * (dp[r][u][i] - delta[u][i]);
      split(pr[r], s[r]), split(ds[r], dp[r]);
    }
    add_products(dv, pr, [&](int db) { return U::columns(ld, db, l16, g); });
    bf16x8 col[NC];
#pragma unroll
    for (int db = 0; db < NC; ++db) col[db] = U::columns(lq, db, l16, g);
    int hn2 = hn, qn2 = qn;
    if (hn < group) qn2 = walk.next(qn), skip(hn2, qn2);
    put();  // the next unit's, which have had one unit's time to arrive
    fetch(min(hn2, group - 1), qn2);
    __builtin_amdgcn_sched_barrier(0);
    add_products(dk, ds, [&](int db) { return col[db]; });
    hg = hn, q0 = qn, hn = hn2, qn = qn2;
  }
  const int64_t dk_row = b * bp.dks[0] + hkv * bp.dks[1] + 4 * g, dv_row = b * bp.dvs[0] + hkv * bp.dvs[1] + 4 * g;
  f32x4 dkv[2 * R][NC];
#pragma unroll
  for (int n = 0; n < 2 * R; ++n)
#pragma unroll
    for (int db = 0; db < NC; ++db) dkv[n][db] = n < R ? dk[n < R ? n : 0][db] : dv[n < R ? 0 : n - R][db];
  const RotateBack rot = rotation_of_kernel<decltype(attn_small_bwd_dkv<D, DOC, R>)>();
  int64_t table[R];
  if (rot.cos) {
#pragma unroll
    for (int r = 0; r < R; ++r) table[r] = rot.row(b, kb0 + 16 * r + l16);
  }
  const auto finish = [&](int n, int db, f32x4 v) {
    if (n >= R) return v;
    return rot.cos ? RotateBack::back<bf16_t>(v * p.scale, rot.angles<bf16_t, 2>(table[n < R ? n : 0], 8 * db + 2 * g)) : v * p.scale;
  };
  join_and_store(dkv, reinterpret_cast<f32x4*>(lds_raw), at, finish, [&](int n, int db, f32x4 v) {
    const int krow = kb0 + 16 * (n < R ? n : n - R) + l16;
    if (at.there && krow < p.Sk)
      store4(n < R ? bp.dk : bp.dv, (n < R ? dk_row + krow * bp.dks[2] : dv_row + krow * bp.dvs[2]) + 16 * db, v, bp.accumulate_f32);
  });
}

bool near(int64_t rows, const int64_t* stride) {  // offsets that row_of can form
  return rows < (1 << 24) && stride[2] < (1 << 23) && ((rows - 1 + kUnit) * stride[2] + 128) * 2 < (int64_t{1} << 32);
}

// Splits of two blocks.  What counts is how many wavefronts are there at once: a second round of them takes as long as the first.  Four splits are one wavefront
// a SIMD to a workgroup, of which two (dK/dV, all of head_dim 128), three (dQ at head_dim 64: 3072 wavefronts) or four (forward at head_dim 64) fit; somewhat more than fit are
// still ahead of two splits of twice the length, and long walks at any number.  Eight splits are ahead only if all fit, two workgroups to a CU where registers do not allow more.
// us, two / four splits (blocks: of 32 rows; units: of 32 rows walked)
//   head_dim 64, causal   forward 1200 blocks, 75 units 39.1 / 33.2    1254, 57 31.5 / 30.2    dQ 768, 32 19.8 / 18.7    832, 64 28.4 / 26.1    832, 32 19.5 / 21.8    900, 50 24.2 / 27.1
//                         dQ 980, 70 30.1 / 32.6    1200, 75 38.9 / 37.2    1450, 145 71.0 / 64.0    dK/dV 828, 69 40.2 / 35.0    864, 32 24.6 / 26.0    1040, 104 68.8 / 51.2    1254, 57 47.9 / 40.1
//   head_dim 128, causal  forward 640, 64 46.7 / 35.7    798, 57 42.1 / 40.6    900, 50 38.5 / 40.2    1008, 48 37.8 / 53.4    dQ 644, 46 40.2 / 35.3    672, 28 30.1 / 31.8    860, 43 37.1 / 41.1
//                         dQ 896, 128 82.6 / 78.9    1024, 256 148 / 142    900, 50 41.2 / 45.0    1008, 48 41.0 / 54.2    1328, 83 67.4 / 74.7    unmasked, 740, 47 53.1 / 49.0
// four / eight
//   head_dim 64           forward 384, 64 25.3 / 24.4    522, 58 20.4 / 20.3    dQ 260, 45 19.5 / 24.3    470, 72 21.7 / 26.0    dK/dV 285, 220 75.9 / 81.5    384, 64 30.3 / 33.5
//   head_dim 128          forward 246, 41 22.2 / 20.4    320, 64 37.5 / 45.5    474, 79 44.9 / 51.3    dQ 246, 41 22.5 / 23.0    320, 64 40.8 / 50.8    490, 35 30.1 / 38.8
//   head_dim 32           forward 322, 46 21.9 / 21.4    dQ 273, 91 31.5 / 29.6    dK/dV 265, 53 29.3 / 32.1
// A causal walk of several heads is uneven: eight of 128 units and more (dK/dV of 2 x 12 (3) x 1836, 345 blocks, 61.8 / 48.1, of 32 (8) x 2048, 512 blocks, 62.2 / 57.6).
struct SplitLines {  // up to how many wavefronts: four splits, four of walks of so many units and more, eight, eight of walks of 128 units and more
  int four, units, four_long, eight, eight_long;
};
constexpr SplitLines split_lines(AttnPass pass, int D) {
  if (pass == ATTN_BWD_DKV) return {3328, 48, 6144, 2048, 4096};
  if (D == 32) return {4092, 128, 4092, 4088, 4088};
  if (D == 96) return {4092, 128, 4092, 2048, 2048};
  if (pass == ATTN_FWD) return D == 64 ? SplitLines{6144, 128, 6144, 4096, 4096} : SplitLines{3072, 56, 4608, 2048, 2048};
  return D == 64 ? SplitLines{3328, 75, 6144, 2048, 2048} : SplitLines{2624, 45, 3584, 2048, 2048};
}
int splits_of_two(AttnPass pass, int D, int64_t blocks, int64_t units) {
  const SplitLines at = split_lines(pass, D);
  const bool long_walk = units >= 128;
  const int least = splits_for(blocks, units, kMaxSplits, 0);  // (that fill half of the chip)
  if (blocks >= (long_walk ? 2304 : kResident) || units < 8) return least;
  const int four = units < at.units ? at.four : long_walk ? std::max(at.four_long, 4608) : at.four_long;
  if (units < 16 || 4 * blocks > four) return std::max(least, 2);
  return std::max(least, units >= 32 && 8 * blocks <= (long_walk ? at.eight_long : at.eight) ? 8 : 4);
}
template <AttnPass PASS, int D, int R>
int splits_of(int64_t blocks, int64_t units) {
  return R == 2 ? splits_of_two(PASS, D, blocks, units) : splits_for(blocks, units, kMaxSplits);
}

template <int D, bool DOC, int R>
int fwd(AttnParams p, hipStream_t st) {
  p.nqt = (p.Sq + 16 * R - 1) / (16 * R);
  const int64_t blocks = static_cast<int64_t>(p.nqt) * p.B * p.Hq;
  MltsKernelTimer timer("attn_fwd", st);
  return launch_splits<attn_small_fwd<D, DOC, R>, kMaxSplits>(blocks, splits_of<ATTN_FWD, D, R>(blocks, (p.Sk + kUnit - 1) / kUnit), R * D * 64, 2 * Unit<D>::BYTES, st, p,
                                                              RowArgs(p, D, true, p.Hq, p.nqt), "mlts_attn_fwd");
}

template <int D, bool DOC, int R>
int bwd_dq(AttnBwdParams bp, hipStream_t st) {
  AttnParams& p = bp.a;
  p.nqt = (p.Sq + 16 * R - 1) / (16 * R);
  const int64_t blocks = static_cast<int64_t>(p.nqt) * p.B * p.Hq;
  MltsKernelTimer timer("attn_bwd_dq", st);
  return launch_splits<attn_small_bwd_dq<D, DOC, R>, kMaxSplits>(blocks, splits_of<ATTN_BWD_DQ, D, R>(blocks, (p.Sk + kUnit - 1) / kUnit), R * D * 64, 2 * Unit<D>::BYTES, st, bp,
                                                                 RowArgs(p, D, true, p.Hq, p.nqt), "mlts_attn_bwd");
}

template <int D, bool DOC, int R>
int bwd_dkv(const AttnBwdParams& bp, hipStream_t st) {
  const AttnParams& p = bp.a;
  const int tiles = (p.Sk + 16 * R - 1) / (16 * R);
  const int64_t blocks = static_cast<int64_t>(tiles) * p.B * p.Hkv, units = static_cast<int64_t>((p.Sq + kUnit - 1) / kUnit) * (p.Hq / p.Hkv);
  MltsKernelTimer timer("attn_bwd_dkdv", st);
  return launch_splits<attn_small_bwd_dkv<D, DOC, R>, kMaxSplits>(blocks, splits_of<ATTN_BWD_DKV, D, R>(blocks, units), 2 * R * D * 64, 2 * Unit<D>::BYTES + 256, st, bp,
                                                                  RowArgs(p, D, true, p.Hkv, tiles), "mlts_attn_bwd");
}

}  // namespace

// Which calls of a pass come here; the others go to the 32-row kernels.
//
// The chain a 32-row workgroup walks has to be long: from 512 rows of the other side on, where those kernels take 12 us and more.  Shorter
// kernels differ by 4 us and less (4 heads x 2 x 200, by events: 10.4, 11.6 and 10.2 us there, 7.5, 7.3 and 7.7 here), which launching them hides: a forward and a
// backward call of that size take 41 us in a row of them and 51 alone with either, the host's time for one being 41; they keep one arithmetic
// for all batch sizes, which a number of splits that depends on the grid does not have.
//
// And the grid has to be small, for a block reads the other side for its 16 or 32 rows only.  us there -> here with one block of 16 rows to a
// wavefront / with two, forward, dQ, dK/dV (causal; blocks: of 16 rows; medians of three runs of 30 calls, all in turn on one GPU):
//   head_dim 64   512 blocks  8 heads x 1023     22.2 -> 13.2 / 14.6   23.9 -> 14.3 / 15.6   22.1 -> 13.5 / 15.1
//                 768         12 x 1024          21.5 -> 13.7 / 15.1   22.9 -> 15.1 / 17.5   21.2 -> 16.1 / 17.7
//                 896         7 x 4 x 512        14.5 -> 11.6 / 11.6   15.6 -> 13.1 / 11.9   14.1 -> 14.3 / 12.3
//                1024         8 x 2048           36.9 -> 23.5 / 21.6   38.4 -> 22.0 / 20.8   36.7 -> 29.2 / 24.2
//                1176         3 x 8 x 777        18.9 -> 16.0 / 15.6   20.7 -> 18.0 / 17.7   21.1 -> 20.0 / 19.7
//                2048         4 x 8 x 1024       22.5 -> 22.7 / 20.8   24.3 -> 21.9 / 21.1   25.4 -> 29.0 / 24.8
//                2048         8 x 4096           67.9 -> 64.8 / 42.5   70.2 -> 60.2 / 46.4   76.2 -> 87.3 / 58.3
//                2560         10 x 8 x 512       15.9 -> 17.0 / 16.2   17.6 -> 20.2 / 18.6   18.5 -> 23.7 / 22.8
//                3072         3 x 8 x 2048       38.8 -> 45.2 / 36.2   41.2 -> 52.6 / 39.2   47.3 -> 74.7 / 48.1
//                4096         4 x 8 x 2048       39.4 -> 55.3 / 42.3   43.8 -> 63.2 / 46.8   52.3 -> 72.3 / 62.2
//   head_dim 128  512         8 x 1023           27.2 -> 16.0 / 18.2   39.8 -> 18.0 / 20.9   35.2 -> 18.5
//                1024         2 x 8 x 1024       28.5 -> 23.1 / 21.4   41.5 -> 25.2 / 24.0   37.5 -> 27.7
//                1536         3 x 8 x 1024       28.8 -> 33.1 / 31.9   42.2 -> 37.3 / 31.9   38.2 -> 40.8
//                2048         2 x 8 x 2048       49.2 -> 58.3 / 45.6   72.3 -> 64.0 / 48.7   65.2 -> 77.2
//                3072         3 x 8 x 2048       55.2 -> 79.7 / 60.0   75.4 -> 92.0 / 67.8   67.6 ->  141
// Without a mask a block's work is twice that of a causal one:
//   head_dim 64   384         6 x 1024           20.3 -> 14.1 / 12.9   22.5 -> 15.2 / 13.1   20.1 -> 18.6 / 14.0
//                1024         2 x 8 x 1024       20.3 -> 18.6 / 17.6   22.9 -> 20.3 / 17.9   21.0 -> 24.1 / 20.1
//                1536         2 x 6 x 2048       35.5 -> 39.9 / 32.2   39.4 -> 42.8 / 33.5   45.6 -> 53.3 / 42.6
//                1536         6 x 8 x 512        13.6 -> 16.5 / 16.3   15.9 -> 18.6 / 17.6   17.4 -> 20.8 / 20.8
//   head_dim 128  512         8 x 1024           25.8 -> 20.1 / 18.8   40.1 -> 22.2 / 21.8   35.3 -> 24.7
//                1024         8 x 2048           45.6 -> 50.2 / 38.3   70.5 -> 55.6 / 42.3   64.0 -> 66.2
//                1536         6 x 4096           90.3 ->  143 / 103     137 ->  159 / 111     129 ->  191
// So two blocks from 832 (384 without a mask) on, short walks apart (8 x 32 heads x 64, head_dim 32, forward 6.8 / 7.9), and long walks, where a 32-row workgroup's chain is longest, up to larger grids.  Several
// query heads to a KV head lengthen the walk of dK/dV: 2 x 16 (4) heads x 1500 95.2 -> 47.9 / 37.8, 16 (4) x 2048 123 -> 46.9 / 47.1.
// (dK/dV of two blocks at head_dim 128 has no registers for its accumulators.)
//
// Documents stay with one block and smaller grids: what a row sees is not known here.  head_dim 64, documents of 64 to 446 rows, 2 x 8 x 1023, 17.0 -> 13.7,
// 17.5 -> 14.4, 18.5 -> 15.8; of 50 to 136, 4 x 4 x 2000, 15.4 -> 16.8, 16.8 -> 19.2, 17.4 -> 22.6; of 64 to 936, 2 x 8 x 2000, 34.0 -> 28.8, 34.0 -> 32.2, 37.4 -> 35.6.
//
// Walks below 704 rows, the 32-row kernels' chains being short: head_dim 64 causal 5 x 8 x 512, 1280 blocks, dK/dV 15.1 -> 17.2 with two; unmasked forward of 768,
// 3 x 8 x 512, 12.4 with one, 13.2 with two, dQ of 384, 3 x 4 x 512, 10.6 / 11.2; head_dim 128 causal dQ of 1280, 5 x 8 x 512, 25.6 -> 27.5, but unmasked of 768 25.7 -> 20.8
// with two.
constexpr int kShortWalk = 704, kLongWalk = 1408;
struct Lines {
  int blocks[3];  // up to which a call is served: of short walks, between, of long ones
};
constexpr Lines kLines[2][2][3] = {  // head_dim 128, causal, pass (forward, dQ, dK/dV)
    {{{{768, 1024, 1536}}, {{768, 1024, 1536}}, {{768, 1024, 1536}}}, {{{2048, 2048, 3072}}, {{2048, 2048, 3072}}, {{1024, 2048, 2560}}}},
    {{{{512, 512, 1024}}, {{1024, 1024, 1536}}, {{512, 512, 512}}}, {{{1024, 1024, 2048}}, {{1024, 2048, 3072}}, {{1024, 1024, 1024}}}}};

static bool half_walked(const AttnParams& p, int mode) { return mode == MLTS_MASK_CAUSAL && p.Sk <= p.Sq + p.Sq / 2; }
static int64_t row_blocks(AttnPass pass, const AttnParams& p) {
  const bool keys = pass == ATTN_BWD_DKV;
  return static_cast<int64_t>(((keys ? p.Sk : p.Sq) + 15) / 16) * p.B * (keys ? p.Hkv : p.Hq);
}

static int64_t walked(AttnPass pass, const AttnParams& p) { return pass == ATTN_BWD_DKV ? static_cast<int64_t>(p.Sq) * (p.Hq / p.Hkv) : p.Sk; }

// Two blocks of 16 rows to a wavefront.  (Of half of the blocks whose walk is that long, eight splits each still fill the chip.)
static bool two_blocks(AttnPass pass, const AttnParams& p, int D, int mode) {
  const int64_t blocks = row_blocks(pass, p), walk = walked(pass, p);
  if (walk < 96) return false;
  if (half_walked(p, mode)) return blocks >= 832 || (blocks >= 512 && walk >= 4096);
  if (walk < kShortWalk && (D == 64 || D == 128)) return D == 128 && blocks >= 512;
  return blocks >= 384;
}

bool mlts_attn_small_serves(AttnPass pass, const AttnParams& p, int D, int mode, const int64_t* dout_stride) {
  if ((pass == ATTN_BWD_DKV ? p.Sq : p.Sk) < 512) return false;
  const int64_t walk = walked(pass, p);
  const int which = pass == ATTN_FWD ? 0 : pass == ATTN_BWD_DQ ? 1 : 2;
  const int limit = mode == MLTS_MASK_DOC ? (D == 64 ? 1024 : 768) : kLines[D == 128][half_walked(p, mode)][which].blocks[walk >= kLongWalk ? 2 : walk >= kShortWalk ? 1 : 0];
  if (row_blocks(pass, p) > limit) return false;
  return near(p.Sq, p.qs) && near(p.Sk, p.ks) && near(p.Sk, p.vs) && near(p.Sq, p.os) && (!dout_stride || near(p.Sq, dout_stride));
}

// Whole passes at head_dim 32 and 96 without documents; bp: of the backward pass.  attn_tile16.hip, which takes rows at any alignment, shares 64-row
// tiles between four wavefronts, which wait for each other twice a tile and walk a row's whole length (us there -> here, forward, dQ, dK/dV; head_dim 32, then 96):
//   causal     8 x 1024           19.3 ->  9.7   19.3 ->  9.8   24.8 -> 11.6      31.6 -> 15.6   30.9 -> 16.7   37.9 -> 17.7
//              4 x 8 x 1024       21.6 -> 18.5   21.7 -> 18.2   29.5 -> 24.2      36.2 -> 29.5   39.4 -> 31.5   59.5 -> 45.7
//              8 x 16 x 1024      51.3 -> 48.1   55.6 -> 46.4   78.4 -> 62.4      92.7 -> 80.5    101 -> 90.1    158 ->  144
//              8 x 32 x 64         8.1 ->  6.9    8.1 ->  6.9    8.0 ->  7.2      10.2 ->  9.2   11.4 ->  9.7   10.9 -> 10.0
//              8 x 32 (8) x 300   15.9 -> 16.0   18.7 -> 17.2   30.8 -> 23.4      31.0 -> 27.6   36.3 -> 32.8   48.0 -> 39.7
//              4 x 32 (8) x 300   13.4 -> 13.1   13.4 -> 13.0   30.0 -> 16.8      23.1 -> 22.1   25.6 -> 26.5   46.2 -> 28.0
//              8 x 16 x 2048       164 ->  138    175 ->  134    263 ->  212       313 ->  272    341 ->  283    561 ->  522
//              2 x 32 (8) x 2048  84.9 -> 85.1   91.6 -> 81.9    165 ->  115       158 ->  134    175 ->  147    355 ->  299
//              16 x 8192           302 ->  305    331 ->  303    498 ->  415       576 ->  508    647 ->  554   1004 ->  949
//              4 x 16 x 8192      1153 ->  988   1259 ->  999   1958 -> 1546      2250 -> 1910   2501 -> 2012   4226 -> 3858
//   unmasked   8 x 8 x 1024       53.0 -> 45.1   55.8 -> 43.3   79.4 -> 61.9      96.5 -> 76.3    103 -> 78.5    148 ->  136
//              4 x 16 x 4096       611 ->  508    656 ->  509   1016 ->  787      1145 ->  944   1270 -> 1007   2076 -> 1880
// No grid up to 4 x 16 heads x 8192 is behind as a pass: two blocks share what a wavefront fetches, and it waits for nobody.  Single kernels are: by 1 % the
// forward at head_dim 32 of grids whose 4096 wavefronts are twice what is resident, by 3 % dQ at head_dim 96 of 4 x 32 (8) x 300, by 7 and 9 % forward and dQ there of 5 x 32 (8) x 120 (12.2, 13.2 us).
// Errors against 64 bits as there or up to a fifth smaller (dQ, dK, dV in fp32, 300 to 1024 rows).
bool mlts_attn_small_serves_parts(const AttnParams& p, int D, int mode, const AttnBwdParams* bp) {
  if ((D != 32 && D != 96) || mode == MLTS_MASK_DOC || p.Sq == 0 || p.Sk == 0) return false;
  const auto rows = [](const void* t, const int64_t* stride, int es) {
    return mlts_aligned16(t) && stride[0] * es % 16 == 0 && stride[1] * es % 16 == 0 && stride[2] * es % 16 == 0;
  };
  if (!rows(p.q, p.qs, 2) || !rows(p.k, p.ks, 2) || !rows(p.v, p.vs, 2) || !rows(p.o, p.os, 2)) return false;
  if (bp && (!rows(bp->dout, bp->dos, 2) || !rows(bp->dq_acc, bp->dqs, bp->dq_f32 ? 4 : 2) || !rows(bp->dk, bp->dks, bp->accumulate_f32 ? 4 : 2) ||
             !rows(bp->dv, bp->dvs, bp->accumulate_f32 ? 4 : 2) || !near(p.Sq, bp->dos)))
    return false;
  return near(p.Sq, p.qs) && near(p.Sk, p.ks) && near(p.Sk, p.vs) && near(p.Sq, p.os);
}

int mlts_attn_small_fwd(AttnParams p, int D, int mode, hipStream_t st) {
  set_causal_off(p, mode);
  if (mode == MLTS_MASK_DOC) return D == 64 ? fwd<64, true, 1>(p, st) : fwd<128, true, 1>(p, st);
  const bool two = two_blocks(ATTN_FWD, p, D, mode);
  if (D == 32) return two ? fwd<32, false, 2>(p, st) : fwd<32, false, 1>(p, st);
  if (D == 96) return two ? fwd<96, false, 2>(p, st) : fwd<96, false, 1>(p, st);
  if (D == 64) return two ? fwd<64, false, 2>(p, st) : fwd<64, false, 1>(p, st);
  return two ? fwd<128, false, 2>(p, st) : fwd<128, false, 1>(p, st);
}

// bp.delta_out and bp.lse2_out receive the row statistics
int mlts_attn_small_bwd_dq(AttnBwdParams bp, int D, int mode, hipStream_t st) {
  set_causal_off(bp.a, mode);
  if (mode == MLTS_MASK_DOC) return D == 64 ? bwd_dq<64, true, 1>(bp, st) : bwd_dq<128, true, 1>(bp, st);
  const bool two = two_blocks(ATTN_BWD_DQ, bp.a, D, mode);
  if (D == 32) return two ? bwd_dq<32, false, 2>(bp, st) : bwd_dq<32, false, 1>(bp, st);
  if (D == 96) return two ? bwd_dq<96, false, 2>(bp, st) : bwd_dq<96, false, 1>(bp, st);
  if (D == 64) return two ? bwd_dq<64, false, 2>(bp, st) : bwd_dq<64, false, 1>(bp, st);
  return two ? bwd_dq<128, false, 2>(bp, st) : bwd_dq<128, false, 1>(bp, st);
}

// reads bp.delta
int mlts_attn_small_bwd_dkv(AttnBwdParams bp, int D, int mode, hipStream_t st) {
  set_causal_off(bp.a, mode);
  if (mode == MLTS_MASK_DOC) return D == 64 ? bwd_dkv<64, true, 1>(bp, st) : bwd_dkv<128, true, 1>(bp, st);
  if (D == 32) return two_blocks(ATTN_BWD_DKV, bp.a, D, mode) ? bwd_dkv<32, false, 2>(bp, st) : bwd_dkv<32, false, 1>(bp, st);
  if (D == 96) return bwd_dkv<96, false, 1>(bp, st);
  if (D == 64) return two_blocks(ATTN_BWD_DKV, bp.a, D, mode) ? bwd_dkv<64, false, 2>(bp, st) : bwd_dkv<64, false, 1>(bp, st);
  return bwd_dkv<128, false, 1>(bp, st);
}

// The splits of a pass whose wavefronts have two blocks of 16 rows each (blocks: pairs of them), walking units of 32 rows; nothing is launched
extern "C" int32_t mlts_attn_small_splits(int32_t pass, int32_t head_dim, int64_t blocks, int64_t units) {
  return splits_of_two(pass == 0 ? ATTN_FWD : pass == 1 ? ATTN_BWD_DQ : ATTN_BWD_DKV, head_dim, blocks, units);
}
