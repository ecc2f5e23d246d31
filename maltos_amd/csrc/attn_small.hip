// bf16 attention at head_dim 64 and 128 on grids that leave most of the chip to few workgroups of the 32-row kernels (attn_fwd_dma.hip,
// attn_bwd_dq_tr.hip, attn_bwd_split.hip).
//
// Those give a workgroup 128 or 256 rows and walk the other side 64 rows at a time, one tile behind the other at about a microsecond each:
// with few rows and heads the kernel lasts as long as one workgroup's chain.  Here a wavefront owns 16 rows (queries in the forward and dQ
// kernels, keys in the dK/dV kernel) and takes every `splits`-th unit of 32 rows of the other side, so that there are up to 64 times as many
// wavefronts, with chains of a few units.  A unit arrives in whole lines, one unit ahead, and goes through LDS of its own wavefront to
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

// A unit of one operand: fetched, put to LDS, read as fragments.
template <int D>
struct Unit : Rows<D> {
  static constexpr int CHUNKS = D / 8, N = kUnit * CHUNKS / 64, BYTES = kUnit * Rows<D>::BYTES;
  bf16x8 raw[N];
  __device__ __forceinline__ void fetch(const bf16_t* base, int64_t stride, int row0, int last, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      raw[i] = *reinterpret_cast<const bf16x8*>(row_of(base, min(row0 + (64 / CHUNKS) * i + lane / CHUNKS, last), stride) + 8 * (lane % CHUNKS));
  }
  __device__ __forceinline__ void put(unsigned char* lds, int lane) const {
#pragma unroll
    for (int i = 0; i < N; ++i) *reinterpret_cast<bf16x8*>(lds + Rows<D>::at((64 / CHUNKS) * i + lane / CHUNKS, lane % CHUNKS)) = raw[i];
  }
};

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

// The splits' sums of N results of 16 rows, and what becomes of them: acc[n][db] are columns 16 db + 4 g ..+3 of this lane's row
template <int NC, int N, typename F>
__device__ __forceinline__ void join_and_store(f32x4 (&acc)[N][NC], f32x4* lds, const Place& at, F store) {
  if (at.splits == 1) {
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
      store(n, db, v);
    }
}

// O and LSE of 16 query rows
template <int D, bool DOC>
__global__ __launch_bounds__(kMaxSplits * 64) void attn_small_fwd(const AttnParams p, const RowArgs a) {
  typedef Unit<D> U;
  constexpr int FRAGS = D / 32, NC = D / 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g;
  // with a causal mask the last blocks are the long ones
  int bh, hq, member;
  const int qt = p.nqt - 1 - a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hq), hkv = a.group.over(hq, &member);
  const int q0 = 16 * qt, qrow = q0 + l16;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1];
  const bf16_t* q_row = row_of(static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1], min(qrow, p.Sq - 1), p.qs[2]);
  bf16x8 qf[FRAGS];
#pragma unroll
  for (int j = 0; j < FRAGS; ++j) qf[j] = *reinterpret_cast<const bf16x8*>(q_row + 32 * j + 8 * g);
  // keys this lane's query sees: up to klim (causal_off is Sk without a causal mask); documents also by the plan's bits
  const int klim = DOC || qrow < p.Sq ? min(p.Sk - 1, DOC ? p.Sk : qrow + p.causal_off) : -1;
  Walk<DOC, true> walk;
  walk.split = at.split, walk.splits = at.splits, walk.lane = lane;
  const unsigned long long* bits = nullptr;
  if (DOC) {
    const int group = q0 >> 6;
    walk.stats = p.k_stats + b * p.nk_stats;
    walk.own = p.q_stats[b * p.nq_stats + group];
    bits = p.doc_bits + (static_cast<int64_t>(b) * p.nq_stats + group) * p.nk_stats * 64 + (qrow & 63);
    walk.end = p.Sk;
  } else {
    walk.end = max(0, min(p.Sk, min(q0 + 16, p.Sq) + p.causal_off));
  }
  const int kend = at.there ? walk.end : 0;
  const int all_klim = DOC ? p.Sk - 1 : min(p.Sk - 1, min(q0, p.Sq - 1) + p.causal_off);  // seen by every row (that exists)

  float m = -INFINITY, l = 0.f;
  f32x4 o[1][NC];
#pragma unroll
  for (int db = 0; db < NC; ++db) o[0][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  U keys, values;
  unsigned char *lk = lds_raw + at.wave * 2 * U::BYTES, *lv = lk + U::BYTES;
  // (past the end the last key is fetched again: a branch around the loads would wait for all of them)
  unsigned long long word = 0, word_now = 0;
  bool masked = false, masked_now = false;
  auto fetch_keys = [&](int k) {
    keys.fetch(K, p.ks[2], k, p.Sk - 1, lane);
    if (DOC) word = bits[static_cast<int64_t>(min(k, p.Sk - 1) >> 6) * 64], masked = walk.masked;
  };
  int k0 = walk.first(0), kn = k0;
  if (k0 < kend) {
    fetch_keys(k0);
    values.fetch(V, p.vs[2], k0, p.Sk - 1, lane);
    keys.put(lk, lane), values.put(lv, lane);
    word_now = word, masked_now = masked;
    kn = walk.next(k0);
    fetch_keys(kn);
    values.fetch(V, p.vs[2], kn, p.Sk - 1, lane);
  }
  while (k0 < kend) {
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) s[u] = mfma32(U::dot(lk, u, j, l16, g), qf[j], s[u]);
    }
    if (k0 + kUnit - 1 > all_klim) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k0 + 16 * u + 4 * g + i > klim) s[u][i] = -INFINITY;
    }
    if (DOC && masked_now) {
      const uint32_t w = static_cast<uint32_t>(word_now >> (k0 & 32));
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (!((w >> (16 * u + 4 * g + i)) & 1)) s[u][i] = -INFINITY;
    }
    const int kn2 = kn < kend ? walk.next(kn) : kn;
    const unsigned long long word_next = word;
    const bool masked_next = masked;
    keys.put(lk, lane);  // the next unit's, which have had one unit's time to arrive
    fetch_keys(kn2);
    __builtin_amdgcn_sched_barrier(0);
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[u][i]);
    mx = max_groups(mx) * p.scale;
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
      const float m_new = fmaxf(m, mx);
      const float alpha = exponential(m - (m_new == -INFINITY ? 0.f : m_new));  // 1 for rows that do not rise, 0 from -inf
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < NC; ++db) o[0][db] *= alpha;
    }
    const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[u][i] = exponential(s[u][i] * p.scale - m_use);
        l += s[u][i];
      }
    const bf16x8 pr = pack(s);
#pragma unroll
    for (int db = 0; db < NC; ++db) o[0][db] = mfma32(U::columns(lv, db, l16, g), pr, o[0][db]);
    values.put(lv, lane);
    values.fetch(V, p.vs[2], kn2, p.Sk - 1, lane);
    k0 = kn, kn = kn2, word_now = word_next, masked_now = masked_next;
  }
  l = sum_groups(l);
  if (at.splits > 1) {  // every split holds some of the keys: all to the largest maximum
    __syncthreads();    // the units' LDS is free
    float* ml = reinterpret_cast<float*>(lds_raw) + at.slot * at.splits * 32;
    if (g == 0) ml[at.split * 32 + l16] = m, ml[at.split * 32 + 16 + l16] = l;
    __syncthreads();
    float m_new = -INFINITY;
    for (int s = 0; s < at.splits; ++s) m_new = fmaxf(m_new, ml[s * 32 + l16]);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exponential(m - m_use);
    l = 0.f;
    for (int s = 0; s < at.splits; ++s) l += ml[s * 32 + 16 + l16] * exponential(ml[s * 32 + l16] - m_use);
    m = m_new;
#pragma unroll
    for (int db = 0; db < NC; ++db) o[0][db] *= alpha;
  }
  const bool mine = at.there && qrow < p.Sq;
  if (mine && g == 0 && at.split == 0)
    p.lse[(static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + qrow] = l > 0.f ? m + logf(l) : -INFINITY;
  const int64_t row = b * p.os[0] + hq * p.os[1] + static_cast<int64_t>(qrow) * p.os[2] + 4 * g;
  const float scale = l > 0.f ? 1.0f / l : 0.f;
  join_and_store(o, reinterpret_cast<f32x4*>(lds_raw), at, [&](int, int db, f32x4 v) {
    if (mine) store4(p.o, row + 16 * db, v * scale, 0);
  });
}

// dQ of 16 query rows: dq = scale * sum_j ds_ij k_j, ds = p (dp - delta), p = exp(scale s - lse).  Runs first in a backward pass and writes
// delta = rowsum(dO * O) for the dK/dV kernel.  bp.dq_f32: dq is fp32 and added to (1) or overwritten (2); 0: bf16.
template <int D, bool DOC>
__global__ __launch_bounds__(kMaxSplits * 64) void attn_small_bwd_dq(const AttnBwdParams bp, const RowArgs a) {
  typedef Unit<D> U;
  constexpr int FRAGS = D / 32, NC = D / 16;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g;
  // with a causal mask the last blocks are the long ones
  int bh, hq, member;
  const int qt = p.nqt - 1 - a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hq), hkv = a.group.over(hq, &member);
  const int q0 = 16 * qt, qrow = q0 + l16, safe = min(qrow, p.Sq - 1);
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1];
  const bf16_t* q_row = row_of(static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hq * p.qs[1], safe, p.qs[2]);
  const bf16_t* do_row = row_of(static_cast<const bf16_t*>(bp.dout) + b * bp.dos[0] + hq * bp.dos[1], safe, bp.dos[2]);
  const bf16_t* o_row = row_of(static_cast<const bf16_t*>(p.o) + b * p.os[0] + hq * p.os[1], safe, p.os[2]);
  bf16x8 qf[FRAGS], dof[FRAGS];
  float delta = 0.f;
#pragma unroll
  for (int j = 0; j < FRAGS; ++j) {
    qf[j] = *reinterpret_cast<const bf16x8*>(q_row + 32 * j + 8 * g);
    dof[j] = *reinterpret_cast<const bf16x8*>(do_row + 32 * j + 8 * g);
    const bf16x8 of = *reinterpret_cast<const bf16x8*>(o_row + 32 * j + 8 * g);
#pragma unroll
    for (int e = 0; e < 8; ++e) delta += static_cast<float>(dof[j][e]) * static_cast<float>(of[e]);
  }
  delta = sum_groups(delta);
  const int64_t stat = (static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + safe;
  float lse = p.lse[stat];
  lse = qrow < p.Sq && lse != -INFINITY ? lse : INFINITY;  // rows that saw no key: every probability 0
  const bool mine = at.there && qrow < p.Sq;
  if (mine && g == 0 && at.split == 0) {  // the statistics of the backward pass, for whichever dK/dV kernel comes next
    bp.delta_out[stat] = delta;
    bp.lse2_out[stat] = lse * 1.44269504088896340736f;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) bp.lse2_out[static_cast<int64_t>(p.B) * p.Hq * p.Sq] = INFINITY;
  const int klim = DOC || qrow < p.Sq ? min(p.Sk - 1, DOC ? p.Sk : qrow + p.causal_off) : -1;
  Walk<DOC, true> walk;
  walk.split = at.split, walk.splits = at.splits, walk.lane = lane;
  const unsigned long long* bits = nullptr;
  if (DOC) {
    const int group = q0 >> 6;
    walk.stats = p.k_stats + b * p.nk_stats;
    walk.own = p.q_stats[b * p.nq_stats + group];
    bits = p.doc_bits + (static_cast<int64_t>(b) * p.nq_stats + group) * p.nk_stats * 64 + (qrow & 63);
    walk.end = p.Sk;
  } else {
    walk.end = max(0, min(p.Sk, min(q0 + 16, p.Sq) + p.causal_off));
  }
  const int kend = at.there ? walk.end : 0;
  const int all_klim = DOC ? p.Sk - 1 : min(p.Sk - 1, min(q0, p.Sq - 1) + p.causal_off);

  f32x4 dq[1][NC];
#pragma unroll
  for (int db = 0; db < NC; ++db) dq[0][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  U keys, values;
  unsigned char *lk = lds_raw + at.wave * 2 * U::BYTES, *lv = lk + U::BYTES;
  unsigned long long word = 0, word_now = 0;
  bool masked = false, masked_now = false;
  auto fetch = [&](int k) {  // (past the end the last key again: a branch around the loads would wait for all of them)
    keys.fetch(K, p.ks[2], k, p.Sk - 1, lane);
    values.fetch(V, p.vs[2], k, p.Sk - 1, lane);
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
    f32x4 s[2], dp[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = dp[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) {
        s[u] = mfma32(U::dot(lk, u, j, l16, g), qf[j], s[u]);
        dp[u] = mfma32(U::dot(lv, u, j, l16, g), dof[j], dp[u]);
      }
    }
    const bool edge = k0 + kUnit - 1 > all_klim;
    const uint32_t w = DOC && masked_now ? static_cast<uint32_t>(word_now >> (k0 & 32)) : ~0u;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float pv = exponential(s[u][i] * p.scale - lse);
        if (edge && k0 + 16 * u + 4 * g + i > klim) pv = 0.f;
        if (DOC && !((w >> (16 * u + 4 * g + i)) & 1)) pv = 0.f;
        s[u][i] = pv * (dp[u][i] - delta);
      }
    const bf16x8 ds = pack(s);
    bf16x8 kc[NC];
#pragma unroll
    for (int db = 0; db < NC; ++db) kc[db] = U::columns(lk, db, l16, g);
    const int kn2 = kn < kend ? walk.next(kn) : kn;
    put();  // the next unit's, which have had one unit's time to arrive
    fetch(kn2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int db = 0; db < NC; ++db) dq[0][db] = mfma32(kc[db], ds, dq[0][db]);
    k0 = kn, kn = kn2;
  }
  const int64_t row = b * bp.dqs[0] + hq * bp.dqs[1] + static_cast<int64_t>(qrow) * bp.dqs[2] + 4 * g;
  join_and_store(dq, reinterpret_cast<f32x4*>(lds_raw), at, [&](int, int db, f32x4 v) {
    if (mine) store4(bp.dq_acc, row + 16 * db, v * p.scale, bp.dq_f32);
  });
}

// dK, dV of 16 key rows of one KV head, summed over the query heads of its group.
template <int D, bool DOC>
__global__ __launch_bounds__(kMaxSplits * 64) void attn_small_bwd_dkv(const AttnBwdParams bp, const RowArgs a) {
  typedef Unit<D> U;
  constexpr int FRAGS = D / 32, NC = D / 16;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g;
  // with a causal mask the first blocks are the long ones
  int bh, hkv;
  const int kt = a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hkv), group = static_cast<int>(a.group.d);
  const int kb0 = kt * 16, krow = kb0 + l16, ksafe = min(krow, p.Sk - 1);
  const bf16_t* k_row = row_of(static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1], ksafe, p.ks[2]);
  const bf16_t* v_row = row_of(static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1], ksafe, p.vs[2]);
  bf16x8 kf[FRAGS], vf[FRAGS];
#pragma unroll
  for (int j = 0; j < FRAGS; ++j) {
    kf[j] = *reinterpret_cast<const bf16x8*>(k_row + 32 * j + 8 * g);
    vf[j] = *reinterpret_cast<const bf16x8*>(v_row + 32 * j + 8 * g);
  }
  const int qlim = DOC ? 0 : krow - p.causal_off;                               // first query that sees this lane's key
  const int all_qmin = DOC ? 0 : min(kb0 + 15, p.Sk - 1) - p.causal_off;        // from here on every key that exists is seen
  Walk<DOC, false> walk;
  walk.split = at.split, walk.splits = at.splits, walk.lane = lane, walk.end = p.Sq;
  const unsigned long long* bits = nullptr;
  int qstart = 0;
  if (DOC) {
    const int tile = kb0 >> 6;
    walk.stats = p.q_stats + b * p.nq_stats;
    walk.own = p.k_stats[b * p.nk_stats + tile];
    bits = p.doc_bits_k + (static_cast<int64_t>(b) * p.nk_stats + tile) * p.nq_stats * 64 + (krow & 63);
  } else {
    qstart = max(0, kb0 - p.causal_off) / kUnit * kUnit;
  }

  f32x4 dkv[2][NC];
#pragma unroll
  for (int db = 0; db < NC; ++db) dkv[0][db] = dkv[1][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  U queries, grads;
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
    queries.fetch(Q0 + head * p.qs[1], p.qs[2], q, p.Sq - 1, lane);
    grads.fetch(dO0 + head * bp.dos[1], bp.dos[2], q, p.Sq - 1, lane);
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
    f32x4 s[2], dp[2], lse[2], delta[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = dp[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) {
        s[u] = mfma32(U::dot(lq, u, j, l16, g), kf[j], s[u]);
        dp[u] = mfma32(U::dot(ld, u, j, l16, g), vf[j], dp[u]);
      }
      lse[u] = *reinterpret_cast<const f32x4*>(lstat + 16 * u + 4 * g);
      delta[u] = *reinterpret_cast<const f32x4*>(lstat + 32 + 16 * u + 4 * g);
    }
    const bool edge = !DOC && q0 < all_qmin;
    const uint32_t w = DOC && masked_now ? static_cast<uint32_t>(word_now >> (q0 & 32)) : ~0u;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float pv = exponential(s[u][i] * p.scale - lse[u][i]);
        if (edge && q0 + 16 * u + 4 * g + i < qlim) pv = 0.f;
        if (DOC && !((w >> (16 * u + 4 * g + i)) & 1)) pv = 0.f;
        s[u][i] = pv;
        dp[u][i] = pv * (dp[u][i] - delta[u][i]);
      }
    const bf16x8 pr = pack(s), ds = pack(dp);
    bf16x8 col[NC];
#pragma unroll
    for (int db = 0; db < NC; ++db) col[db] = U::columns(ld, db, l16, g);
#pragma unroll
    for (int db = 0; db < NC; ++db) dkv[1][db] = mfma32(col[db], pr, dkv[1][db]);
#pragma unroll
    for (int db = 0; db < NC; ++db) col[db] = U::columns(lq, db, l16, g);
    int hn2 = hn, qn2 = qn;
    if (hn < group) qn2 = walk.next(qn), skip(hn2, qn2);
    put();  // the next unit's, which have had one unit's time to arrive
    fetch(min(hn2, group - 1), qn2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int db = 0; db < NC; ++db) dkv[0][db] = mfma32(col[db], ds, dkv[0][db]);
    hg = hn, q0 = qn, hn = hn2, qn = qn2;
  }
  const bool mine = at.there && krow < p.Sk;
  const int64_t dk_row = b * bp.dks[0] + hkv * bp.dks[1] + static_cast<int64_t>(krow) * bp.dks[2] + 4 * g;
  const int64_t dv_row = b * bp.dvs[0] + hkv * bp.dvs[1] + static_cast<int64_t>(krow) * bp.dvs[2] + 4 * g;
  join_and_store(dkv, reinterpret_cast<f32x4*>(lds_raw), at, [&](int n, int db, f32x4 v) {
    if (mine) store4(n == 0 ? bp.dk : bp.dv, (n == 0 ? dk_row : dv_row) + 16 * db, n == 0 ? v * p.scale : v, bp.accumulate_f32);
  });
}

bool near(int64_t rows, const int64_t* stride) {  // offsets that row_of can form
  return rows < (1 << 24) && stride[2] < (1 << 23) && ((rows - 1) * stride[2] + 128) * 2 < (int64_t{1} << 32);
}

template <int D, bool DOC>
int fwd(AttnParams p, hipStream_t st) {
  p.nqt = (p.Sq + 15) / 16;
  const int64_t blocks = static_cast<int64_t>(p.nqt) * p.B * p.Hq;
  MltsKernelTimer timer("attn_fwd", st);
  return launch_splits<attn_small_fwd<D, DOC>, kMaxSplits>(blocks, splits_for(blocks, (p.Sk + kUnit - 1) / kUnit, kMaxSplits), D * 64, 2 * Unit<D>::BYTES, st, p,
                                                           RowArgs(p, D, true, p.Hq, p.nqt), "mlts_attn_fwd");
}

template <int D, bool DOC>
int bwd_dq(AttnBwdParams bp, hipStream_t st) {
  AttnParams& p = bp.a;
  p.nqt = (p.Sq + 15) / 16;
  const int64_t blocks = static_cast<int64_t>(p.nqt) * p.B * p.Hq;
  MltsKernelTimer timer("attn_bwd_dq", st);
  return launch_splits<attn_small_bwd_dq<D, DOC>, kMaxSplits>(blocks, splits_for(blocks, (p.Sk + kUnit - 1) / kUnit, kMaxSplits), D * 64, 2 * Unit<D>::BYTES, st, bp,
                                                              RowArgs(p, D, true, p.Hq, p.nqt), "mlts_attn_bwd");
}

template <int D, bool DOC>
int bwd_dkv(const AttnBwdParams& bp, hipStream_t st) {
  const AttnParams& p = bp.a;
  const int tiles = (p.Sk + 15) / 16;
  const int64_t blocks = static_cast<int64_t>(tiles) * p.B * p.Hkv, units = static_cast<int64_t>((p.Sq + kUnit - 1) / kUnit) * (p.Hq / p.Hkv);
  MltsKernelTimer timer("attn_bwd_dkdv", st);
  return launch_splits<attn_small_bwd_dkv<D, DOC>, kMaxSplits>(blocks, splits_for(blocks, units, kMaxSplits), 2 * D * 64, 2 * Unit<D>::BYTES + 256, st, bp,
                                                               RowArgs(p, D, true, p.Hkv, tiles), "mlts_attn_bwd");
}

}  // namespace

// Which calls of a pass come here; the others go to the 32-row kernels.
//
// The chain a 32-row workgroup walks has to be long: from 512 rows of the other side on, where those kernels take 12 us and more.  Shorter
// calls differ by 3 us and less (4 heads x 2 x 200: 8.4 us there, 5.5 here), which launching them hides; they keep one arithmetic for all
// batch sizes, which a number of splits that depends on the grid does not have.
//
// And the grid has to be small, for a 16-row block reads the other side for 16 rows only.  us there -> here, forward, dQ, dK/dV (causal):
//   head_dim 64    512 blocks  8 heads x 1024      20.0 21.7 18.8 ->  9.5 10.4 10.8     4 x 2048       34.0 35.8 33.5 -> 13.8 14.4 17.0
//                 1024 blocks  2 x 8 heads x 1024  20.1 21.9 19.4 -> 14.5 15.2 18.1     8 x 2048       35.0 36.9 35.0 -> 22.2 23.2 28.1
//                 1176 blocks  3 x 8 heads x 777   16.8 18.3 18.0 -> 13.9 16.2 17.6
//                 1536 blocks  3 x 8 heads x 1024  20.5 22.7 21.7 -> 18.2 20.7 22.2    12 x 2048       35.3 37.9 39.1 -> 26.0 31.2 37.1
//                 2048 blocks  4 x 8 heads x 1024  20.8 23.5 24.0 -> 21.2 24.8 28.4     8 x 4096       67.6 71.0 78.1 -> 66.2 77.4 98.3
//   head_dim 128   512 blocks  8 heads x 1024      24.8 38.5 33.1 -> 15.2 17.0 17.1     2 x 4096         85  129  113 ->   34   35   43
//                  768 blocks  3 x 4 heads x 1024  24.8 38.6 33.5 -> 22.4 26.0 26.6
//                 1024 blocks  8 x 4 heads x 512   16.1 24.6 20.7 -> 18.4 22.2 22.0
//   documents     1280 blocks  20 heads x 1023      15.2 16.4      -> 15.2 17.3
//                 1024 blocks  2 x 8 heads x 1023  15.3 16.1 17.0 -> 12.3 14.2 14.1  (a row of 1023, pieces of 1 to 255, 8 heads: 15.0 16.0
//                                                                                      15.8 ->  9.9 11.0 10.6)
//   two query heads and more to a KV head: dK/dV walks all of them.  2 x 16 (4) heads x 777 53.8 -> 26.0, 1 x 16 (4) x 2048 121 -> 49
// Without a mask a block's work is twice that of a causal one: head_dim 64 768 blocks 6 x 2048 32.7 36.4 33.5 -> 22.8 26.2 29.9, but 1024
// blocks 8 x 2048 32.5 37.4 34.8 -> 30.8 34.7 43.5; head_dim 128 256 blocks 4 x 1024 22.9 38.4 32.2 -> 13.5 15.6 15.6.
//
// The lines are one number of blocks for every length of the walk, up to which no measured call is behind.  They are not the
// break-even, which moves up with the length: of the calls above that are past their line, and so left to the 32-row kernels, these
// would be ahead here: 1536 causal blocks, forward and dQ of 3 x 8 heads x 1024 (11 and 9 %) and of 12 x 2048 (26 and 18 %), dK/dV of
// the latter (5 %); 1024 unmasked blocks, forward and dQ of 8 x 2048 (5 and 7 %).  The rule has no term for the length.
bool mlts_attn_small_serves(AttnPass pass, const AttnParams& p, int D, int mode, const int64_t* dout_stride) {
  const bool keys = pass == ATTN_BWD_DKV;
  if ((keys ? p.Sq : p.Sk) < 512) return false;
  const int64_t blocks = static_cast<int64_t>(((keys ? p.Sk : p.Sq) + 15) / 16) * p.B * (keys ? p.Hkv : p.Hq);
  const bool doc = mode == MLTS_MASK_DOC, half = doc || (mode == MLTS_MASK_CAUSAL && p.Sk <= p.Sq + p.Sq / 2);
  if (blocks > (D == 64 ? (!half ? 768 : keys || doc ? 1024 : 1280) : (half ? 768 : 384))) return false;
  return near(p.Sq, p.qs) && near(p.Sk, p.ks) && near(p.Sk, p.vs) && near(p.Sq, p.os) && (!dout_stride || near(p.Sq, dout_stride));
}

int mlts_attn_small_fwd(AttnParams p, int D, int mode, hipStream_t st) {
  set_causal_off(p, mode);
  if (mode == MLTS_MASK_DOC) return D == 64 ? fwd<64, true>(p, st) : fwd<128, true>(p, st);
  return D == 64 ? fwd<64, false>(p, st) : fwd<128, false>(p, st);
}

// bp.delta_out and bp.lse2_out receive the row statistics
int mlts_attn_small_bwd_dq(AttnBwdParams bp, int D, int mode, hipStream_t st) {
  set_causal_off(bp.a, mode);
  if (mode == MLTS_MASK_DOC) return D == 64 ? bwd_dq<64, true>(bp, st) : bwd_dq<128, true>(bp, st);
  return D == 64 ? bwd_dq<64, false>(bp, st) : bwd_dq<128, false>(bp, st);
}

// reads bp.delta
int mlts_attn_small_bwd_dkv(AttnBwdParams bp, int D, int mode, hipStream_t st) {
  set_causal_off(bp.a, mode);
  if (mode == MLTS_MASK_DOC) return D == 64 ? bwd_dkv<64, true>(bp, st) : bwd_dkv<128, true>(bp, st);
  return D == 64 ? bwd_dkv<64, false>(bp, st) : bwd_dkv<128, false>(bp, st);
}
