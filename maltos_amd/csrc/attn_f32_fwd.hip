// fp32 attention forward at any head_dim <= 192 (attn_f32.hpp has the layout of the work).
#include "attn_f32.hpp"

namespace {

// O and LSE of 16 query rows.  DP: head_dim rounded up to a multiple of 32 (the padding is zero in every dot product).
template <int DP, bool DOC, int LAYOUT>
__global__ __launch_bounds__(max_splits(DP, LAYOUT) * 64) void attn_f32_fwd(const AttnParams p, const RowArgs a) {
  constexpr int FRAGS = DP / 16, NC = DP / 16;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g, splits = at.splits, split = at.split, slot = at.slot;
  const bool there = at.there;
  // with a causal mask the last blocks are the long ones
  int bh, hq, member;
  const int qt = p.nqt - 1 - a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hq), hkv = a.group.over(hq, &member);
  const int q0 = 16 * qt, qrow = q0 + l16;
  const float* K = static_cast<const float*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const float* V = static_cast<const float*>(p.v) + b * p.vs[0] + hkv * p.vs[1];
  const float* q_row = row_of<LAYOUT>(static_cast<const float*>(p.q) + b * p.qs[0] + hq * p.qs[1], min(qrow, p.Sq - 1), p.qs[2]);
  f32x4 qf[FRAGS];
#pragma unroll
  for (int j = 0; j < FRAGS; ++j) qf[j] = inside<LAYOUT>(load_dot<LAYOUT>(q_row, 16 * j + 4 * g, a.D), 16 * j + 4 * g, a.D);
  // keys this lane's query sees: up to klim (causal_off is Sk without a causal mask); documents also by their ids
  const int klim = qrow < p.Sq ? min(p.Sk - 1, qrow + p.causal_off) : -1;
  int qpos = 0, qseq = -1;
  Units<DOC, true> units;
  units.split = split, units.splits = splits, units.lane = lane;
  if (DOC) {
    units.pos = p.k_pos + static_cast<int64_t>(b) * p.Sk;
    units.seq = p.k_seq + static_cast<int64_t>(b) * p.Sk;
    const int32_t *qp = p.q_pos + static_cast<int64_t>(b) * p.Sq, *qs = p.q_seq + static_cast<int64_t>(b) * p.Sq;
    if (qrow < p.Sq) qpos = qp[qrow], qseq = qs[qrow];
    units.own = id_range(qp, qs, q0, 16, p.Sq, lane);
    units.end = p.Sk;
  } else {
    units.end = max(0, min(p.Sk, min(q0 + 16, p.Sq) + p.causal_off));
  }
  const int kend = there ? units.end : 0;
  const int all_klim = DOC ? 0 : min(p.Sk - 1, min(q0, p.Sq - 1) + p.causal_off);  // seen by every row (that exists)

  float m = -INFINITY, l = 0.f;
  f32x4 o[1][NC];
#pragma unroll
  for (int db = 0; db < NC; ++db) o[0][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 kf[FRAGS];
  Columns<NC> vf[4];
  int kp[4], ks[4];
  auto fetch_k = [&](int k) {
    const float* row = row_of<LAYOUT>(K, min(k + l16, p.Sk - 1), p.ks[2]);
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) kf[j] = load_dot<LAYOUT>(row, 16 * j + 4 * g, a.D);
    if (DOC) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = min(k + 4 * g + i, p.Sk - 1);
        kp[i] = units.pos[key], ks[i] = units.seq[key];
      }
    }
  };
  auto fetch_v = [&](int k) {
#pragma unroll
    for (int i = 0; i < 4; ++i) vf[i].template load<LAYOUT>(row_of<LAYOUT>(V, min(k + 4 * g + i, p.Sk - 1), p.vs[2]), NC * l16, a.D);
  };
  int k0 = units.first(0);
  if (k0 < kend) fetch_k(k0), fetch_v(k0);
  while (k0 < kend) {
    const int kn = units.next(k0);
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      const f32x4 k = inside<LAYOUT>(kf[j], 16 * j + 4 * g, a.D);
#pragma unroll
      for (int c = 0; c < 4; ++c) s = mfma4(k[c], qf[j][c], s);
    }
    if (DOC) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!(kp[i] <= qpos && ks[i] == qseq && qseq >= 0 && k0 + 4 * g + i < p.Sk)) s[i] = -INFINITY;
    } else if (k0 + 15 > all_klim) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k0 + 4 * g + i > klim) s[i] = -INFINITY;
    }
    fetch_k(kn);  // (past the end the last key is fetched again: a branch around the loads would wait for all of them)
    const float mx = max_groups(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))) * p.scale;
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
    for (int i = 0; i < 4; ++i) {
      s[i] = exponential(s[i] * p.scale - m_use);
      l += s[i];
    }
    accumulate(o[0], vf, s);
    fetch_v(kn);
    k0 = kn;
  }
  l = sum_groups(l);
  if (splits > 1) {  // every split holds some of the keys: all to the largest maximum
    float* ml = lds + slot * splits * 32;
    if (g == 0) ml[split * 32 + l16] = m, ml[split * 32 + 16 + l16] = l;
    __syncthreads();
    float m_new = -INFINITY;
    for (int s = 0; s < splits; ++s) m_new = fmaxf(m_new, ml[s * 32 + l16]);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exponential(m - m_use);
    l = 0.f;
    for (int s = 0; s < splits; ++s) l += ml[s * 32 + 16 + l16] * exponential(ml[s * 32 + l16] - m_use);
    m = m_new;
#pragma unroll
    for (int db = 0; db < NC; ++db) o[0][db] *= alpha;
  }
  if (there && g == 0 && split == 0 && qrow < p.Sq)
    p.lse[(static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + qrow] = l > 0.f ? m + logf(l) : -INFINITY;
  float* const row[1] = {there && qrow < p.Sq ? static_cast<float*>(p.o) + b * p.os[0] + hq * p.os[1] + static_cast<int64_t>(qrow) * p.os[2] : nullptr};
  const float scale[1] = {l > 0.f ? 1.0f / l : 0.f};
  join_and_store(o, lds + slot * splits * NC * 256, split, splits, row, scale, lane, a.D, a.vec_out, false, AsIs{});
}

template <int DP, bool DOC, int LAYOUT>
int fwd(AttnParams p, int D, bool vec_out, hipStream_t st) {
  p.nqt = (p.Sq + 15) / 16;
  const int64_t blocks = static_cast<int64_t>(p.nqt) * p.B * p.Hq;
  const int splits = splits_for(blocks, (p.Sk + 15) / 16, max_splits(DP, LAYOUT));
  MltsKernelTimer timer("attn_fwd", st);
  return launch_splits<attn_f32_fwd<DP, DOC, LAYOUT>, max_splits(DP, LAYOUT)>(blocks, splits, DP * 64, 0, st, p, RowArgs(p, D, vec_out, p.Hq, p.nqt),
                                                                              "mlts_attn_fwd");
}

}  // namespace

int mlts_attn_f32_fwd(AttnParams p, int D, int mode, hipStream_t st) {
  set_causal_off(p, mode);
  const bool vec = D % 4 == 0 && rows_vec(p.qs, p.q) && rows_vec(p.ks, p.k) && rows_vec(p.vs, p.v);
  const bool whole = vec && D % 32 == 0 && rows_near(p.Sq, p.qs[2], D) && rows_near(p.Sk, p.ks[2], D) && rows_near(p.Sk, p.vs[2], D);
  MLTS_F32_DISPATCH(fwd, p, D, vec && rows_vec(p.os, p.o), st);
}
