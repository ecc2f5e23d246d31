// fp32 attention backward at any head_dim <= 192 (attn_f32.hpp has the layout of the work).
#include "attn_f32.hpp"

namespace {

// dQ: dq = scale * sum_j ds_ij k_j, ds = p (dp - delta), p = exp(scale s - lse).  Runs first in a backward pass and writes
// delta = rowsum(dO * O) for the dK/dV kernel.  bp.dq_f32: dq is added to (1) or overwritten (0, 2).
template <int DP, int R, bool DOC, int LAYOUT>
__global__ __launch_bounds__(max_splits(DP, LAYOUT) * 64) void attn_f32_bwd_dq(const AttnBwdParams bp, const RowArgs a) {
  constexpr int FRAGS = DP / 16, NC = DP / 16, ROWS = 16 * R;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g, splits = at.splits, split = at.split, slot = at.slot;
  const bool there = at.there;
  // with a causal mask the last blocks are the long ones
  int bh, hq, member;
  const int qt = p.nqt - 1 - a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hq), hkv = a.group.over(hq, &member);
  const int q0 = qt * ROWS;
  const float* K = static_cast<const float*>(p.k) + b * p.ks[0] + hkv * p.ks[1];
  const float* V = static_cast<const float*>(p.v) + b * p.vs[0] + hkv * p.vs[1];

  f32x4 qf[R][FRAGS], dof[R][FRAGS];
  float delta[R], lse[R];
  int klim[R], qpos[R], qseq[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int qrow = q0 + 16 * r + l16;
    const int safe = min(qrow, p.Sq - 1);
    const float* q_row = row_of<LAYOUT>(static_cast<const float*>(p.q) + b * p.qs[0] + hq * p.qs[1], safe, p.qs[2]);
    const float* do_row = row_of<LAYOUT>(static_cast<const float*>(bp.dout) + b * bp.dos[0] + hq * bp.dos[1], safe, bp.dos[2]);
    const float* o_row = row_of<LAYOUT>(static_cast<const float*>(p.o) + b * p.os[0] + hq * p.os[1], safe, p.os[2]);
    delta[r] = 0.f;
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      const int d = 16 * j + 4 * g;
      qf[r][j] = inside<LAYOUT>(load_dot<LAYOUT>(q_row, d, a.D), d, a.D);
      dof[r][j] = inside<LAYOUT>(load_dot<LAYOUT>(do_row, d, a.D), d, a.D);
      const f32x4 of = inside<LAYOUT>(load_dot<LAYOUT>(o_row, d, a.D), d, a.D);
#pragma unroll
      for (int e = 0; e < 4; ++e) delta[r] += dof[r][j][e] * of[e];
    }
    delta[r] = sum_groups(delta[r]);
    const int64_t stat = (static_cast<int64_t>(b) * p.Hq + hq) * p.Sq + safe;
    lse[r] = p.lse[stat];
    lse[r] = (qrow < p.Sq && lse[r] != -INFINITY) ? lse[r] : INFINITY;  // rows that saw no key: every probability 0
    if (there && g == 0 && split == 0 && qrow < p.Sq) bp.delta_out[stat] = delta[r];
    klim[r] = qrow < p.Sq ? min(p.Sk - 1, qrow + p.causal_off) : -1;
  }
  Units<DOC, true> units;
  units.split = split, units.splits = splits, units.lane = lane;
  const int32_t *kpos = nullptr, *kseq = nullptr;
  if (DOC) {
    kpos = units.pos = p.k_pos + static_cast<int64_t>(b) * p.Sk;
    kseq = units.seq = p.k_seq + static_cast<int64_t>(b) * p.Sk;
    const int32_t *qp = p.q_pos + static_cast<int64_t>(b) * p.Sq, *qs = p.q_seq + static_cast<int64_t>(b) * p.Sq;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int qrow = q0 + 16 * r + l16;
      qpos[r] = qrow < p.Sq ? qp[qrow] : 0;
      qseq[r] = qrow < p.Sq ? qs[qrow] : -1;
    }
    units.own = id_range(qp, qs, q0, ROWS, p.Sq, lane);
    units.end = p.Sk;
  } else {
    units.end = max(0, min(p.Sk, min(q0 + ROWS, p.Sq) + p.causal_off));
  }
  const int kend = there ? units.end : 0;
  const int all_klim = DOC ? 0 : min(p.Sk - 1, min(q0, p.Sq - 1) + p.causal_off);

  f32x4 dq[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int db = 0; db < NC; ++db) dq[r][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 kf[FRAGS], vf[FRAGS];
  float* turn = lds + at.wave * Turn<DP>::FLOATS;
  int kp[4], ks[4], kp_now[4], ks_now[4];
  auto fetch = [&](int k) {
    const int safe = min(k + l16, p.Sk - 1);
    const float *k_row = row_of<LAYOUT>(K, safe, p.ks[2]), *v_row = row_of<LAYOUT>(V, safe, p.vs[2]);
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) kf[j] = load_dot<LAYOUT>(k_row, 16 * j + 4 * g, a.D), vf[j] = load_dot<LAYOUT>(v_row, 16 * j + 4 * g, a.D);
    if (DOC) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = min(k + 4 * g + i, p.Sk - 1);
        kp[i] = kpos[key], ks[i] = kseq[key];
      }
    }
  };
  int k0 = units.first(0);
  if (k0 < kend) fetch(k0);
  while (k0 < kend) {
    const int kn = units.next(k0);  // (past the end the last key is fetched again: a branch around the loads would wait for all of them)
    f32x4 s[R], dp[R];
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = dp[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      const f32x4 k = inside<LAYOUT>(kf[j], 16 * j + 4 * g, a.D), v = inside<LAYOUT>(vf[j], 16 * j + 4 * g, a.D);
      Turn<DP>::put(turn, j, kf[j], l16, g);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          s[r] = mfma4(k[c], qf[r][j][c], s[r]);
          dp[r] = mfma4(v[c], dof[r][j][c], dp[r]);
        }
    }
    if (DOC) {
#pragma unroll
      for (int i = 0; i < 4; ++i) kp_now[i] = kp[i], ks_now[i] = ks[i];
    }
    __builtin_amdgcn_sched_barrier(0);  // (the compiler moves the loads behind the products that they would arrive under)
    fetch(kn);
    __builtin_amdgcn_sched_barrier(0);
    const bool masked = !DOC && k0 + 15 > all_klim;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float pv = exponential(s[r][i] * p.scale - lse[r]);
        if (DOC) {
          if (!(kp_now[i] <= qpos[r] && ks_now[i] == qseq[r] && qseq[r] >= 0 && k0 + 4 * g + i < p.Sk)) pv = 0.f;
        } else if (masked && k0 + 4 * g + i > klim[r]) {
          pv = 0.f;
        }
        s[r][i] = pv * (dp[r][i] - delta[r]);
      }
    Columns<NC> ka[4];
    Turn<DP>::get(ka, turn, l16, g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int db = 0; db < NC; ++db)
#pragma unroll
        for (int r = 0; r < R; ++r) dq[r][db] = mfma4(ka[i].v[db], s[r][i], dq[r][db]);
    k0 = kn;
  }
  float* dQ = bp.dq_acc + b * bp.dqs[0] + hq * bp.dqs[1];
  float* row[R];
  float scale[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int qrow = q0 + 16 * r + l16;
    row[r] = there && qrow < p.Sq ? dQ + static_cast<int64_t>(qrow) * bp.dqs[2] : nullptr;
    scale[r] = p.scale;
  }
  if (!bp.rot.cos) {  // (known from the start, unlike what rotation_of_kernel fetches: forward and backward of 2 x 8 (4) x 777 of 64, us: 93.4 / 92.3)
    join_and_store(dq, lds + slot * splits * R * NC * 256, split, splits, row, scale, lane, a.D, a.vec_out, bp.dq_f32 == 1, AsIs{});
    return;
  }
  const RotateBack rot = rotation_of_kernel<decltype(attn_f32_bwd_dq<DP, R, DOC, LAYOUT>)>();
  Back<R> back{rot, {}};
#pragma unroll
  for (int r = 0; r < R; ++r) back.table[r] = rot.row(b, q0 + 16 * r + l16);
  join_and_store(dq, lds + slot * splits * R * NC * 256, split, splits, row, scale, lane, a.D, a.vec_out, bp.dq_f32 == 1, back);
}

template <int DP>
constexpr int kDkvFloats = 2 * Turn<DP>::FLOATS + 32;  // LDS of a wavefront

// dK, dV of R * 16 key rows of one KV head, summed over the query heads of its group.
template <int DP, int R, bool DOC, int LAYOUT>
__global__ __launch_bounds__(max_splits(DP, LAYOUT) * 64) void attn_f32_bwd_dkv(const AttnBwdParams bp, const RowArgs a) {
  constexpr int FRAGS = DP / 16, NC = DP / 16, ROWS = 16 * R;
  const AttnParams& p = bp.a;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const Place at(a);
  const int lane = at.lane, l16 = at.l16, g = at.g, splits = at.splits, split = at.split, slot = at.slot;
  const bool there = at.there;
  // with a causal mask the first blocks are the long ones
  int bh, hkv;
  const int kt = a.rank(a.batch_heads.over(at.block, &bh)), b = a.heads.over(bh, &hkv), group = static_cast<int>(a.group.d);
  const int kb0 = kt * ROWS;
  f32x4 kf[R][FRAGS], vf[R][FRAGS];
  int qlim[R], kpos[R], kseq[R];  // qlim: first query that sees this lane's key
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int krow = kb0 + 16 * r + l16;
    const int64_t ksafe = min(krow, p.Sk - 1);
    const float* K = static_cast<const float*>(p.k) + b * p.ks[0] + hkv * p.ks[1] + ksafe * p.ks[2];
    const float* V = static_cast<const float*>(p.v) + b * p.vs[0] + hkv * p.vs[1] + ksafe * p.vs[2];
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      const int d = 16 * j + 4 * g;
      kf[r][j] = inside<LAYOUT>(load_dot<LAYOUT>(K, d, a.D), d, a.D);
      vf[r][j] = inside<LAYOUT>(load_dot<LAYOUT>(V, d, a.D), d, a.D);
    }
    qlim[r] = krow < p.Sk ? krow - p.causal_off : 0x7fffffff;
    kpos[r] = 0, kseq[r] = -2;
  }
  const int all_qmin = min(kb0 + ROWS - 1, p.Sk - 1) - p.causal_off;  // from here on every key that exists is seen
  const bool ragged = kb0 + ROWS > p.Sk;
  Units<DOC, false> units;
  units.split = split, units.splits = splits, units.lane = lane, units.end = p.Sq;
  int qstart = 0;
  if (DOC) {
    const int32_t *kp = p.k_pos + static_cast<int64_t>(b) * p.Sk, *ks = p.k_seq + static_cast<int64_t>(b) * p.Sk;
    units.pos = p.q_pos + static_cast<int64_t>(b) * p.Sq;
    units.seq = p.q_seq + static_cast<int64_t>(b) * p.Sq;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int krow = kb0 + 16 * r + l16;
      if (krow < p.Sk) kpos[r] = kp[krow], kseq[r] = ks[krow];
    }
    units.own = id_range(kp, ks, kb0, ROWS, p.Sk, lane);
  } else {
    qstart = max(0, kb0 - p.causal_off) / 16 * 16;
  }

  f32x4 dkv[2 * R][NC];  // dK of each block, dV of each
#pragma unroll
  for (int n = 0; n < 2 * R; ++n)
#pragma unroll
    for (int db = 0; db < NC; ++db) dkv[n][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 qf[FRAGS], dof[FRAGS];
  float *turn_q = lds + at.wave * kDkvFloats<DP>, *turn_do = turn_q + Turn<DP>::FLOATS;
  float* lstat = turn_do + Turn<DP>::FLOATS;  // lse and delta of the unit's queries: a lane fetches one, and reads four of each
  float stat = 0.f;
  int row_fetched = 0;
  int qp[4], qs[4];
  const float* Q0 = static_cast<const float*>(p.q) + b * p.qs[0];
  const float* dO0 = static_cast<const float*>(bp.dout) + b * bp.dos[0];
  auto fetch = [&](int hg, int q) {
    const int head = hkv * group + hg;
    const float *Q = Q0 + head * p.qs[1], *dO = dO0 + head * bp.dos[1];
    const int safe = min(q + l16, p.Sq - 1);
    const float *q_row = row_of<LAYOUT>(Q, safe, p.qs[2]), *do_row = row_of<LAYOUT>(dO, safe, bp.dos[2]);
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) qf[j] = load_dot<LAYOUT>(q_row, 16 * j + 4 * g, a.D), dof[j] = load_dot<LAYOUT>(do_row, 16 * j + 4 * g, a.D);
    row_fetched = q + l16;
    stat = (lane & 16 ? bp.delta : p.lse)[(static_cast<int64_t>(b) * p.Hq + head) * p.Sq + min(row_fetched, p.Sq - 1)];
    if (DOC) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ok = min(q + 4 * g + i, p.Sq - 1);
        qp[i] = units.pos[ok], qs[i] = units.seq[ok];
      }
    }
  };
  // the units of all heads of the group, one after the other
  int hg = there ? 0 : group, q0 = units.first(qstart);
  auto skip = [&](int& h, int& q) {
    while (q >= p.Sq && ++h < group) q = units.first(qstart);
  };
  skip(hg, q0);
  if (hg < group) fetch(hg, q0);
  while (hg < group) {
    int hn = hg, qn = units.next(q0);
    skip(hn, qn);
    f32x4 s[R], dp[R];
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = dp[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) {
      const f32x4 q = inside<LAYOUT>(qf[j], 16 * j + 4 * g, a.D), o = inside<LAYOUT>(dof[j], 16 * j + 4 * g, a.D);
      Turn<DP>::put(turn_q, j, qf[j], l16, g);
      Turn<DP>::put(turn_do, j, dof[j], l16, g);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          s[r] = mfma4(q[c], kf[r][j][c], s[r]);
          dp[r] = mfma4(o[c], vf[r][j][c], dp[r]);
        }
    }
    // probability 0: rows past the end, rows that saw no key
    lstat[lane & 31] = (lane & 16) == 0 && (row_fetched >= p.Sq || stat == -INFINITY) ? INFINITY : stat;
    int qp_now[4], qs_now[4];
    if (DOC) {
#pragma unroll
      for (int i = 0; i < 4; ++i) qp_now[i] = qp[i], qs_now[i] = qs[i];
    }
    // (past the end the last query is fetched again: a branch around the loads would wait for all of them; without the barriers the
    // compiler moves them behind the products that they would arrive under)
    __builtin_amdgcn_sched_barrier(0);
    fetch(min(hn, group - 1), qn);
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 lse_now = *reinterpret_cast<const f32x4*>(lstat + 4 * g), delta_now = *reinterpret_cast<const f32x4*>(lstat + 16 + 4 * g);
    const bool masked = !DOC && (q0 < all_qmin || ragged);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float pv = exponential(s[r][i] * p.scale - lse_now[i]);
        if (DOC) {
          if (!(kpos[r] <= qp_now[i] && kseq[r] == qs_now[i] && qs_now[i] >= 0)) pv = 0.f;
        } else if (masked && q0 + 4 * g + i < qlim[r]) {
          pv = 0.f;
        }
        s[r][i] = pv;
        dp[r][i] = pv * (dp[r][i] - delta_now[i]);
      }
    Columns<NC> rows[4];
    Turn<DP>::get(rows, turn_do, l16, g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int db = 0; db < NC; ++db)
#pragma unroll
        for (int r = 0; r < R; ++r) dkv[R + r][db] = mfma4(rows[i].v[db], s[r][i], dkv[R + r][db]);
    Turn<DP>::get(rows, turn_q, l16, g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int db = 0; db < NC; ++db)
#pragma unroll
        for (int r = 0; r < R; ++r) dkv[r][db] = mfma4(rows[i].v[db], dp[r][i], dkv[r][db]);
    hg = hn, q0 = qn;
  }
  float* row[2 * R];
  float scale[2 * R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t krow = kb0 + 16 * r + l16;
    const bool mine = there && krow < p.Sk;
    row[r] = mine ? static_cast<float*>(bp.dk) + b * bp.dks[0] + hkv * bp.dks[1] + krow * bp.dks[2] : nullptr;
    row[R + r] = mine ? static_cast<float*>(bp.dv) + b * bp.dvs[0] + hkv * bp.dvs[1] + krow * bp.dvs[2] : nullptr;
    scale[r] = p.scale, scale[R + r] = 1.f;
  }
  if (!bp.rot.cos) {
    join_and_store(dkv, lds + slot * splits * 2 * R * NC * 256, split, splits, row, scale, lane, a.D, a.vec_out, bp.accumulate_f32 != 0, AsIs{});
    return;
  }
  const RotateBack rot = rotation_of_kernel<decltype(attn_f32_bwd_dkv<DP, R, DOC, LAYOUT>)>();
  Back<2 * R> back{rot, {}};
#pragma unroll
  for (int r = 0; r < R; ++r) back.table[r] = rot.row(b, kb0 + 16 * r + l16), back.table[R + r] = -1;
  join_and_store(dkv, lds + slot * splits * 2 * R * NC * 256, split, splits, row, scale, lane, a.D, a.vec_out, bp.accumulate_f32 != 0, back);
}

template <int DP, int R, bool DOC, int LAYOUT>
int bwd_dq(AttnBwdParams bp, int D, hipStream_t st) {
  AttnParams& p = bp.a;
  p.nqt = (p.Sq + 16 * R - 1) / (16 * R);
  const int64_t blocks = static_cast<int64_t>(p.nqt) * p.B * p.Hq;
  const RowArgs a(p, D, LAYOUT != ROWS_ANY && rows_vec(bp.dqs, bp.dq_acc), p.Hq, p.nqt);
  MltsKernelTimer timer("attn_bwd_dq", st);
  const int splits = splits_for(blocks, (p.Sk + 15) / 16, max_splits(DP, LAYOUT));
  return launch_splits<attn_f32_bwd_dq<DP, R, DOC, LAYOUT>, max_splits(DP, LAYOUT)>(blocks, splits, R * DP * 64, Turn<DP>::FLOATS * 4, st, bp, a,
                                                                                    "mlts_attn_bwd");
}

template <int DP, int R, bool DOC, int LAYOUT>
int bwd_dkv(const AttnBwdParams& bp, int D, hipStream_t st) {
  const AttnParams& p = bp.a;
  const int tiles = (p.Sk + 16 * R - 1) / (16 * R);
  const int64_t blocks = static_cast<int64_t>(tiles) * p.B * p.Hkv;
  const RowArgs a(p, D, LAYOUT != ROWS_ANY && rows_vec(bp.dks, bp.dk) && rows_vec(bp.dvs, bp.dv), p.Hkv, tiles);
  MltsKernelTimer timer("attn_bwd_dkdv", st);
  const int splits = splits_for(blocks, static_cast<int64_t>((p.Sq + 15) / 16) * (p.Hq / p.Hkv), max_splits(DP, LAYOUT));
  return launch_splits<attn_f32_bwd_dkv<DP, R, DOC, LAYOUT>, max_splits(DP, LAYOUT)>(blocks, splits, 2 * R * DP * 64, kDkvFloats<DP> * 4, st, bp, a,
                                                                                     "mlts_attn_bwd");
}

template <int DP, bool DOC, int LAYOUT>
int bwd(AttnBwdParams bp, int D, hipStream_t st) {
  constexpr int TWO = DP <= 64 ? 2 : 1;  // blocks of 16 rows to a wavefront: attn_f32.hpp has both sides of the lines
  const AttnParams& p = bp.a;
  if (p.Sq > 0) {
    const bool two = static_cast<int64_t>((p.Sq + 31) / 32) * p.B * p.Hq >= kResident / 2;
    if (int rc = two ? bwd_dq<DP, TWO, DOC, LAYOUT>(bp, D, st) : bwd_dq<DP, 1, DOC, LAYOUT>(bp, D, st); rc != MLTS_OK) return rc;
  }
  if (p.Sk == 0) return MLTS_OK;
  const bool two = static_cast<int64_t>((p.Sk + 31) / 32) * p.B * p.Hkv >= (DP == 32 ? 512 : 352) && static_cast<int64_t>(p.Sq) * (p.Hq / p.Hkv) > 256;
  return two ? bwd_dkv<DP, TWO, DOC, LAYOUT>(bp, D, st) : bwd_dkv<DP, 1, DOC, LAYOUT>(bp, D, st);
}

}  // namespace

// bp.delta_out receives rowsum(dO * O); bp.delta must point at the same buffer
int mlts_attn_f32_bwd(AttnBwdParams bp, int D, int mode, hipStream_t st) {
  set_causal_off(bp.a, mode);
  const AttnParams& p = bp.a;
  const bool vec = D % 4 == 0 && rows_vec(p.qs, p.q) && rows_vec(p.ks, p.k) && rows_vec(p.vs, p.v) && rows_vec(p.os, p.o) && rows_vec(bp.dos, bp.dout);
  const bool whole = vec && D % 32 == 0 && rows_near(p.Sq, p.qs[2], D) && rows_near(p.Sk, p.ks[2], D) && rows_near(p.Sk, p.vs[2], D) &&
                     rows_near(p.Sq, p.os[2], D) && rows_near(p.Sq, bp.dos[2], D);
  MLTS_F32_DISPATCH(bwd, bp, D, st);
}
