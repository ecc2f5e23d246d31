// Attention backward, dK and dV, head_dim 64, bf16, large grids.
//
// A wavefront owns 32 keys of one KV head with both accumulators (dK, dV) and both operands (K, V) in registers: at this head_dim they fit
// beside the scores of a tile.  The four wavefronts of a workgroup walk the 64-row query tiles that can see their keys (all query heads of
// the group) together: Q, dO, lse2 and delta of a tile go through LDS once for all of them, two stages, one barrier a tile; the tile behind
// the next is on its way from memory.  Two workgroups share a compute unit and fill each other's waits.
//
// Against the two-role kernel of attn_bwd_split.hip, whose wavefronts hand the probabilities over in LDS (head_dim 128 has no registers for
// anything else): no hand-over, no second barrier chain, and the arithmetic of one wavefront beside the products of another.  8 x 8 heads x
// 2048 causal 114 -> 97 us, 4 x 16 x 4096 412 -> 329 us (290 on another card).  By counters the matrix cores are busy 37 % of that time (44 %
// in the larger call) and the vector port 48 % (54 %): what is left is what of the two does not overlap.
#include "attn_bf16.hpp"

namespace {

constexpr int kTile = 64;  // query rows

constexpr int R = 2;       // 16-key blocks of a wavefront

struct Dkv64Args {
  Divisor heads, batch;
};

// element i of the lanes of 16-lane group g <-> element g of those of group i
__device__ __forceinline__ void transpose_groups(uint32_t (&v)[4]) {
  const auto swap32 = [&](int i, int j) {
    const auto r = __builtin_amdgcn_permlane32_swap(v[i], v[j], false, false);
    v[i] = r[0], v[j] = r[1];
  };
  const auto swap16 = [&](int i, int j) {
    const auto r = __builtin_amdgcn_permlane16_swap(v[i], v[j], false, false);
    v[i] = r[0], v[j] = r[1];
  };
  swap32(0, 2), swap32(1, 3), swap16(0, 1), swap16(2, 3);
}

template <int MODE, bool ROTATED>
__global__ __launch_bounds__(256, 2) void attn_bwd_dkv64_kernel(const AttnBwdParams bp, const float* __restrict__ lse2, const Dkv64Args a) {
  typedef Rows<64> L;
  constexpr bool DOC = MODE == MLTS_MASK_DOC, CAUSAL = MODE == MLTS_MASK_CAUSAL;
  constexpr int NC = 4, KEYS = 64 * R, OPERAND = kTile * L::BYTES;
  constexpr int STAGE = 2 * OPERAND + 512 + (DOC ? KEYS * 8 : 0);
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * STAGE];
  const AttnParams& p = bp.a;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // with a causal mask the first blocks are the long ones; documents: the plan's order
  int hkv, b;
  int entry = a.heads.over(static_cast<int>(blockIdx.x), &hkv);
  if (DOC && p.kblock_order) entry = p.kblock_order[entry];
  const int kt = a.batch.over(entry, &b);
  const int kb0 = kt * KEYS, kw = kb0 + 16 * R * wave;  // first key of the workgroup, of the wavefront
  const int tiles = (p.Sq + kTile - 1) / kTile, group = p.Hq / p.Hkv;

  bf16x8 kf[R][2], vf[R][2];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = min(kw + 16 * r + l16, p.Sk - 1);
    const bf16_t* k_row = static_cast<const bf16_t*>(p.k) + b * p.ks[0] + hkv * p.ks[1] + row * p.ks[2] + 8 * g;
    const bf16_t* v_row = static_cast<const bf16_t*>(p.v) + b * p.vs[0] + hkv * p.vs[1] + row * p.vs[2] + 8 * g;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      kf[r][j] = *reinterpret_cast<const bf16x8*>(k_row + 32 * j);
      vf[r][j] = *reinterpret_cast<const bf16x8*>(v_row + 32 * j);
    }
  }

  // the query tiles, one after the other, of every head of the group
  DocTileScan scan;
  int4 grp[R], own{};
  const int4* stats = nullptr;
  if (DOC) {
    stats = p.q_stats + static_cast<int64_t>(b) * p.nq_stats;
#pragma unroll
    for (int i = 0; i < R; ++i) grp[i] = p.k_stats[static_cast<int64_t>(b) * p.nk_stats + min((kb0 >> 6) + i, p.nk_stats - 1)];
    own = wave >> 1 ? grp[1] : grp[0];
  }
  const int first = CAUSAL ? max(0, kb0 - p.causal_off) / kTile : 0;
  struct Tile {
    int head, j, cls;  // cls: how the wavefront's keys are seen (documents)
  };
  auto find = [&](Tile t) {  // the first tile from t on
    for (;;) {
      if (DOC) t.j = doc_scan_next<R, false>(scan, t.j, tiles, p.nq_stats, stats, grp, own, lane);
      if (t.j < tiles || t.head + 1 >= group) break;
      ++t.head, t.j = first;
    }
    if (DOC && t.j < tiles) t.cls = doc_scan_class(scan, t.j);
    return t;
  };
  auto after = [&](Tile t) {
    if (t.j < tiles) ++t.j;
    return find(t);
  };

  u32x4 raw[4];
  float stat = 0.f;
  unsigned long long word = 0;
  const bf16_t* Q0 = static_cast<const bf16_t*>(p.q) + b * p.qs[0] + hkv * group * p.qs[1] + 8 * (tid & 7);
  const bf16_t* dO0 = static_cast<const bf16_t*>(bp.dout) + b * bp.dos[0] + hkv * group * bp.dos[1] + 8 * (tid & 7);
  const int64_t stat0 = (static_cast<int64_t>(b) * p.Hq + hkv * group) * p.Sq;
  auto fetch = [&](const Tile& t) {  // (past the end the last row again: a branch around the loads would wait for all of them)
    const int q0 = min(t.j, tiles - 1) * kTile;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t row = min(q0 + 32 * i + (tid >> 3), p.Sq - 1);
      raw[i] = *reinterpret_cast<const u32x4*>(Q0 + t.head * p.qs[1] + row * p.qs[2]);
      raw[2 + i] = *reinterpret_cast<const u32x4*>(dO0 + t.head * bp.dos[1] + row * bp.dos[2]);
    }
    const int row = q0 + (tid & 63);
    const float* src = tid & 64 ? bp.delta : lse2;
    stat = src[stat0 + static_cast<int64_t>(t.head) * p.Sq + min(row, p.Sq - 1)];
    stat = tid & 64 ? -stat : row < p.Sq ? stat : INFINITY;  // queries past the end: probability 0
    if (DOC)
      word = p.doc_bits_k[((static_cast<int64_t>(b) * p.nk_stats + min((kb0 >> 6) + ((tid >> 6) & 1), p.nk_stats - 1)) * p.nq_stats +
                           min(t.j, tiles - 1)) * 64 + (tid & 63)];
  };
  auto put = [&](int stage) {
    unsigned char* s = lds + stage * STAGE;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(s + (i >> 1) * OPERAND + L::at(32 * (i & 1) + (tid >> 3), tid & 7)) = raw[i];
    if (tid < 128) {
      reinterpret_cast<float*>(s + 2 * OPERAND)[tid] = stat;
      if (DOC && tid < KEYS) reinterpret_cast<unsigned long long*>(s + 2 * OPERAND + 512)[tid] = word;
    }
  };

  f32x4 dk[R][NC], dv[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int db = 0; db < NC; ++db) dk[r][db] = dv[r][db] = f32x4{0.f, 0.f, 0.f, 0.f};

  Tile now = find({0, first, TILE_FULL}), next = now;
  if (now.j < tiles) {
    fetch(now);
    put(0);
    next = after(now);
    fetch(next);
  }
  int stage = 0;
  while (now.j < tiles) {
    __syncthreads();  // this tile is in LDS, and nobody reads the other stage any more
    put(stage ^ 1);
    const Tile then = after(next);
    fetch(then);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char *lq = lds + stage * STAGE, *ld = lq + OPERAND;
    const float* lstat = reinterpret_cast<const float*>(ld + OPERAND);
    const unsigned long long* words = reinterpret_cast<const unsigned long long*>(lstat + 128) + 16 * R * wave + l16;
    f32x4 s[2][R][2], dp[2][R][2];
    bf16x8 pr[R], ds[R];
    auto scores = [&](int u) {
      const unsigned char *uq = lq + 32 * u * L::BYTES, *ud = ld + 32 * u * L::BYTES;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const f32x4 delta = *reinterpret_cast<const f32x4*>(lstat + 64 + 32 * u + 16 * v + 4 * g);
#pragma unroll
        for (int r = 0; r < R; ++r) s[u][r][v] = f32x4{0.f, 0.f, 0.f, 0.f}, dp[u][r][v] = delta;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const bf16x8 q = L::dot(uq, v, j, l16, g), o = L::dot(ud, v, j, l16, g);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            s[u][r][v] = mfma32(q, kf[r][j], s[u][r][v]);
            dp[u][r][v] = mfma32(o, vf[r][j], dp[u][r][v]);
          }
        }
      }
    };
    auto probabilities = [&](int u) {
      f32x4 lse[2];
#pragma unroll
      for (int v = 0; v < 2; ++v) lse[v] = *reinterpret_cast<const f32x4*>(lstat + 32 * u + 16 * v + 4 * g);
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float pv = __builtin_amdgcn_exp2f(fmaf(s[u][r][v][i], p.scale_log2, -lse[v][i]));
            s[u][r][v][i] = pv;
            dp[u][r][v][i] *= pv;
          }
        pr[r] = pack(s[u][r]), ds[r] = pack(dp[u][r]);
      }
    };
    auto products = [&](int u) {
      const unsigned char *uq = lq + 32 * u * L::BYTES, *ud = ld + 32 * u * L::BYTES;
#pragma unroll
      for (int db = 0; db < NC; ++db) {
        const bf16x8 o = L::columns(ud, db, l16, g), q = L::columns(uq, db, l16, g);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          dv[r][db] = mfma32(o, pr[r], dv[r][db]);
          dk[r][db] = mfma32(q, ds[r], dk[r][db]);
        }
      }
    };
    const int q0 = now.j * kTile;
    if (DOC ? now.cls == TILE_FULL : !CAUSAL || q0 >= kw + 16 * R - 1 - p.causal_off) {
      scores(0);
      scores(1);  // (beside the arithmetic of the first half)
      probabilities(0);
      products(0);
      probabilities(1);
      products(1);
    } else if (!DOC || now.cls != TILE_SKIP) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint32_t w[R];
        bool any = !DOC && q0 + 32 * u + 31 >= kw - p.causal_off;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          w[r] = 0;
          if (DOC) {
            w[r] = static_cast<uint32_t>(words[16 * r] >> (32 * u));
            any = any || w[r] != 0;
            w[r] >>= 4 * g;
          }
        }
        if (__builtin_amdgcn_ballot_w64(any) == 0) continue;
        scores(u);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (DOC ? !(w[r] & (1u << (16 * v + i))) : q0 + 32 * u + 16 * v + 4 * g + i < kw + 16 * r + l16 - p.causal_off) s[u][r][v][i] = -INFINITY;
        probabilities(u);
        products(u);
      }
    }
    now = next, next = then, stage ^= 1;
  }

  const int64_t dk0 = b * bp.dks[0] + hkv * bp.dks[1] + 4 * g, dv0 = b * bp.dvs[0] + hkv * bp.dvs[1] + 4 * g;
  if constexpr (ROTATED) {  // (dk and dv in bf16, overwritten)
    const RotateBack rot = rotation_of_kernel<decltype(attn_bwd_dkv64_kernel<MODE, ROTATED>)>();
    // A quarter of a table row each for the lanes of a gradient row, on its way while dV is written; transposed it is every lane's own pairs.  8 x 8 heads x
    // 2048 causal, us: not rotated 96.7, so 99.2, fetched as the pairs are used (sixteen loads of 4 bytes) 103.8; the pass over dQ and dK took 14.9, of which dQ here keeps 3.9.
    uint32_t quarter[R][2][NC];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t table = rot.row(b, kw + 16 * r + l16);
      const auto lo = rot.angles<bf16_t, 4>(table, 8 * g), hi = rot.angles<bf16_t, 4>(table, 8 * g + 4);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const u32x2 c = __builtin_bit_cast(u32x2, (i ? hi : lo).c), sine = __builtin_bit_cast(u32x2, (i ? hi : lo).s);
#pragma unroll
        for (int e = 0; e < 2; ++e) quarter[r][0][2 * i + e] = c[e], quarter[r][1][2 * i + e] = sine[e];
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t row = kw + 16 * r + l16;
      if (row >= p.Sk) continue;
#pragma unroll
      for (int db = 0; db < NC; ++db) store4(bp.dv, dv0 + row * bp.dvs[2] + 16 * db, dv[r][db], 0);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t row = kw + 16 * r + l16;
      transpose_groups(quarter[r][0]), transpose_groups(quarter[r][1]);  // (all lanes)
      if (row >= p.Sk) continue;
#pragma unroll
      for (int db = 0; db < NC; ++db)
        store4(bp.dk, dk0 + row * bp.dks[2] + 16 * db,
               RotateBack::back<bf16_t>(dk[r][db] * p.scale, {__builtin_bit_cast(bf16x2, quarter[r][0][db]), __builtin_bit_cast(bf16x2, quarter[r][1][db])}), 0);
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = kw + 16 * r + l16;
    if (row >= p.Sk) continue;
    const int64_t dk_at = dk0 + row * bp.dks[2], dv_at = dv0 + row * bp.dvs[2];
    f32x4 old[2][NC];
#pragma unroll
    for (int db = 0; db < NC; ++db) old[0][db] = old[1][db] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (bp.accumulate_f32) {  // (all loads before the first store, which the compiler would not move them over)
#pragma unroll
      for (int db = 0; db < NC; ++db) {
        old[0][db] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(bp.dk) + dk_at + 16 * db);
        old[1][db] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(bp.dv) + dv_at + 16 * db);
      }
    }
#pragma unroll
    for (int db = 0; db < NC; ++db) {
      store4(bp.dk, dk_at + 16 * db, old[0][db] + dk[r][db] * p.scale, bp.accumulate_f32 ? 2 : 0);
      store4(bp.dv, dv_at + 16 * db, old[1][db] + dv[r][db], bp.accumulate_f32 ? 2 : 0);
    }
  }
}

template <int MODE>
int launch(const AttnBwdParams& bp, const float* lse2, hipStream_t st) {
  const AttnParams& p = bp.a;
  const int64_t blocks = static_cast<int64_t>((p.Sk + 64 * R - 1) / (64 * R)) * p.B * p.Hkv;
  MLTS_REQUIRE(blocks <= 0x7fffffffLL, "mlts_attn_bwd: too many workgroups");
  auto kern = bp.rot.cos ? attn_bwd_dkv64_kernel<MODE, true> : attn_bwd_dkv64_kernel<MODE, false>;
  MltsKernelTimer timer("attn_bwd_dkdv", st);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, bp, lse2, Dkv64Args{Divisor(p.Hkv), Divisor(p.B)});
  return mlts_check_launch("mlts_attn_bwd");
}

}  // namespace

// Grids that give every compute unit two workgroups and more; a wavefront alone on its SIMD waits too long, and the two-role kernel has two
// to the same keys.  us there -> here:
//   no mask   384 workgroups 3 x 8 heads x 2048 85 -> 74
//   causal    512            8 x 8 x 1024 38.1 -> 38.2, 32 x 2048 55 -> 57, 16 x 4096 103 -> 108, 8 x 16 (4) x 2048 195 -> 199
//             640            5 x 8 x 2048 75 -> 62
//             896            16 x 8 x 777 45.2 -> 40.1
//            1024            16 x 8 x 1024 66 -> 60, 16 x 16 (4) x 2048 377 -> 310; 32 x 8 x 512 45.2 -> 41.3
//   documents 384            3 x 8 x 2048 25.8 -> 27.0, 2 x 8 x 3072 39.6 -> 40.0
//             512            2 x 16 (4) x 8192 245 -> 244
//            1024            2 x 16 (8) x 8192 198 -> 133, 8 x 8 x 2048 81 -> 58
// Walks of less than 512 queries stay where one arithmetic serves all batch sizes.
bool mlts_attn_bwd_dkv64_serves(const AttnParams& p, int mode) {
  const int64_t blocks = static_cast<int64_t>((p.Sk + 64 * R - 1) / (64 * R)) * p.B * p.Hkv;
  return p.Sq >= 512 && blocks >= (mode == MLTS_MASK_NONE ? 384 : mode == MLTS_MASK_CAUSAL ? 640 : 512);
}

// lse2: B * Hq * Sq of them, as the dQ kernel writes them
int mlts_attn_bwd_dkv64(const AttnBwdParams& bp, int mode, const float* lse2, hipStream_t st) {
  if (mode == MLTS_MASK_NONE) return launch<MLTS_MASK_NONE>(bp, lse2, st);
  return mode == MLTS_MASK_CAUSAL ? launch<MLTS_MASK_CAUSAL>(bp, lse2, st) : launch<MLTS_MASK_DOC>(bp, lse2, st);
}
