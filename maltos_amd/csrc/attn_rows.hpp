// Attention kernels whose wavefronts own 16 rows (32) and walk the other side alone: the place of a wavefront in the launch, and what they
// share besides (attn_f32_*.hip, attn_small.hip).
#pragma once
#include "attn_common.hpp"

#include <algorithm>

namespace {

// e^x.  Scores, maxima and log-sum-exps stay in natural units and are subtracted first: what is rounded on the way into the hardware's
// 2^x is then a difference that is near 0 wherever the probability counts, and not a score (with the scores multiplied by log2 e
// before the subtraction the errors against 64 bits were up to 1.25 times as large).
__device__ __forceinline__ float exponential(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

// Over the four 16-lane groups: the lanes that share an own row.  (The swaps exchange the odd groups of one register with the even ones of
// the other; of a value with itself that leaves both halves of every pair side by side, without a way through LDS.)
__device__ __forceinline__ float sum_groups(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  x = __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) + __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  return __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) + __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}
__device__ __forceinline__ float max_groups(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  x = fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(r[0])), __builtin_bit_cast(float, static_cast<uint32_t>(r[1])));
  r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  return fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(r[0])), __builtin_bit_cast(float, static_cast<uint32_t>(r[1])));
}

// n / d for 0 <= n < 2^31 as (n * magic) >> shift: a division in the kernel takes 30 instructions, three of them as long as a load
struct Divisor {
  uint32_t d, magic, shift;
  explicit Divisor(int value) : d(static_cast<uint32_t>(value)) {
    uint32_t s = 0;
    while ((uint64_t{1} << s) < d) ++s;
    shift = 31 + s;
    magic = static_cast<uint32_t>(((uint64_t{1} << shift) + d - 1) / d);
  }
  __device__ __forceinline__ int over(int n, int* rest) const {
    const int q = static_cast<int>((static_cast<uint64_t>(static_cast<uint32_t>(n)) * magic) >> shift);
    *rest = n - q * static_cast<int>(d);
    return q;
  }
};

// A workgroup has a wavefront for every SIMD at least: with fewer splits, of several row blocks.  (Wavefronts of workgroups of one or
// two are not spread evenly over the SIMDs of a compute unit: dK/dV of 4 x 8 heads x 1024 keys, two wavefronts a SIMD, took 184 to 240 us.)
constexpr int kMinWaves = 4;

struct RowArgs {
  int D;
  bool vec_out;  // the outputs' rows are 16-byte aligned and D a multiple of 4
  Divisor heads, batch_heads, group;
  int tiles, half;  // row blocks of a head; those walked most work first, the others least work first
  int splits, blocks;
  RowArgs(const AttnParams& p, int head_dim, bool vec, int per_batch, int row_blocks)
      : D(head_dim), vec_out(vec), heads(per_batch), batch_heads(p.B * per_batch), group(p.Hq / p.Hkv), tiles(row_blocks), half(row_blocks), splits(1), blocks(0) {}
  // the row block at a place in the order (0: the one with most work under a causal mask)
  __device__ __forceinline__ int rank(int place) const { return place < half ? place : tiles - 1 - (place - half); }
};

// Which row block and which of its splits a wavefront is.
struct Place {
  int lane, l16, g, wave, splits, split, slot, block;  // slot: the block's place in the workgroup
  bool there;                                          // else it only keeps the barriers
  __device__ __forceinline__ explicit Place(const RowArgs& a) {
    lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), splits = a.splits, split = wave & (splits - 1);
    const int waves = static_cast<int>(blockDim.x) >> 6;
    slot = splits < kMinWaves ? wave >> (splits - 1) : 0;  // (one or two splits: shift by 0 or 1)
    block = splits < kMinWaves ? static_cast<int>(blockIdx.x) * (waves >> (splits - 1)) + slot : static_cast<int>(blockIdx.x);
    there = block < a.blocks;
    block = min(block, a.blocks - 1);
  }
};

// Wavefronts that run at once (two a SIMD: a wavefront takes up to 256 registers).  A grid that fits is all there from the start, and
// what shares a SIMD should be a long and a short row block: after half of the blocks the short ones come first.  In a larger one a
// compute unit that is done takes the next block, and the longest ones come first.
constexpr int64_t kResident = 2048;

// Wavefronts to a row block: until they fill the chip, with eight units each, or until half of it, with two.  Measured at 1, 2, 4, 8 (us,
// head_dim 64, causal): 2 x 8 heads x 777 (784 blocks, 25 units on the mean) forward 36 31 24 27, dQ 49 42 36 41; with four KV heads dK/dV
// (392 blocks, 49 units) 137 81 54 45; 8 x 4 x 256 (512 blocks, 8 units) forward 14.3 10.7 9.5 11.8, dQ 18.6 13.7 13.6 18.3, dK/dV 26 17 15
// 18; 4 x 8 x 1024 without a mask (2048 blocks) forward 87 - 97 99, dQ 127 - 148 151.
inline int splits_for(int64_t blocks, int64_t units, int most, int64_t fill = kResident) {
  int s = 1;
  while (s < most && ((blocks * s < fill && units >= 8 * s) || (blocks * s < kResident / 2 && units >= 2 * s))) s *= 2;
  return s;
}

// join: bytes of LDS in which a split's sums meet the others'; own: bytes of a wavefront's own LDS before that
template <auto KERN, int MOST, typename P>
int launch_splits(int64_t blocks, int splits, int join, int own, hipStream_t st, const P& params, RowArgs a, const char* what) {
  MLTS_REQUIRE(blocks <= 0x7fffffffLL, "%s: too many workgroups", what);
  static MltsLdsOptIn opt_in;
  if (blocks * splits <= kResident) a.half = (a.tiles + 1) / 2;
  auto bytes = [&](int s) { return std::max(s, kMinWaves) * std::max(s > 1 ? join : 0, own); };
  const int lds = bytes(splits), most = std::max(bytes(MOST), bytes(2));
  if (most > 48 * 1024) {
    if (hipError_t e = opt_in.reserve(reinterpret_cast<const void*>(KERN), most); e != hipSuccess) {
      mlts_set_error("%s: cannot reserve %d bytes of LDS: %s", what, most, hipGetErrorString(e));
      return MLTS_ERR_LAUNCH;
    }
  }
  a.splits = splits, a.blocks = static_cast<int>(blocks);
  const int waves = std::max(splits, kMinWaves), per = waves / splits;
  hipLaunchKernelGGL(KERN, dim3(static_cast<unsigned>((blocks + per - 1) / per)), dim3(waves * 64), lds, st, params, a);
  return mlts_check_launch(what);
}

// p.causal_off: the last key query i sees is i + causal_off; without a causal mask it is past every key
inline void set_causal_off(AttnParams& p, int mode) {
  if (mode != MLTS_MASK_CAUSAL) p.causal_off = p.Sk > p.Sq ? p.Sk : p.Sq;
}

}  // namespace
