// bf16 attention on v_mfma_f32_16x16x32_bf16: what attn_small.hip (head_dim 32, 64, 96 and 128) and attn_bwd_dkv64.hip (64) share.  Scores are computed
// transposed, walked rows x own rows: a lane then holds the probabilities of one own row and the next product takes them from the registers
// they are in, rounded to bf16 once (attn_small.hip at head_dim 32 and 96: in three parts).
#pragma once
#include "attn_rows.hpp"

namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));
#define MLTS_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Rows of an operand in LDS, read as fragments.  (16 bytes behind a row.  128-byte rows with permuted chunks, without the bank conflicts that
// are left here, changed nothing: the dK/dV kernel of head_dim 64 took 159 us at 8 x 8 heads x 2048 unmasked either way.)
template <int D>
struct Rows {
  static constexpr int BYTES = D * 2 + 16;  // of a row
  static __device__ __forceinline__ int at(int row, int chunk) { return row * BYTES + chunk * 16; }
  // rows 16 b + l16, columns 32 j + 8 g ..+7
  static __device__ __forceinline__ bf16x8 dot(const unsigned char* lds, int b, int j, int l16, int g) {
    return *reinterpret_cast<const bf16x8*>(lds + at(16 * b + l16, 4 * j + g));
  }
  // column 16 db + l16 of rows 4 g ..+3 and 16 + 4 g ..+3: in the order in which a lane holds scores
  static __device__ __forceinline__ bf16x8 columns(const unsigned char* lds, int db, int l16, int g) {
    const unsigned char* src = lds + at(4 * g + (l16 >> 2), 2 * db) + (l16 & 3) * 8;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src + 16 * BYTES));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

__device__ __forceinline__ bf16x8 pack(const f32x4 (&x)[2]) {
  bf16x8 v;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[4 * b + i] = static_cast<bf16_t>(x[b][i]);
  return v;
}

// mode 0: bf16, overwritten; 1: fp32, added to; 2: fp32, overwritten
__device__ __forceinline__ void store4(void* base, int64_t off, f32x4 v, int mode) {
  if (mode == 0) {
    bf16x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = static_cast<bf16_t>(v[e]);
    *reinterpret_cast<bf16x4*>(static_cast<bf16_t*>(base) + off) = w;
  } else {
    f32x4* p = reinterpret_cast<f32x4*>(static_cast<float*>(base) + off);
    *p = mode == 1 ? *p + v : v;
  }
}

}  // namespace
