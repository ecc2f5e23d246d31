// Matrix products of the linear layers: C = A B for row-major operands in the three forms a layer needs,
//   NT  y  = x W^T      A [M, K], B [N, K]     both contiguous along the contraction
//   NN  dx = dy W       A [M, K], B [K, N]
//   TN  dW = dy^T x     A [K, M], B [K, N]     optionally added onto C, the contraction split over workgroups
// in bf16 (v_mfma_f32_32x32x16_bf16) and fp32 (v_mfma_f32_32x32x2_f32, or the bf16 instruction on elements in three parts: Multiply).  fp32 accumulation, one
// rounding at the end.
//
// Why not the vendor library for these: through torch a product costs 18 us of host time whatever its size (a launch is 4), and
// for 1000-token micro-batches of 512-wide layers the library's kernels take 9-20 us where the work is 0.5-3 GFLOP.
//
// A workgroup computes a BM x BN tile of C.  A [BM][128 bytes] slab of A and of B travels global -> registers -> LDS, two LDS
// stages: while a slab is multiplied the next one is written to the other stage and the one after that is on its way from
// memory, with one barrier per slab.  Loads go through buffer descriptors, whose bounds check supplies the zeros past the end
// of an operand.  Rows along the contraction are padded by 16 bytes in LDS (16-byte fragment reads conflict free); rows along
// M or N by 64 (transpose reads, bf16) or 32 bytes (4-byte reads, fp32); those of parts are permuted instead, so that two tiles of 128 x 64 fit a CU.  The product is computed with the operands swapped, so
// that a lane holds four neighbouring columns of one row of C, and leaves through LDS in whole row segments.
#include "common.hpp"

#include <algorithm>

namespace {

constexpr int FORM_NT = MLTS_GEMM_NT, FORM_NN = MLTS_GEMM_NN, FORM_TN = MLTS_GEMM_TN;

typedef short i16x4 __attribute__((ext_vector_type(4)));
#define MLTS_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr uint32_t kOutside = 0x80000000u;  // an offset past every operand (operands are smaller than 2 GiB)

// How a tile multiplies.  bf16: as it is.  fp32 whole: by fp32 matrix instructions (true fp32 products and sums).  fp32 in three parts: every element is the sum of three
// bf16 values, 24 bits, and a product of two elements the sum of the six products of parts above 2^-24 of it, by bf16 matrix instructions with fp32 sums, which take 192 cycles for
// what the fp32 ones take 512.  The product of both first parts has a sum of its own, so that it is rounded once in sixteen terms.  Errors against 64 bits, in three parts / whole: N(0, 1)
// operands, 64 terms 0.5e-7 / 1.4e-7, 256 0.9e-7 / 2.9e-7, 2048 2.7e-7 / 8.1e-7, 8192 5.7e-7 / 16e-7; likewise with positive operands, operands of very different size, and small ones (1e-30).
enum { BF16, F32_WHOLE, F32_PARTS };
template <int KIND>
struct Multiply {
  typedef bf16x8 frag;
  static constexpr int STEP = 16;  // contraction elements of a fragment
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Multiply<F32_WHOLE> {
  typedef f32x4 frag;
  static constexpr int STEP = 8;
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], c, 0, 0, 0);
    return c;
  }
};
// Elements are split times 2^24 and the sums taken back by 2^-48: every fp32 number but zero is then a multiple of 2^-125, and so is each of its parts, which bf16 holds without denormal numbers.
// (Without it an element below 2^-110 loses bits of its third part and one below 2^-134 all of them, which a large enough other operand lifts into the result: 2.7e-4 relative
// at 1e-37 times 1e25, zero for 3e-41 times 1e20.)  Elements from 2^104 and sums from 2^80 on leave the range instead, and are computed whole one by one (gemm_tile).  us, without the scale / with it: NT 2048 x
// 256 x 256 5.93 / 5.92, 2048 x 768 x 256 11.0 / 11.7, 4096 x 2048 x 2048 178.5 / 180.8, TN 688 x 256 x 2048 13.9 / 14.5.
constexpr float kPartsScale = 0x1p24f, kPartsUnscale = 0x1p-48f;
// v times kPartsScale as its parts: their sum is that, unless it is infinite, NaN or rounded to infinity in bf16
__device__ __forceinline__ void split(f32x4 v, u32x2 (&parts)[3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    f32x2 rest = {v[2 * i] * kPartsScale, v[2 * i + 1] * kPartsScale};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t pair = parts[p][i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2));
      const float lo = __builtin_bit_cast(float, pair << 16), hi = __builtin_bit_cast(float, pair & 0xffff0000u);
      // (from v again: 180.8 us for 184.9 of the third product above, with the scaled elements kept)
      if (p == 0) rest[0] = __builtin_fmaf(v[2 * i], kPartsScale, -lo), rest[1] = __builtin_fmaf(v[2 * i + 1], kPartsScale, -hi);
      if (p == 1) rest[0] -= lo, rest[1] -= hi;
    }
  }
}

// One operand's slab: ROWS rows (of C's rows or columns), KC: the contraction is its contiguous dimension.  TWO: the upper half of the rows
// are those of a second matrix.
template <typename T, int KIND, int ROWS, bool KC, int THREADS, int SETS, bool TWO = false>
struct Slab {
  static constexpr int ES = static_cast<int>(sizeof(T));
  static constexpr int BK = 128 / ES;                          // contraction elements: 128 bytes
  static constexpr int PARTS = KIND == F32_PARTS ? 3 : 1, LS = KIND == F32_PARTS ? 2 : ES;  // LS: bytes of an element in LDS
  static constexpr int LINES = KC ? ROWS : BK;                 // lines in memory order
  static constexpr int PAD = PARTS > 1 ? 0 : KC ? 16 : ES == 2 ? 64 : 32;  // bytes behind a line in LDS
  static constexpr int STRIDE = (KC ? BK : ROWS) * LS + PAD;   // bytes of a line of a part in LDS
  static constexpr int PART_BYTES = LINES * STRIDE, BYTES = PARTS * PART_BYTES;
  static constexpr int CHUNKS = (KC ? BK : ROWS) * ES / 16;    // 16-byte chunks per line in memory
  static constexpr int PER = LINES * CHUNKS / THREADS;         // chunks per lane
  static_assert(LINES * CHUNKS % THREADS == 0, "whole chunks per lane");

  __amdgpu_buffer_rsrc_t rsrc, rsrc2;
  uint32_t offset[PER];
  uint32_t advance;
  u32x4 reg[SETS][PER];

  // Lines without padding: what the place of a byte in line i is changed by, so that the lines that are read together lie in different banks (a function of i % 16 for KC,
  // of i % 4 otherwise)
  static __device__ __forceinline__ int moved(int i) {
    if constexpr (PAD != 0) return 0;
    else if constexpr (KC) return (i >> 2 & 3) << 4;
    else return ROWS >= 128 ? (i & 3) << 6 : ROWS == 64 ? (i >> 1 & 1) << 6 : 0;
  }

  // base: first element of the slab's first row (KC) or column; ld: elements between lines; lines / line_elems: what exists
  __device__ __forceinline__ void init(const T* base, int64_t ld, int64_t lines, int64_t line_elems, int64_t k_begin) {
    const int64_t bytes = lines > 0 ? ((lines - 1) * ld + line_elems) * ES : 0;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, static_cast<int>(bytes), 0x00020000);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = i * THREADS + threadIdx.x - (second(i) ? LINES / 2 * CHUNKS : 0);
      const int64_t line = idx / CHUNKS + (KC ? 0 : k_begin);
      offset[i] = static_cast<uint32_t>((line * ld + (KC ? k_begin : 0)) * ES + (idx % CHUNKS) * 16);
    }
    advance = static_cast<uint32_t>(KC ? 128 : BK * ld * ES);
  }
  static __device__ __forceinline__ bool second(int i) {
    if constexpr (TWO && PER == 1) return __builtin_amdgcn_readfirstlane(threadIdx.x) >= THREADS / 2;
    return TWO && i >= PER / 2;
  }
  // of the second matrix, as many lines with the same stride
  __device__ __forceinline__ void init_second(const T* base, int64_t ld, int64_t lines, int64_t line_elems) {
    static_assert(!TWO || (KC && (PER == 1 || PER % 2 == 0)), "a wavefront's chunk is of one matrix");
    const int64_t bytes = lines > 0 ? ((lines - 1) * ld + line_elems) * ES : 0;
    rsrc2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, static_cast<int>(bytes), 0x00020000);
  }
  // chunk i of the slab at the current offsets; k_left: contraction elements from there to the end
  __device__ __forceinline__ void fetch(int set, int i, int k_left) {
    const int idx = i * THREADS + threadIdx.x;
    const int k = KC ? (idx % CHUNKS) * (16 / ES) : idx / CHUNKS;
    reg[set][i] = __builtin_amdgcn_raw_buffer_load_b128(second(i) ? rsrc2 : rsrc, k < k_left ? offset[i] : kOutside, 0, 0);
    offset[i] += advance;
  }
  __device__ __forceinline__ void store(int set, int i, unsigned char* lds) const {
    const int idx = i * THREADS + threadIdx.x;
    const int line = idx / CHUNKS;
    unsigned char* at = lds + line * STRIDE + ((idx % CHUNKS) * (16 / ES * LS) ^ moved(line));
    if constexpr (PARTS == 1) {
      *reinterpret_cast<u32x4*>(at) = reg[set][i];
    } else {
      u32x2 parts[3];
      split(__builtin_bit_cast(f32x4, reg[set][i]), parts);
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(at + p * PART_BYTES) = parts[p];
    }
  }
  // fragment of rows row0 .. row0 + 31 (of a part), contraction step ks; lane: row l % 32, contraction STEP * ks + (STEP / 2) * (l / 32) ..
  static __device__ __forceinline__ typename Multiply<KIND>::frag fragment(const unsigned char* lds, int row0, int ks, int lane) {
    const int l32 = lane & 31, hh = lane >> 5;
    if constexpr (KC) {
      return *reinterpret_cast<const typename Multiply<KIND>::frag*>(lds + (row0 + l32) * STRIDE + ((2 * ks + hh) * 16 ^ moved(l32)));
    } else if constexpr (LS == 2) {
      const int l16 = lane & 15;
      const unsigned char* src = lds + (16 * ks + 8 * hh + (l16 >> 2)) * STRIDE + ((row0 + (l32 >> 4) * 16 + (l16 & 3) * 4) * 2 ^ moved(l16 >> 2));
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

// The slabs of a 256 x 256 tile of bf16 in the TN form, eight wavefronts of 128 x 64: 32 contraction elements a stage, five stages, straight from memory to LDS: no
// registers hold them, so that three to four stages are on their way at any time (a slab of 64 in registers beside eight accumulator blocks: one), and there are no LDS
// writes through registers.  One barrier a stage.  Bound by the matrix pipes' clock under load (0.54 PFLOP in 448 us, where the largest products reach 1.21 PFLOP/s).
// us, slabs through registers / here: dW of 32000 x 512, 16384 rows 502 / 475, in a training step 502 (the library) / 448; 2752 x 512, 16384 rows 70 / 65; 2752 x 3072, 8192 rows 174 / 154; 70
// products 0.95 on the mean, 0.88 to 1.02.  Operands with the contraction contiguous have 64 bytes a line and stage, half a cache line: of 40 NT products half are slower, by up to
// 13 % (16384 x 1536 x 872 55.6 / 63.1), NN ones of long contractions by 3 to 5 % (12000 x 512 x 8192 112 / 116).
struct Ring {
  static constexpr int BK = 32, STAGES = 5, THREADS = 512, LINE = 256 * 2, OPERAND = BK * LINE, STAGE = 2 * OPERAND, BYTES = STAGES * STAGE, LOADS = 4;  // LOADS: of a lane a stage
  struct Operand {
    u32x4 rsrc;
    uint32_t offset[2], advance;
    int k[2];  // a chunk's contraction element in the stage
    // Chunks of 16 bytes lie in LDS in the order of the lanes that fetch them.  Which chunk of its line that is depends on the line, so that the four lines a fragment is read from
    // together lie in different banks.
    __device__ __forceinline__ void init(const bf16_t* base, int64_t ld, int64_t lines, int64_t line_elems, int64_t k_begin) {
      const uint64_t address = reinterpret_cast<uint64_t>(base);
      const int64_t bytes = lines > 0 ? ((lines - 1) * ld + line_elems) * 2 : 0;
      rsrc = u32x4{static_cast<uint32_t>(address), static_cast<uint32_t>(address >> 32) & 0xffff, static_cast<uint32_t>(bytes), 0x00020000};  // (as Slab's)
#pragma unroll
      for (int e = 0; e < 4; ++e) rsrc[e] = __builtin_amdgcn_readfirstlane(rsrc[e]);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int slot = i * THREADS + static_cast<int>(threadIdx.x), line = slot >> 5, chunk = (slot & 31) ^ ((line & 3) << 2);
        offset[i] = static_cast<uint32_t>((line + k_begin) * ld * 2 + chunk * 16);
        k[i] = line;
      }
      advance = static_cast<uint32_t>(BK * ld * 2);
    }
    // the next stage, to LDS address `to` (of the wavefront's first chunk); k_left: contraction elements from there to the end
    __device__ __forceinline__ void fetch(uint32_t to, int k_left) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t from = k[i] < k_left ? offset[i] : kOutside;
        // (through the builtin the compiler would wait for all loads before any read of LDS)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to + i * THREADS * 16), "v"(from), "s"(rsrc) : "memory", "m0");
#pragma clang diagnostic pop
        offset[i] += advance;
      }
    }
  };
  // as Slab::fragment
  static __device__ __forceinline__ bf16x8 fragment(const unsigned char* lds, int row0, int ks, int lane) {
    const int l32 = lane & 31, hh = lane >> 5, l16 = lane & 15;
    const unsigned char* src = lds + (16 * ks + 8 * hh + (l16 >> 2)) * LINE + ((row0 + (l32 >> 4) * 16 + (l16 & 3) * 4) * 2 ^ (l16 >> 2) << 6);
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MLTS_LDS_PTR(i16x4, src + 4 * LINE));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  // Of this wavefront all but the last N loads to LDS are there and nothing that it reads there is outstanding; then likewise of all wavefronts of the workgroup.  (Reads carried over
  // the barrier, which their slot allows: 475 -> 498 us; matrix instructions at a higher priority: no change.)
  template <int N>
  static __device__ __forceinline__ void wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

  // acc += the tile's product over k_left contraction elements
  static __device__ __forceinline__ void multiply(Operand a, Operand b, int k_left, unsigned char* lds, int wm, int wn, f32x16 (&acc)[4][2]) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const uint32_t own = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(MLTS_LDS_PTR(unsigned char, lds))) + wave * 1024);
    const int stages = (k_left + BK - 1) / BK;
    uint32_t to = 0;  // the stage that is written next
    auto fetch = [&] {  // (past the end: zeros)
      a.fetch(own + to, k_left), b.fetch(own + to + OPERAND, k_left);
      k_left -= BK;
      to = to + STAGE == BYTES ? 0 : to + STAGE;
    };
    bf16x8 fa[2][4], fb[2][2];
    auto read = [&](uint32_t stage, int ks) {
      const unsigned char* from = lds + stage;
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[ks][j] = fragment(from + OPERAND, wn + 32 * j, ks, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) fa[ks][i] = fragment(from, wm + 32 * i, ks, lane);
    };
    auto products = [&](int ks) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = Multiply<BF16>::mma(fb[ks][j], fa[ks][i], acc[i][j]);
    };
#pragma unroll
    for (int f = 0; f < STAGES - 1; ++f) fetch();
    wait<2 * LOADS>();
    uint32_t from = 0;
    read(from, 0);
    for (int s = 0; s < stages; ++s) {
      // here stages s and s + 1 are in LDS, s + 2 and s + 3 on their way, and s - 1 is read by nobody any more: s + 4 takes its place
      fetch();
      const uint32_t next = from + STAGE == BYTES ? 0 : from + STAGE;
      read(from, 1);
      __builtin_amdgcn_sched_barrier(0);
      products(0);
      __builtin_amdgcn_sched_barrier(0);
      read(next, 0);
      __builtin_amdgcn_sched_barrier(0);
      products(1);
      from = next;
      wait<2 * LOADS>();
    }
    wait<0>();  // (the zeros past the end)
  }
};

// One product of a launch, as small as can be: kernel arguments are read from host memory.  (Operands are smaller than 2 GiB, so
// their strides and lengths fit 32 bits.)
struct Product {
  const void *a, *b;
  void* c;
  float* partial;  // split contraction: [slices][M][N] fp32 in place of c
  int lda, ldb, ldc, K;
  int k_slice;     // contraction elements per slice (a multiple of the slab)
  int M, N;
  int tiles_m, tiles_n, slices;
  int form, accumulate;
  int xcds;  // log2 of the parts its slices, tile rows and tile columns are divided into for the eight XCDs, four bits each; kRuns: a run of its tiles each
};
constexpr int kMaxProducts = 4;  // of a call
constexpr int kRuns = -1;
// Two NT products of one shape that share A and meet in the end (gate and up of an MLP): C = A B^T, C2 = A B2^T, h = round(silu(C)) * C2 of
// the rounded C and C2; N, ldb and ldc are those of one of them.  C and C2 may be null.
struct Pair {
  const void* b2;
  void *c2, *h;
  int ldh;
  bool large;  // gate and up are kept, and h does not fit the L2s
};
// Rotary positions on the way out of an NT product whose rows are tokens and whose columns are heads: rounded x_even, x_odd become
// x_even cos - x_odd sin, x_even sin + x_odd cos with the roundings of the pass over them (mlts_rope).
struct Rotation {
  const void *cos, *sin;  // [max_pos][D / 2]
  const int32_t* positions;
  int max_pos, position_offset, seq, D;
  int columns[kMaxProducts][4];  // of each product: two ranges of whole heads
  // of row + step; in_seq: row's place in its sequence, for calls without positions
  template <typename T, typename C2>
  __device__ __forceinline__ void angles(int row, int step, int in_seq, int last, int pair, C2* c, C2* s) const {
    int pos;
    if (positions) {
      pos = positions[min(row + step, last)];
    } else {
      pos = in_seq + step;
      if (pos >= seq) pos = pos < 2 * seq ? pos - seq : static_cast<int>(static_cast<uint32_t>(pos) % static_cast<uint32_t>(seq));  // (a division takes 30 instructions)
      pos += position_offset;
    }
    pos = pos < 0 ? 0 : pos >= max_pos ? max_pos - 1 : pos;  // host validated; keeps reads in bounds
    const int64_t at = static_cast<int64_t>(pos) * (D / 2) + pair;
    *c = *reinterpret_cast<const C2*>(static_cast<const T*>(cos) + at), *s = *reinterpret_cast<const C2*>(static_cast<const T*>(sin) + at);
  }
};
template <typename T>
__device__ __forceinline__ void rotate(float& even, float& odd, float c, float s) {
#pragma clang fp contract(off)
  const float xe = round_to<T>(even), xo = round_to<T>(odd);
  even = round_to<T>(xe * c) - round_to<T>(xo * s);
  odd = round_to<T>(xe * s) + round_to<T>(xo * c);
}
// Buffer stores past the caches: of what is not read again before more than they hold was written.  Gate and up that are kept for a backward pass are (16384 x 2 x 688 x 384 48 -> 35 us,
// 8192 x 2 x 1376 x 512 46 -> 40, 4096 x 2 x 1024 x 256 14.1 -> 12.9), also where the last-level cache would hold them until then (the training step of the 50M model from a graph, gate and up cached /
// past the caches: 512 tokens 1421 / 1421, 1023 1761 / 1751, 2046 2329 / 2317, 3000 2863 / 2853, 4092 3326 / 3305, 6000 4485 / 4425, 8192 5601 / 5548, 16384 8870 / 8783); so is h beside them where it exceeds the 32 MB of the eight L2s (16384 x 2 x 1376 x 512 94 -> 92 without it,
// -> 74; a training step of 16384 tokens of the 50M model 8777 -> 8674, of 4000 tokens 3201 -> 3188).  Below that, and where gate and up are not kept, the product behind reads h out of the
// caches (evaluation of 2331 tokens with h past them 617 -> 649).  No gain, or a loss, in steps: the rotated q, k, v, dense C, d gate and d up likewise, gate and up read so.
constexpr int kNontemporal = 2;
// Where a tile's rows are read and written four columns at a time: the bounds check of a buffer descriptor stands for a branch over the rows and
// columns past the end at every access, which all passes of a tile would wait behind.  (Rows too far apart for the descriptor's 32-bit
// offsets: pointers.)
template <typename T>
struct Window {
  typedef T t4 __attribute__((ext_vector_type(4)));
  static constexpr int ES = static_cast<int>(sizeof(T));
  __amdgpu_buffer_rsrc_t rsrc;
  T* at;  // of this lane's first row and column
  int64_t ld;
  uint32_t offset;
  int rows;   // that exist, from this lane's first one on
  bool near;
  // base: the tile's first row; rows: of the tile that exist; row, col: this lane's first row in the tile and its column of `columns`
  template <int BM>
  __device__ __forceinline__ void init(const void* base, int64_t stride, int tile_rows, int columns, int row, int col) {
    ld = stride, near = stride < (int64_t{1} << 31) / (BM * ES);
    const int existing = min(tile_rows, BM);
    const uint32_t bytes = near ? static_cast<uint32_t>(((existing - 1) * ld + columns) * ES) : 0;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
    offset = col < columns ? static_cast<uint32_t>(row * static_cast<uint32_t>(stride) + col) * ES : kOutside;
    at = static_cast<T*>(const_cast<void*>(base)) + row * ld + col;
    rows = col < columns ? existing - row : 0;
  }
  template <int POLICY = 0>
  __device__ __forceinline__ void put(int row, t4 v) const {
    if (near) {
      if constexpr (ES == 2) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc, offset + row * static_cast<uint32_t>(ld * ES), 0, POLICY);
      else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, offset + row * static_cast<uint32_t>(ld * ES), 0, POLICY);
    } else if (row < rows) {
      *reinterpret_cast<t4*>(at + row * ld) = v;
    }
  }
  __device__ __forceinline__ t4 get(int row) const {
    if (near) {
      if constexpr (ES == 2) return __builtin_bit_cast(t4, __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset + row * static_cast<uint32_t>(ld * ES), 0, 0));
      else return __builtin_bit_cast(t4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset + row * static_cast<uint32_t>(ld * ES), 0, 0));
    }
    return row < rows ? *reinterpret_cast<const t4*>(at + row * ld) : t4{};
  }
};
// What becomes of dh = dy W_down, an NN product, instead of being written: d gate and d up of the activation (mlts_swiglu_bwd_rows of the
// rounded dh).  Strides in elements.
struct Activation {
  const void *gate, *up;
  void *dgate, *dup;
  int ld_in, ld_out;
};
// The contraction of the NN form may be a concatenation (dx = sum dy_i W_i of layers that share their input): what follows the
// first part.  In bf16 each part is rounded, and added to the parts before it in bf16: the values of separate products whose
// results are added, bit for bit.
constexpr int kMaxSegments = 3;
struct MoreSegments {
  const void *a[kMaxSegments - 1], *b[kMaxSegments - 1];
  int lda[kMaxSegments - 1], ldb[kMaxSegments - 1], K[kMaxSegments - 1];
  int count, product;  // how many, of which product
};

// The tile of a workgroup.  Consecutive workgroups go to the eight XCDs in turn, each with an L2 of its own: an XCD gets a rectangle of a
// product's tiles (split contractions: of some of the slices), so that it reads few rows of A and few columns of B, or a run of them (spread()), and walks
// them along N.
struct Tile {
  int slice, m, n;
  bool there;
  __device__ __forceinline__ Tile(const Product& g, int block) {
    const int xcd = block & 7;
    int rest = block >> 3, n0 = 0, m0 = 0, s0 = 0, width = g.tiles_n, height = g.tiles_m, depth = g.slices;
    if (g.xcds == kRuns) {
      const int tiles = width * height * depth, per = tiles >> 3, more = tiles & 7;
      there = rest < per + (xcd < more);
      rest += xcd * per + min(xcd, more);
    } else {
      const int ls = g.xcds & 15, lm = (g.xcds >> 4) & 15, ln = g.xcds >> 8;
      const int xn = xcd & ((1 << ln) - 1), xm = (xcd >> ln) & ((1 << lm) - 1), xs = xcd >> (ln + lm);
      n0 = (g.tiles_n * xn) >> ln, width = ((g.tiles_n * (xn + 1)) >> ln) - n0;
      m0 = (g.tiles_m * xm) >> lm, height = ((g.tiles_m * (xm + 1)) >> lm) - m0;
      s0 = (g.slices * xs) >> ls, depth = ((g.slices * (xs + 1)) >> ls) - s0;
      there = rest < width * height * depth;
    }
    const int row = there ? rest / width : 0;
    n = n0 + rest - row * width;
    slice = depth > 1 ? row / height : 0;
    m = m0 + row - slice * height, slice += s0;
  }
};

template <typename T, int FORM, int BM, int BN, int WM, int WN, int KG, bool PAIR = false>
struct TileShape {
  static constexpr int WAVES_N = BN / WN, WAVES = (BM / WM) * WAVES_N * KG, THREADS = WAVES * 64;
  static constexpr int MB = WM / 32, NB = WN / 32;
  static constexpr bool SHARED = KG > 1 && WAVES == KG, GROUPS = KG > 1 && WAVES > KG;  // one wavefront to a group; several
  static constexpr int KIND = sizeof(T) == 2 ? BF16 : SHARED ? F32_WHOLE : F32_PARTS;  // (in a tile of 32 x 32 the parts are more work than they save)
  static constexpr bool RING = KIND == BF16 && BM == 256 && BN == 256 && FORM == FORM_TN;  // (Ring)
  static constexpr int SETS = MB * NB >= 8 ? 1 : 2;  // (eight accumulator blocks leave no registers for a second set)
  typedef Slab<T, KIND, BM, FORM != FORM_TN, THREADS, SETS> SA;
  typedef Slab<T, KIND, BN, FORM == FORM_NT, THREADS, SETS, PAIR> SB;
  static constexpr int STAGE = SA::BYTES + SB::BYTES;
  static constexpr int OUT = WAVES / (GROUPS ? KG : 1) * 32 * (WN + 4) * 4;
  static_assert(!GROUPS || (KG - 1) * BM * BN * 4 <= 2 * STAGE, "the groups' sums meet where the slabs were");
  static_assert(!PAIR || (FORM == FORM_NT && !SHARED && WAVES_N % 2 == 0), "the products of a pair side by side in a tile, half of the wavefronts each");
  static constexpr int SLABS = RING ? Ring::BYTES : 2 * STAGE;
  static constexpr int LDS = SLABS > OUT ? SLABS : OUT;
};

// One tile of one product.  KG > 1, SHARED: the wavefronts share the tile and each multiply their part of every slab; their sums meet in
// LDS, where all of them add up and write out a part of the tile (us, one of them / all: fp32 NT 2048 x 256 x 256 7.2 / 6.7,
// 500 x 512 x 512 8.0 / 7.0).  GROUPS: KG groups of wavefronts each multiply their part of every slab (64 x 64 of parts, one / two: NT 2048 x 256 x 688 14.5 / 12.3, TN 1376 x 256 x 2048
// whole 36 / 30; four or eight tiles to a CU the same).
template <typename T, int FORM, int BM, int BN, int WM, int WN, int KG, bool SEGMENTS, bool PAIR = false, bool ROPE = false, bool ACT = false>
__device__ __forceinline__ void gemm_tile(const Product& g, const Tile& tile, unsigned char* lds, const MoreSegments& more, int segs, const Pair* pair = nullptr,
                                          const Rotation* rot = nullptr, int product = 0, const Activation* act = nullptr) {
  typedef TileShape<T, FORM, BM, BN, WM, WN, KG, PAIR> S;
  constexpr int WAVES_N = S::WAVES_N, MB = S::MB, NB = S::NB, SETS = S::SETS, STAGE = S::STAGE;
  typedef typename S::SA SA;
  typedef typename S::SB SB;
  typedef Multiply<S::KIND> Mul;
  constexpr int BK = SA::BK, PARTS = SA::PARTS, STEPS = BK / Mul::STEP / KG;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int MEMBERS = S::WAVES / KG;  // wavefronts of a group
  constexpr bool SHARED = S::SHARED, GROUPS = S::GROUPS;
  const int group = wave / MEMBERS, member = wave % MEMBERS;
  const int wm = (member / WAVES_N) * WM, wn = (member % WAVES_N) * WN;
  const int slice = tile.slice, m0 = tile.m * BM, n0 = tile.n * (PAIR ? BN / 2 : BN);

  SA sa;
  SB sb;
  int k_left = 0;                  // contraction elements of the segment behind the slab that is fetched next
  int seg = 0, seg_slabs = 0;      // segments opened after the first, slabs of the open one that are not fetched yet
  auto open = [&](const void* a, int64_t lda, const void* b, int64_t ldb, int64_t K, int64_t k_begin, int64_t k_end) {
    if (FORM == FORM_TN) sa.init(static_cast<const T*>(a) + m0, lda, K, g.M - m0, k_begin);
    else sa.init(static_cast<const T*>(a) + m0 * lda, lda, g.M - m0, K, k_begin);
    if (FORM == FORM_NT) sb.init(static_cast<const T*>(b) + n0 * ldb, ldb, g.N - n0, K, k_begin);
    else sb.init(static_cast<const T*>(b) + n0, ldb, K, g.N - n0, k_begin);
    if constexpr (PAIR) sb.init_second(static_cast<const T*>(pair->b2) + n0 * ldb, ldb, g.N - n0, K);
    k_left = static_cast<int>(k_end - k_begin);
    seg_slabs = (k_left + BK - 1) / BK;
  };
  const int k_begin = slice * g.k_slice;
  int slabs;
  if constexpr (SEGMENTS) {  // a slice is a run of the slabs of all segments
    int skip = k_begin / BK, left = (g.K + BK - 1) / BK;
    slabs = left - skip;
    for (int i = 0; i < segs; ++i) {
      const int more_slabs = (more.K[i] + BK - 1) / BK;
      slabs += more_slabs;
      if (seg == i && skip >= left) skip -= left, left = more_slabs, ++seg;
    }
    slabs = min(slabs, g.k_slice / BK);
    if (seg == 0) open(g.a, g.lda, g.b, g.ldb, g.K, skip * BK, g.K);
    else open(more.a[seg - 1], more.lda[seg - 1], more.b[seg - 1], more.ldb[seg - 1], more.K[seg - 1], skip * BK, more.K[seg - 1]);
  } else {
    open(g.a, g.lda, g.b, g.ldb, g.K, k_begin, min(g.K, k_begin + g.k_slice));
    slabs = seg_slabs;
  }
  auto next_slab = [&] {  // before the first chunk of a slab is fetched
    if constexpr (SEGMENTS) {
      while (seg_slabs == 0 && seg < segs) {
        open(more.a[seg], more.lda[seg], more.b[seg], more.ldb[seg], more.K[seg], 0, more.K[seg]);
        ++seg;
      }
      --seg_slabs;
    }
  };

  f32x16 acc[MB][NB], low[PARTS > 1 ? MB : 1][PARTS > 1 ? NB : 1];  // low: the products of all but both first parts
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f, low[PARTS > 1 ? i : 0][PARTS > 1 ? j : 0][e] = 0.f;

  // One slab ahead in LDS, the next SETS in registers: chunk c of slab s + 1 goes to the other stage and its registers fetch
  // chunk c of slab s + 1 + SETS, spread behind the products of the fragment steps.  (Past the end: zeros, never multiplied.)
  // With one set a load has the time of one slab to arrive, which short contractions out of HBM exceed; more than two sets
  // bring nothing (1024 x 512 x 512: 5.2 us with 2, 4, 5.5 with 6).
  constexpr int CHUNKS = SA::PER + SB::PER;
  auto store = [&](int set, int c, unsigned char* stage) {
    if (c < SA::PER) sa.store(set, c, stage);
    else sb.store(set, c - SA::PER, stage + SA::BYTES);
  };
  auto fetch = [&](int set, int c) {
    if (c < SA::PER) sa.fetch(set, c, k_left);
    else sb.fetch(set, c - SA::PER, k_left);
  };
#pragma unroll
  for (int f = 0; f < (S::RING ? 0 : SETS); ++f) {
    next_slab();
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) fetch(f, c);
    k_left -= BK;
  }
  // What the result is added to, for small tiles: fetched here, behind the first slabs, where the end of the tile would wait for
  // it (a gradient that was last touched a step ago; dW and dx of a 512-wide layer at 1023 tokens: four launches a layer, 40 us
  // of a training step of 8 layers).
  constexpr int OUT_LANES = SHARED ? S::THREADS : 64;  // that write a block of 32 rows of C
  constexpr int LPR = WN / 4, RPP = OUT_LANES / LPR, PASSES = 32 / RPP;  // out: lanes per row, four columns each, rows per pass
  constexpr bool EARLY = !PAIR && !ROPE && !ACT && (SHARED || MB * NB <= 2);
  typedef T t4 __attribute__((ext_vector_type(4)));
  t4 old[EARLY ? MB * PASSES : 1];
  constexpr int HALF = WAVES_N / 2;  // PAIR: wavefronts of a row of blocks that have the first product; HALF further on is the second one of the same columns
  const int out_lane = SHARED ? tid : lane, c4 = (out_lane % LPR) * 4, col = n0 + (PAIR ? wn % (BN / 2) : wn) + c4;
  const int tile_row = wm + out_lane / LPR, out_row = m0 + tile_row, rows_here = g.M - m0;  // out_row: of pass 0 of the first block
  const bool vec = PAIR || ACT || ROPE || ((g.N & 3) == 0 && (g.ldc & 3) == 0);
  Window<T> out;
  if (!ACT) out.template init<BM>(static_cast<const T*>(g.c) + m0 * static_cast<int64_t>(g.ldc), g.ldc, rows_here, g.N, tile_row, col);
  const bool add = !PAIR && !ROPE && !ACT && g.accumulate && !g.partial;
  auto fetch_old = [&] {
    if (EARLY && add && vec) {
#pragma unroll
      for (int i = 0; i < (EARLY ? MB * PASSES : 0); ++i) old[i] = out.get(i * RPP);
    }
  };
  // ... and the activation's operands, and what it is rotated by, likewise.  Larger tiles fetch the activation's operands, and the old C, behind
  // the last slab, where the registers of the slabs are free.
  constexpr bool SMALL = MB * NB == 1;
  t4 gates[ACT ? MB * PASSES : 1], ups[ACT ? MB * PASSES : 1];
  auto fetch_gates = [&] {
    if constexpr (ACT) {
      Window<T> gate, up;
      gate.template init<BM>(static_cast<const T*>(act->gate) + m0 * static_cast<int64_t>(act->ld_in), act->ld_in, rows_here, g.N, tile_row, col);
      up.template init<BM>(static_cast<const T*>(act->up) + m0 * static_cast<int64_t>(act->ld_in), act->ld_in, rows_here, g.N, tile_row, col);
#pragma unroll
      for (int r = 0; r < MB * PASSES; ++r) gates[r] = gate.get(r * RPP), ups[r] = up.get(r * RPP);
    }
  };
  if (SMALL) fetch_old(), fetch_gates();
  typedef T t2 __attribute__((ext_vector_type(2)));
  constexpr bool EARLY_ANGLES = SMALL, ALL_ANGLES = MB * NB <= 4;  // (the largest tiles: a block of rows at a time)
  constexpr int ANGLES = (ALL_ANGLES ? MB : 1) * PASSES;
  t2 cosines[ROPE ? ANGLES : 1], sines[ROPE ? ANGLES : 1];
  bool rotated = false;
  int pair_of_head = 0, in_seq = 0;
  auto fetch_angles = [&](int i) {
    if constexpr (ROPE) {
      if (rotated) {
#pragma unroll
        for (int r = 0; r < ANGLES; ++r) rot->angles<T>(out_row, 32 * i + r * RPP, in_seq, g.M - 1, pair_of_head, &cosines[r], &sines[r]);
      }
    }
  };
  if constexpr (ROPE) {
    const int* range = rot->columns[product];
    rotated = (col >= range[0] && col < range[1]) || (col >= range[2] && col < range[3]);
    pair_of_head = static_cast<int>(static_cast<uint32_t>(col - (col >= range[2] && col < range[3] ? range[2] : range[0])) % static_cast<uint32_t>(rot->D)) / 2;
    if (!rot->positions) in_seq = static_cast<int>(static_cast<uint32_t>(out_row) % static_cast<uint32_t>(rot->seq));
    if (EARLY_ANGLES) fetch_angles(0);
  }
  if constexpr (!S::RING) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) store(0, c, lds);
    next_slab();
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) fetch(0, c);
  }
  constexpr bool FOLD = SEGMENTS && sizeof(T) == 2;
  f32x16 parts[FOLD ? MB : 1][FOLD ? NB : 1];  // sum of the parts before
  int part = 0, part_end = FOLD ? (g.K + BK - 1) / BK : 0;
  auto fold = [&] {
    if constexpr (FOLD) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float v = to_f32<T>(from_f32<T>(acc[i][j][e]));
            parts[i][j][e] = part == 0 ? v : to_f32<T>(from_f32<T>(parts[i][j][e] + v));
            acc[i][j][e] = 0.f;
          }
    }
  };
  auto slab = [&](int s, int set) {  // set: registers of slab s + 1
    k_left -= BK;
    next_slab();
    __syncthreads();  // stage s & 1 is written everywhere, and nobody reads the other one any more
    const unsigned char* la = lds + (s & 1) * STAGE;
    const unsigned char* lb = la + SA::BYTES;
    unsigned char* next = lds + (~s & 1) * STAGE;
    typename Mul::frag fa[2][MB][PARTS], fb[2][NB][PARTS];  // (reading the whole slab's first instead changes nothing)
    auto read = [&](int ks) {
#pragma unroll
      for (int p = PARTS - 1; p >= 0; --p) {
#pragma unroll
        for (int j = 0; j < NB; ++j) fb[ks & 1][j][p] = SB::fragment(lb + p * SB::PART_BYTES, wn + 32 * j, group * STEPS + ks, lane);
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[ks & 1][i][p] = SA::fragment(la + p * SA::PART_BYTES, wm + 32 * i, group * STEPS + ks, lane);
      }
    };
    read(0);
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks) {
      if (ks + 1 < STEPS) read(ks + 1);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          if constexpr (PARTS > 1) {
#pragma unroll
            for (int sum = 2; sum > 0; --sum)  // smallest products first; those of 2^-24 and less are left out
#pragma unroll
              for (int p = 0; p <= sum; ++p) low[i][j] = Mul::mma(fb[ks & 1][j][p], fa[ks & 1][i][sum - p], low[i][j]);
          }
          acc[i][j] = Mul::mma(fb[ks & 1][j][0], fa[ks & 1][i][0], acc[i][j]);
        }
#pragma unroll
      for (int c = ks * CHUNKS / STEPS; c < (ks + 1) * CHUNKS / STEPS; ++c) {
        store(set, c, next);
        fetch(set, c);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto after = [&](int s) {  // slab s was multiplied: the last of its part?
    if constexpr (FOLD)
      while (part < segs && s + 1 == part_end) {
        fold();
        part_end += (more.K[part++] + BK - 1) / BK;
      }
  };
  if constexpr (FOLD) after(-1);
  if constexpr (S::RING) {
    Ring::Operand a, b;
    a.init(static_cast<const bf16_t*>(g.a) + m0, g.lda, g.K, g.M - m0, k_begin);
    b.init(static_cast<const bf16_t*>(g.b) + n0, g.ldb, g.K, g.N - n0, k_begin);
    Ring::multiply(a, b, k_left, lds, wm, wn, acc);
  } else if constexpr (SETS == 1) {
    for (int s = 0; s < slabs; ++s) slab(s, 0);
  } else {
    // (Whole rounds of the sets with nothing to jump over: a way round one slab of a round leaves fewer loads behind, and the waits
    // of the next round are set for that way.  1023 x 512 x 512 6.4 -> 5.7 us, x 1376 11.8 -> 10.2 us with weights out of HBM.)
    int s = 0;
    for (; s + SETS <= slabs; s += SETS) {
#pragma unroll
      for (int u = 0; u < SETS; ++u) {
        slab(s + u, (u + 1) % SETS);
        after(s + u);
      }
    }
#pragma unroll
    for (int u = 0; u < SETS - 1; ++u) {
      if (s + u < slabs) {
        slab(s + u, (u + 1) % SETS);
        after(s + u);
      }
    }
  }
  if constexpr (FOLD) {
    if (segs > 0) {
      fold();
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = parts[i][j];
    }
  }

  if constexpr (PARTS > 1) {
    float finite = 0.f;  // NaN if a sum is not
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[i][j] = (acc[i][j] + low[i][j]) * kPartsUnscale;
#pragma unroll
        for (int e = 0; e < 16; ++e) finite = __builtin_fmaf(acc[i][j][e], 0.f, finite);
      }
    if (__builtin_amdgcn_ballot_w64(finite != 0.f)) {
      // Infinities, NaN, and numbers that leave the range of the scaled parts or of their sums: blocks of this wavefront that have such elements once more, by fp32 matrix instructions straight
      // from memory (us, 4096 x 2048 x 2048: 183, with a row of NaN 335, all NaN 1908; elements of 1e-36 192).  The others of a block stay as they are, so that an element's bits depend on its own row and column alone; and what lies beside the operands in
      // memory, which lanes past the last row or column may hold, is no reason.
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int row = m0 + wm + 32 * i + l32, block = wn + 32 * j, in_pair = block % (BN / 2);
          const bool second = PAIR && block >= BN / 2;
          const int column = n0 + (PAIR ? in_pair : block) + l32;
          const auto in_range = [&](int e) { return __builtin_fabsf(acc[i][j][e]) < INFINITY; };
          bool all = true;
#pragma unroll
          for (int e = 0; e < 16; ++e) all = all && (in_range(e) || row >= g.M || column - l32 + 8 * (e / 4) + 4 * hh + e % 4 >= g.N);
          if (!__builtin_amdgcn_ballot_w64(!all)) continue;
          f32x16 sum;
#pragma unroll
          for (int e = 0; e < 16; ++e) sum[e] = 0.f;
          for (int part = 0, before = 0; part <= (SEGMENTS ? segs : 0); ++part) {
            const float* a = static_cast<const float*>(part ? more.a[part - 1] : g.a);
            const float* b = static_cast<const float*>(part ? more.b[part - 1] : second ? pair->b2 : g.b);
            const int64_t lda = part ? more.lda[part - 1] : g.lda, ldb = part ? more.ldb[part - 1] : g.ldb;
            const int K = part ? more.K[part - 1] : g.K, from = max(0, k_begin - before), to = min(K, k_begin + g.k_slice - before);
            before += (K + BK - 1) / BK * BK;
            for (int k0 = from; k0 < to; k0 += 8) {
              if (GROUPS && (k0 - from) / Mul::STEP % KG != group) continue;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int k = k0 + 4 * hh + e;
                const float x = row < g.M && k < to ? a[FORM == FORM_TN ? k * lda + row : row * lda + k] : 0.f;
                const float y = column < g.N && k < to ? b[FORM == FORM_NT ? column * ldb + k : k * ldb + column] : 0.f;
                sum = __builtin_amdgcn_mfma_f32_32x32x2f32(y, x, sum, 0, 0, 0);
              }
            }
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = in_range(e) ? acc[i][j][e] : sum[e];
        }
    }
  }

  if constexpr (GROUPS) {  // the first group takes the others' sums, and writes the tile
    static_assert(MB * NB == 1);
    f32x4* sums = reinterpret_cast<f32x4*>(lds) + member * 256 + lane;
    __syncthreads();
    if (group > 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) sums[(group - 1) * MEMBERS * 256 + q * 64] = f32x4{acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2], acc[0][0][4 * q + 3]};
    }
    __syncthreads();
    if (group > 0) return;  // (a barrier waits for the wavefronts that are left)
#pragma unroll
    for (int o = 0; o < KG - 1; ++o)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = sums[o * MEMBERS * 256 + q * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0][0][4 * q + e] += v[e];
      }
  }

  if (!SMALL) fetch_old(), fetch_gates();
  if (!EARLY_ANGLES && ALL_ANGLES) fetch_angles(0);
  Window<T> out2, out_h;
  if constexpr (PAIR) {
    out2.template init<BM>(static_cast<T*>(pair->c2) + m0 * static_cast<int64_t>(g.ldc), g.ldc, rows_here, g.N, tile_row, col);
    out_h.template init<BM>(static_cast<T*>(pair->h) + m0 * static_cast<int64_t>(pair->ldh), pair->ldh, rows_here, g.N, tile_row, col);
  }
  if constexpr (ACT) {
    out.template init<BM>(static_cast<T*>(act->dgate) + m0 * static_cast<int64_t>(act->ld_out), act->ld_out, rows_here, g.N, tile_row, col);
    out2.template init<BM>(static_cast<T*>(act->dup) + m0 * static_cast<int64_t>(act->ld_out), act->ld_out, rows_here, g.N, tile_row, col);
  }
  Window<float> sums;
  if (!PAIR && !ROPE && !ACT && g.partial) sums.template init<BM>(g.partial + (static_cast<int64_t>(slice) * g.M + m0) * g.N, g.N, rows_here, g.N, tile_row, col);
  // acc[i][j][4 q + r]: row wm + 32 i + l % 32 of C, column wn + 32 j + 8 q + 4 hh + r.  Out through LDS, 32 rows at a time.
  __syncthreads();
  constexpr int ROW = WN + 4;  // floats
  float* stage = reinterpret_cast<float*>(lds) + (SHARED ? 0 : wave * 32 * ROW);
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if ((SHARED || PAIR) && i > 0) __syncthreads();
    if (!ALL_ANGLES) fetch_angles(i);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        *reinterpret_cast<f32x4*>(stage + ((SHARED ? group : 0) * 32 + l32) * ROW + 32 * j + 8 * q + 4 * hh) = v;
      }
    if (SHARED || PAIR) __syncthreads();  // (alone, a wavefront reads only what it wrote: LDS operations of a wavefront complete in order)
    if constexpr (PAIR) {  // the two wavefronts of a pair of blocks take half of the rows each
      const int second = wave % WAVES_N / HALF;
      const float* first = reinterpret_cast<const float*>(lds) + (wave - second * HALF) * 32 * ROW;
#pragma unroll
      for (int r = 0; r < PASSES / 2; ++r) {
        const int rr = second * 16 + r * RPP, at = (rr + lane / LPR) * ROW + c4;
        const f32x4 a = *reinterpret_cast<const f32x4*>(first + at), b = *reinterpret_cast<const f32x4*>(first + HALF * 32 * ROW + at);
        t4 gate, up, h;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          gate[e] = from_f32<T>(a[e]), up[e] = from_f32<T>(b[e]);
          h[e] = from_f32<T>(round_to<T>(silu(to_f32<T>(gate[e]))) * to_f32<T>(up[e]));
        }
        if (g.c) out.template put<kNontemporal>(32 * i + rr, gate), out2.template put<kNontemporal>(32 * i + rr, up);
        if (pair->large) out_h.template put<kNontemporal>(32 * i + rr, h);
        else out_h.put(32 * i + rr, h);
      }
      continue;
    }
#pragma unroll
    for (int r = 0; r < PASSES; ++r) {
      const int at = (r * RPP + out_lane / LPR) * ROW + c4, row = 32 * i + r * RPP;
      f32x4 v = *reinterpret_cast<const f32x4*>(stage + at);
#pragma unroll
      for (int o = 1; o < (SHARED ? KG : 1); ++o) v += *reinterpret_cast<const f32x4*>(stage + o * 32 * ROW + at);
      if constexpr (ACT) {
        t4 dgate, dup;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float dg, du;
          swiglu_grads(round_to<T>(v[e]), to_f32<T>(gates[ACT ? i * PASSES + r : 0][e]), to_f32<T>(ups[ACT ? i * PASSES + r : 0][e]), &dg, &du);
          dgate[e] = from_f32<T>(dg), dup[e] = from_f32<T>(du);
        }
        out.put(row, dgate), out2.put(row, dup);
        continue;
      }
      if constexpr (ROPE) {
        if (__builtin_amdgcn_ballot_w64(rotated)) {
          const t2 c = cosines[ROPE ? (i * PASSES + r) % ANGLES : 0], s = sines[ROPE ? (i * PASSES + r) % ANGLES : 0];
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            float even = v[e], odd = v[e + 1];
            rotate<T>(even, odd, to_f32<T>(c[e / 2]), to_f32<T>(s[e / 2]));
            v[e] = rotated ? even : v[e], v[e + 1] = rotated ? odd : v[e + 1];
          }
        }
      }
      if (!ROPE && g.partial) {
        if ((g.N & 3) == 0) {
          sums.put(row, v);
        } else if (row + tile_row < rows_here) {
          float* p = g.partial + (static_cast<int64_t>(slice) * g.M + out_row + row) * g.N + col;
          for (int e = 0; e < 4 && col + e < g.N; ++e) p[e] = v[e];
        }
        continue;
      }
      if (vec) {
        if (add) {
          const t4 before = EARLY ? old[EARLY ? i * PASSES + r : 0] : out.get(row);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += to_f32<T>(before[e]);
        }
        t4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(v[e]);
        out.put(row, w);
      } else if (row + tile_row < rows_here) {  // (columns that are not whole groups of four)
        T* p = static_cast<T*>(g.c) + static_cast<int64_t>(out_row + row) * g.ldc + col;
        if (col + 4 <= g.N && (g.ldc & 3) == 0) {
          t4 w;
          const t4 before = add ? *reinterpret_cast<const t4*>(p) : t4{};
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(add ? v[e] + to_f32<T>(before[e]) : v[e]);
          *reinterpret_cast<t4*>(p) = w;
        } else {
          for (int e = 0; e < 4 && col + e < g.N; ++e) p[e] = from_f32<T>(v[e] + (add ? to_f32<T>(p[e]) : 0.f));
        }
      }
    }
  }
}

template <typename T, int FORM, int BM, int BN, int WM, int WN, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_kernel(const Product g) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const Tile tile(g, static_cast<int>(blockIdx.x));
  if (tile.there) gemm_tile<T, FORM, BM, BN, WM, WN, KG, false>(g, tile, lds, MoreSegments{}, 0);
}

// us in a training step, product and pass / rotated here: q, k, v of 1023 rows as one 1536 x 512 product 7.5 + 3.7 / 9.1; of 2331 rows as
// three 11.9 + 4.0 / 12.8; of 16384 rows as one 32 (the library's selected kernel) + 15 / 48; fp32 of 2048 rows as three 256 x 256 12.8 + 3.9 / 14.1.
template <typename T, int BM, int BN, int WM, int WN, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_rope_kernel(const Product g, const Rotation rot) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const Tile tile(g, static_cast<int>(blockIdx.x));
  if (tile.there) gemm_tile<T, FORM_NT, BM, BN, WM, WN, KG, false, false, true>(g, tile, lds, MoreSegments{}, 0, nullptr, &rot);
}

// us, one product and the pass over gate and up / the pair / without gate and up (weights out of HBM, x just written): 1376 + 1376 x 512 bf16
// 200 rows 5.8 + 4.2 / 6.3 / 6.0, 1023 rows 11.0 + 4.4 / 12.0 / 10.9, 2331 rows 15.5 + 5.8 / 17.7 / 16.1, 16384 rows in a training step 80 (the library's selected kernel) + 23 / 82;
// 688 + 688 x 256 fp32 2048 rows 20.1 + 4.8 / 20.9 / 18.9.
template <typename T, int BM, int BN, int WM, int WN, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_pair_kernel(const Product g, const Pair pair) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const Tile tile(g, static_cast<int>(blockIdx.x));
  if (tile.there) gemm_tile<T, FORM_NT, BM, BN, WM, WN, KG, false, true>(g, tile, lds, MoreSegments{}, 0, &pair);
}

// Several small products in one launch: what a linear layer's backward needs (dx and dW), or projections that share their input.
// Each alone leaves most of the chip idle and pays a launch: 1024 x 512 x 512 dx and dW are 128 and 64 tiles for 256 CUs.
enum { FORMS_NT, FORMS_NN, FORMS_ANY, FORMS_SEGMENTS };  // the products' forms, as far as they change the code
struct Products {
  int first[kMaxProducts];  // the first workgroup of each; past the last one INT_MAX
  Product p[kMaxProducts];
  MoreSegments more;
};
template <typename T, int FORMS, int BM, int BN, int WM, int WN, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_multi_kernel(const Products ps) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int block = static_cast<int>(blockIdx.x);
  int i = 0, first = ps.first[0];
#pragma unroll
  for (int k = 1; k < kMaxProducts; ++k)
    if (block >= ps.first[k]) i = k, first = ps.first[k];
  const Product& g = ps.p[i];
  const Tile tile(g, block - first);
  if (!tile.there) return;
  if (FORMS == FORMS_NT || (FORMS != FORMS_NN && g.form == FORM_NT)) gemm_tile<T, FORM_NT, BM, BN, WM, WN, KG, false>(g, tile, lds, ps.more, 0);
  else if (FORMS == FORMS_NN || g.form == FORM_NN) gemm_tile<T, FORM_NN, BM, BN, WM, WN, KG, FORMS == FORMS_SEGMENTS>(g, tile, lds, ps.more, i == ps.more.product ? ps.more.count : 0);
  else gemm_tile<T, FORM_TN, BM, BN, WM, WN, KG, false>(g, tile, lds, ps.more, 0);
}

template <typename T, int BM, int BN, int WM, int WN, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_multi_rope_kernel(const Products ps, const Rotation rot) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int block = static_cast<int>(blockIdx.x);
  int i = 0, first = ps.first[0];
#pragma unroll
  for (int k = 1; k < kMaxProducts; ++k)
    if (block >= ps.first[k]) i = k, first = ps.first[k];
  const Product& g = ps.p[i];
  const Tile tile(g, block - first);
  if (tile.there) gemm_tile<T, FORM_NT, BM, BN, WM, WN, KG, false, false, true>(g, tile, lds, ps.more, 0, nullptr, &rot, i);
}

// dW = dy^T h (if it is wanted), and dh = dy W on its way through the activation (1376 x 512, us: 1023 rows 13.4 and 5.1 for the pass /
// 16.3 here; 16384 rows in a training step, dh alone, 47 (the library's selected kernel) and 37 / 71, with dW 48 and 6 more (row slices and their sum) / 103)
template <typename T, int BM, int BN, int WM, int WN, int KG>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KG * 64) void gemm_multi_act_kernel(const Products ps, const Activation act) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int block = static_cast<int>(blockIdx.x), i = block >= ps.first[1] ? 1 : 0;
  const Product& g = ps.p[i];
  const Tile tile(g, block - ps.first[i]);
  if (!tile.there) return;
  if (g.form == FORM_NN) gemm_tile<T, FORM_NN, BM, BN, WM, WN, KG, false, false, false, true>(g, tile, lds, ps.more, 0, nullptr, nullptr, 0, &act);
  else gemm_tile<T, FORM_TN, BM, BN, WM, WN, KG, false>(g, tile, lds, ps.more, 0);
}

// C (+)= sum of the slices' fp32 partial products, one rounding; up to kMaxProducts outputs
struct Joins {
  struct Output {
    void* c;
    const float* partial;
    int slices, accumulate, first_block;
    int64_t n4;  // groups of four elements
  } p[kMaxProducts];
  int count;
};
template <typename T>
__global__ __launch_bounds__(256) void gemm_join_kernel(const Joins js) {
  int o = 0;
  while (o + 1 < js.count && static_cast<int>(blockIdx.x) >= js.p[o + 1].first_block) ++o;
  const auto& g = js.p[o];
  const int64_t i = static_cast<int64_t>(static_cast<int>(blockIdx.x) - g.first_block) * 256 + threadIdx.x, n4 = g.n4;
  if (i >= n4) return;
  typedef T t4 __attribute__((ext_vector_type(4)));
  const f32x4* p = reinterpret_cast<const f32x4*>(g.partial) + i;
  t4* c = reinterpret_cast<t4*>(g.c) + i;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  int k = 0;
  for (; k + 4 <= g.slices; k += 4) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = p[static_cast<int64_t>(k + u) * n4];
#pragma unroll
    for (int u = 0; u < 4; ++u) s += v[u];
  }
  for (; k < g.slices; ++k) s += p[static_cast<int64_t>(k) * n4];
  t4 out;
  if (g.accumulate) {
    const t4 old = *c;
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += to_f32<T>(old[e]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = from_f32<T>(s[e]);
  *c = out;
}

// ---- which tile, which split ----------------------------------------------------------------------------------------------
constexpr int kSmall = 0, k128 = 1, k256x128 = 2, k256 = 3, k128x64 = 4, k32 = 5, kTiles = 6;  // (small: 64 x 64; the 256s: bf16; 32: fp32)
constexpr int kTileM[kTiles] = {64, 128, 256, 256, 128, 32}, kTileN[kTiles] = {64, 128, 128, 256, 64, 32};
int64_t tiles_of(int64_t M, int64_t N, int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); }
int slab_of(int dtype) { return dtype == MLTS_BF16 ? 64 : 32; }
int64_t slabs_of(const mlts_gemm_product& p, int bk) {
  int64_t n = 0;
  for (int i = 0; i < p.segments; ++i) n += (p.k[i] + bk - 1) / bk;
  return n;
}

void set_slices(Product& g, int64_t slices, int64_t slabs, int bk) {
  const int64_t part = std::max<int64_t>(1, (slabs + slices - 1) / slices);
  g.k_slice = static_cast<int>(part * bk);
  g.slices = static_cast<int>(std::max<int64_t>(1, (slabs + part - 1) / part));
}

// (the parts of a bf16 sum are rounded one by one)
bool splittable(const mlts_gemm_product& p, int dtype) { return (p.segments == 1 || dtype == MLTS_F32) && p.N % 4 == 0 && p.ldc == p.N; }

// The rectangles of the eight XCDs (Tile), bm x bn the tile; returns the tiles of the largest one.
int64_t divide(Product& g, int bm, int bn) {
  auto part = [](int64_t n, int l) { return (n + (int64_t{1} << l) - 1) >> l; };
  const int64_t mean = (static_cast<int64_t>(g.tiles_m) * g.tiles_n * g.slices + 7) / 8;
  int64_t most = 0;
  double best = 0;
  for (int ls = 0; ls <= 3; ++ls)
    for (int lm = 0; lm + ls <= 3; ++lm) {
      const int ln = 3 - ls - lm;
      const int64_t depth = part(g.slices, ls), rows = part(g.tiles_m, lm), columns = part(g.tiles_n, ln), tiles = depth * rows * columns;
      const double cost = static_cast<double>(depth * (rows * bm + columns * bn)) * static_cast<double>(std::max<int64_t>(tiles, 32)) / static_cast<double>(std::max<int64_t>(mean, 32));
      if (most == 0 || cost < best) most = tiles, best = cost, g.xcds = ls | lm << 4 | ln << 8;
    }
  return most;
}

// Divides the products of a launch; each: the tiles of an XCD, returns their sum.  In runs of equal length where the largest rectangles would give a CU of their XCD
// one tile more: that costs more than what they save in L2.  (us, rectangles / runs, 33 to 36 tiles for the 32 CUs of an XCD and 32: bf16 NN 5352 x 768 x 768
// 15.9 / 11.8, 2678 x 384 x 1488 11.7 / 9.4, dx and dW of 1407 x 640 x 3408 34.6 / 26.4.  Elsewhere
// rectangles are ahead: NT 541 x 2304 x 768 7.4 / 8.9, 524 x 5456 x 1024 12.2 / 13.7.)  In fp32, whose tiles are bound by their arithmetic, in runs wherever the largest rectangle has a tile more
// (60 products and launches of dW and dx: equal, 0.4 % on the mean; tiles of 32 x 32, four on a CU for three: NN 1206 x 640 x 640 14.7 / 12.4).
int64_t spread(Product* ps, int count, int tile, int dtype, int64_t* each) {
  constexpr int64_t cus = 32;  // of an XCD
  int64_t rectangles = 0, runs = 0;
  const auto run_of = [](const Product& g) { return (static_cast<int64_t>(g.tiles_m) * g.tiles_n * g.slices + 7) / 8; };
  for (int i = 0; i < count; ++i) rectangles += each[i] = divide(ps[i], kTileM[tile], kTileN[tile]), runs += run_of(ps[i]);
  if (dtype == MLTS_BF16 ? (rectangles + cus - 1) / cus <= (runs + cus - 1) / cus : rectangles <= runs) return rectangles;
  for (int i = 0; i < count; ++i) each[i] = run_of(ps[i]), ps[i].xcds = kRuns;
  return runs;
}

// Tile and split by estimated time (us).  A launch takes `fixed`, then what the CU with the most workgroups takes for their slabs (`busy` each, one after the
// other; alone, a workgroup takes `chain`), then what is written; a split also the launch that joins the slices and their fp32 sums.
struct TileCost {
  double fixed, chain, busy, out;  // out: of a million elements
};
struct Costs {
  TileCost tile[kTiles];
  int tiles[5], count;           // that there are
  double join_fixed, join_sums;  // ... of a million partial sums
};
// bf16: fitted to 900 products in the three forms, 3 to 32000 rows, 64
// to 4096 wide, 2e6 to 2.4e10 multiplications, each on all tiles and splits; of 900 others it is off by 9 % (rms), and the choice by 0.6 % from the best (1 % of them by
// more than 11 %); of 500 launches of dW and dx by 2.3 %, 1.5 of them because a weight gradient keeps the split that it has alone.
// What a workgroup fetches decides: loads alone, with neither LDS nor matrix instructions, take as
// long as the kernel (2048 x 2048 x 1536, tiles of 64 x 64: 29 us of 30.5), and a tile of 128 x 128 fetches half as much for its work
// (us, 64 x 64 / 128 x 128: NT 2331 x 1536 x 512 12.0 / 9.4, 8192 x 2752 x 512 45.3 / 34.9, NN 16384 x 1376 x 512 48.8 / 36.5).
constexpr Costs kBf16Costs{{{2.5, 0.24, 0.24, 0.55}, {3.2, 0.52, 0.52, 0.55}, {3.95, 0.83, 0.83, 0.69}, {6.2, 1.26, 1.26, 0.56}, {3.1, 0.373, 0.373, 0.71}, {}},
                           {kSmall, k128, k256x128, k256, k128x64}, 5, 2.55, 1.73};
// fp32: fitted to 400 products in the three forms, 64 to 4096 rows, 64 to 2048 wide (and vocabularies of 8192 to 32000), 2e6 to 2.5e10 multiplications, each on all tiles and splits:
// off by 4 to 6 % (rms), the choice by 0.4 % from the best.  32 x 32, whose four wavefronts share the contraction and multiply whole elements, has the
// shortest chain; where CUs have several of them, the tiles of elements in three parts are ahead, larger ones the more so (us, 32 x 32 / 64 x 64 / 128 x 128, and the larger of these in fp32 matrix
// instructions before: NT 2048 x 256 x 256 5.9 / 7.1 / 12, 2048 x 1376 x 256 20 / 14.3 / 13.8, before 16.7; 2048 x 8192 x 256 - / 64 / 55, before 75; 4096 x 2048 x 2048 - / 216 / 172, before 245).  Of the 400 the time
// is 0.92 of that before on the geometric mean, from 5e8 multiplications on 0.55 to 0.85, and there 0.6 to 1.09 of the library's, 0.75 on the mean.
// What bounds the parts: a slab of 128 x 128 takes a CU 1.0 us, of which the matrix instructions are 1536 cycles, the LDS 1000 (192 KB) and a wavefront's splitting and addresses 500; vector
// and matrix instructions of a SIMD's wavefronts hardly overlap.  (No change: vector instructions spread between matrix instructions; twice the slabs in flight 7.1 -> 7.5.)
constexpr Costs kF32Costs{{{3.29, 0.4, 0.384, 1.22}, {4.16, 0.99, 0.99, 1.33}, {}, {}, {3.87, 0.796, 0.663, 1.13}, {2.71, 0.191, 0.15, 1.02}}, {kSmall, k128, k128x64, k32}, 4, 2.44, 2.26};
const Costs& costs_of(int dtype) { return dtype == MLTS_BF16 ? kBf16Costs : kF32Costs; }
// A second workgroup on a CU overlaps the first on 64 x 64 in bf16, by so much a slab (us, 64 x 64 / 128 x 64, of 37 and 19 tiles to an XCD: NT 2331 x 512 x 512 6.5 / 6.95, NN 6.5 /
// 6.95, dW and dx of it on 64 x 64 / 128 x 128 12.4 / 13.5).  Of 600 products and 200 launches of dW and dx the choice is 0.51 and 0.74 % from the best, 0.74 and 0.86 %
// without it.  Launches with a pass, fitted without it, go without it.
constexpr double kSmallOverlap = 0.06;
// What a pass on the way out adds in bf16 on each tile: of a launch, of a million elements; the larger ones have fewer wavefronts to overlap its latency with.  (Fitted to 250
// rotated products, 170 launches of three, 400 pairs and 300 launches of dW and dh, the choice 0.3, 0.1, 0.3 and 0.9 % from the best.)
struct PassCost {
  double fixed[kTiles], out[kTiles];
};
constexpr PassCost kRotationCost{{1.0, 1.7, 3.9, 7.2, 1.8}, {0, 0.16, 0.35, 0.38, 0.06}},
    kJointRotationCost{{1.0, 3.7}, {0, 0.16}}, kPairCost{{0.7, 1.5}, {0.5, 0.8}}, kActivationCost{{1.9, 4.0}, {1.8, 1.3}};
constexpr TileCost kRotationApart{2.0, 0, 0, 0.6};  // a launch of its own, after a split product (110 of the two, in a graph: 0.7 % from the best)
double pass_time(const PassCost& c, int tile, int64_t M, int64_t N) { return c.fixed[tile] + c.out[tile] * 1e-6 * static_cast<double>(M) * static_cast<double>(N); }

// The time of products in one launch, the slices of each given
double launch_time(int dtype, const mlts_gemm_product* const* ps, int count, int tile, const int64_t* slices, bool pass) {
  const Costs& costs = costs_of(dtype);
  const TileCost& c = costs.tile[tile];
  double longest = 0, work = 0, workgroups = 0, out = 0, sums = 0;
  int64_t of_an_xcd = 0;
  for (int i = 0; i < count; ++i) {
    const int64_t slabs = slabs_of(*ps[i], slab_of(dtype)), part = (slabs + slices[i] - 1) / slices[i];
    const int64_t tiles = tiles_of(ps[i]->M, ps[i]->N, kTileM[tile], kTileN[tile]) * (part ? (slabs + part - 1) / part : 1);
    const double elements = 1e-6 * static_cast<double>(ps[i]->M) * static_cast<double>(ps[i]->N);
    longest = std::max(longest, static_cast<double>(part));
    work += static_cast<double>(part) * static_cast<double>(tiles), workgroups += static_cast<double>(tiles);
    of_an_xcd += (tiles + 7) / 8;
    (slices[i] > 1 ? sums : out) += elements * static_cast<double>(slices[i] > 1 ? slices[i] : 1);
  }
  const double of_a_cu = static_cast<double>((of_an_xcd + 31) / 32);
  const double overlap = dtype == MLTS_BF16 && tile == kSmall && of_a_cu > 1 && !pass ? kSmallOverlap : 0;
  const double slabs = workgroups > 0 ? std::max(longest * c.chain, work / workgroups * (of_a_cu * c.busy - overlap)) : 0;
  return c.fixed + slabs + out * c.out + (sums > 0 ? costs.join_fixed + costs.join_sums * sums : 0);
}

// ... of a product in a launch by itself, its outputs rotated on their way out (split, by a launch after it) or not
double alone_time(int dtype, const mlts_gemm_product& p, int tile, int64_t slices, bool rotation) {
  const mlts_gemm_product* const one = &p;
  const double time = launch_time(dtype, &one, 1, tile, &slices, rotation);
  if (!rotation) return time;
  if (slices > 1) return time + kRotationApart.fixed + kRotationApart.out * 1e-6 * static_cast<double>(p.M) * static_cast<double>(p.N);
  return time + (dtype == MLTS_BF16 ? pass_time(kRotationCost, tile, p.M, p.N) : 0);
}

// The best tile (or `only` that) and split of a product that runs alone
int choose_tile(int dtype, const mlts_gemm_product& p, int64_t* slices, bool rotation, int only = -1) {
  const Costs& costs = costs_of(dtype);
  const int64_t slabs = slabs_of(p, slab_of(dtype));
  *slices = 1;
  if (p.segments > 1 && only < 0) return kSmall;
  int best = kSmall;
  double least = 0;
  for (int t = 0; t < costs.count; ++t) {
    if (only >= 0 && costs.tiles[t] != only) continue;
    // (32 x 32 equal within what the fit is off by: the parts, whose errors are a third)
    const double weight = costs.tiles[t] == k32 ? 1.07 : 1;
    for (int64_t s = 1; s == 1 || (splittable(p, dtype) && s <= 16 && slabs / s >= 4); s *= 2) {
      const double time = weight * alone_time(dtype, p, costs.tiles[t], s, rotation);
      if (least == 0 || time < least) least = time, best = costs.tiles[t], *slices = s;
    }
  }
  return best;
}

struct LaunchPlan {
  int tile[kMaxProducts];
  int64_t slices[kMaxProducts];
  bool together[kMaxProducts] = {};  // in the launch of several products, all of one tile
  int64_t workspace = 0;             // bytes

  // All products in one launch of small (in fp32 also 32 x 32) or of 128 x 128 tiles, or each by itself.  A weight gradient's split is the one it has alone (in fp32, on these tiles), so that
  // in bf16 its bits do not depend on what shares its launch; in fp32 they may, with the tile (mlts_gemm_multi says so).  activation: an NN product that is not split, whose output goes through the activation
  LaunchPlan(const mlts_gemm_product* ps, int count, int dtype, bool activation = false, bool rotation = false) {
    const Costs& costs = costs_of(dtype);
    const mlts_gemm_product* all[kMaxProducts];
    double apart = 0;
    int joins = 0;
    int64_t columns = 0;  // of the products of a rotated call, which share their rows
    bool parts = false;
    for (int i = 0; i < count; ++i) {
      all[i] = &ps[i];
      tile[i] = choose_tile(dtype, ps[i], &slices[i], rotation);
      apart += alone_time(dtype, ps[i], tile[i], slices[i], rotation);
      columns += ps[i].N;
      joins += slices[i] > 1;
      parts = parts || ps[i].segments > 1;
    }
    apart -= joins > 1 ? (joins - 1) * costs.join_fixed : 0;  // one launch joins them all
    if (count > 1 || parts || activation) {
      double least = 0;
      int best = -1;
      int64_t best_slices[kMaxProducts], s[kMaxProducts];
      for (int t : {kSmall, k128, k32}) {
        if ((t == k128 && parts) || (t == k32 && dtype == MLTS_BF16)) continue;
        int64_t weight[kMaxProducts];
        std::copy(slices, slices + count, weight);
        if (dtype == MLTS_F32)
          for (int i = 0; i < count; ++i) choose_tile(dtype, ps[i], &weight[i], false, t);
        for (int64_t dx = 1; dx <= (activation ? 1 : 4); dx *= 2) {
          for (int i = 0; i < count; ++i) s[i] = ps[i].form == FORM_TN ? weight[i] : ps[i].form == FORM_NN && splittable(ps[i], dtype) && slabs_of(ps[i], slab_of(dtype)) / dx >= 4 ? dx : 1;
          double time = launch_time(dtype, all, count, t, s, rotation || activation);
          if (dtype == MLTS_BF16 && rotation) time += pass_time(kJointRotationCost, t, ps[0].M, columns);
          if (dtype == MLTS_BF16 && activation) time += pass_time(kActivationCost, t, ps[count - 1].M, ps[count - 1].N);
          if (best < 0 || time < least) least = time, best = t, std::copy(s, s + count, best_slices);
        }
      }
      if (parts || activation || least <= apart) std::fill(tile, tile + count, best), std::fill(together, together + count, true), std::copy(best_slices, best_slices + count, slices);
    }
    for (int i = 0; i < count; ++i)
      if (slices[i] > 1) workspace += ps[i].M * ps[i].N * 4 * slices[i];
  }
};

// a product's tiles and slices as product i of a plan
void set_tiles(Product& g, const mlts_gemm_product& p, const LaunchPlan& plan, int i, int dtype) {
  const int bm = kTileM[plan.tile[i]], bn = kTileN[plan.tile[i]];
  g.tiles_m = static_cast<int>((p.M + bm - 1) / bm), g.tiles_n = static_cast<int>((p.N + bn - 1) / bn);
  set_slices(g, plan.slices[i], slabs_of(p, slab_of(dtype)), slab_of(dtype));
}

template <typename S>
int opt_in_lds(MltsLdsOptIn& once, const void* kern, int bytes, S what) {
  if (bytes <= 48 * 1024) return MLTS_OK;
  if (hipError_t e = once.reserve(kern, bytes); e != hipSuccess) {
    mlts_set_error("%s: cannot reserve %d bytes of LDS: %s", what, bytes, hipGetErrorString(e));
    return MLTS_ERR_LAUNCH;
  }
  return MLTS_OK;
}

// 64 x 64 in fp32: two groups of four wavefronts, a half of every slab each
template <typename T>
constexpr int kGroups = sizeof(T) == 4 ? 2 : 1;

template <typename T, int FORM, int BM, int BN, int WM, int WN, int KG = 1>
int launch_tile(const Product& g, unsigned grid, hipStream_t st) {
  typedef TileShape<T, FORM, BM, BN, WM, WN, KG> S;
  static_assert(S::LDS <= 160 * 1024, "LDS");
  auto kern = gemm_kernel<T, FORM, BM, BN, WM, WN, KG>;
  static MltsLdsOptIn once;
  if (int rc = opt_in_lds(once, reinterpret_cast<const void*>(kern), S::LDS, "mlts_gemm"); rc != MLTS_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(S::THREADS), S::LDS, st, g);
  return MLTS_OK;
}
// (128 x 128 in eight wavefronts: in bf16 of 128 registers, so that two tiles share a CU (us, four wavefronts / eight: NT 2331 x 1536 x 512 10.6 / 9.4, NN
// 8192 x 1376 x 512 23.2 / 21.8))

template <typename T, int FORM>
int launch_form(int tile, const Product& g, unsigned grid, hipStream_t st) {
  if (tile == k128) return launch_tile<T, FORM, 128, 128, 64, 32>(g, grid, st);
  if (tile == k128x64) return launch_tile<T, FORM, 128, 64, 64, 32>(g, grid, st);
  if constexpr (sizeof(T) == 4) {
    if (tile == k32) return launch_tile<T, FORM, 32, 32, 32, 32, 4>(g, grid, st);
  } else {
    if (tile == k256x128) return launch_tile<T, FORM, 256, 128, 64, 64>(g, grid, st);
    if (tile == k256) return launch_tile<T, FORM, 256, 256, 128, 64>(g, grid, st);
  }
  return launch_tile<T, FORM, 64, 64, 32, 32, kGroups<T>>(g, grid, st);
}
template <typename T>
int launch_alone(int tile, const Product& g, unsigned grid, hipStream_t st) {
  if (g.form == FORM_NT) return launch_form<T, FORM_NT>(tile, g, grid, st);
  return g.form == FORM_NN ? launch_form<T, FORM_NN>(tile, g, grid, st) : launch_form<T, FORM_TN>(tile, g, grid, st);
}

template <typename T, int BM, int BN, int WM, int WN, int KG = 1>
int launch_rope_tile(const Product& g, const Rotation& rot, unsigned grid, hipStream_t st) {
  typedef TileShape<T, FORM_NT, BM, BN, WM, WN, KG> S;
  auto kern = gemm_rope_kernel<T, BM, BN, WM, WN, KG>;
  static MltsLdsOptIn once;
  if (int rc = opt_in_lds(once, reinterpret_cast<const void*>(kern), S::LDS, "mlts_gemm_rope"); rc != MLTS_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(S::THREADS), S::LDS, st, g, rot);
  return MLTS_OK;
}
template <typename T>
int launch_rope_alone(int tile, const Product& g, const Rotation& rot, unsigned grid, hipStream_t st) {
  if (tile == k128) return launch_rope_tile<T, 128, 128, 64, 32>(g, rot, grid, st);
  if (tile == k128x64) return launch_rope_tile<T, 128, 64, 64, 32>(g, rot, grid, st);
  if constexpr (sizeof(T) == 4) {
    if (tile == k32) return launch_rope_tile<T, 32, 32, 32, 32, 4>(g, rot, grid, st);
  } else {
    if (tile == k256x128) return launch_rope_tile<T, 256, 128, 64, 64>(g, rot, grid, st);
    if (tile == k256) return launch_rope_tile<T, 256, 256, 128, 64>(g, rot, grid, st);
  }
  return launch_rope_tile<T, 64, 64, 32, 32, kGroups<T>>(g, rot, grid, st);
}
template <typename T, int BM, int BN, int WM, int WN, int KG>
int launch_rope_joint(const Products& ps, const Rotation& rot, int blocks, hipStream_t st) {
  typedef TileShape<T, FORM_NT, BM, BN, WM, WN, KG> S;
  auto kern = gemm_multi_rope_kernel<T, BM, BN, WM, WN, KG>;
  static MltsLdsOptIn once;
  if (int rc = opt_in_lds(once, reinterpret_cast<const void*>(kern), S::LDS, "mlts_gemm_rope"); rc != MLTS_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(S::THREADS), S::LDS, st, ps, rot);
  return MLTS_OK;
}

template <typename T, int BM, int BN, int WM, int WN, int KG>
int launch_act_joint(const Products& ps, const Activation& act, int blocks, hipStream_t st) {
  typedef TileShape<T, FORM_NN, BM, BN, WM, WN, KG> S;
  constexpr int bytes = std::max(S::LDS, TileShape<T, FORM_TN, BM, BN, WM, WN, KG>::LDS);
  auto kern = gemm_multi_act_kernel<T, BM, BN, WM, WN, KG>;
  static MltsLdsOptIn once;
  if (int rc = opt_in_lds(once, reinterpret_cast<const void*>(kern), bytes, "mlts_gemm_swiglu_bwd"); rc != MLTS_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(S::THREADS), bytes, st, ps, act);
  return MLTS_OK;
}

template <typename T, int FORMS, int BM, int BN, int WM, int WN, int KG>
int launch_joint(const Products& ps, int blocks, hipStream_t st) {
  typedef TileShape<T, FORM_NT, BM, BN, WM, WN, KG> S;
  constexpr int nn = TileShape<T, FORM_NN, BM, BN, WM, WN, KG>::LDS, tn = TileShape<T, FORM_TN, BM, BN, WM, WN, KG>::LDS;
  constexpr int bytes = FORMS == FORMS_NT ? S::LDS : FORMS == FORMS_NN ? nn : std::max(S::LDS, std::max(nn, tn));
  auto kern = gemm_multi_kernel<T, FORMS, BM, BN, WM, WN, KG>;
  static MltsLdsOptIn once;
  if (int rc = opt_in_lds(once, reinterpret_cast<const void*>(kern), bytes, "mlts_gemm"); rc != MLTS_OK) return rc;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(S::THREADS), bytes, st, ps);
  return MLTS_OK;
}
template <typename T, int BM, int BN, int WM, int WN, int KG>
int launch_joint_forms(int forms, const Products& ps, int blocks, hipStream_t st) {
  switch (forms) {
    case FORMS_NT: return launch_joint<T, FORMS_NT, BM, BN, WM, WN, KG>(ps, blocks, st);
    case FORMS_NN: return launch_joint<T, FORMS_NN, BM, BN, WM, WN, KG>(ps, blocks, st);
    case FORMS_ANY: return launch_joint<T, FORMS_ANY, BM, BN, WM, WN, KG>(ps, blocks, st);
    default:
      if constexpr (WM * WN == 32 * 32) return launch_joint<T, FORMS_SEGMENTS, BM, BN, WM, WN, KG>(ps, blocks, st);
      else return MLTS_ERR_INVALID;  // (plans leave parts to the small tiles)
  }
}

const char* why_not(const mlts_gemm_product& p, int dtype) {
  if (p.form < FORM_NT || p.form > FORM_TN) return "unknown form";
  if (p.segments < 1 || p.segments > (p.form == FORM_NN ? kMaxSegments : 1)) return "bad number of segments";
  if (p.M < 0 || p.N < 0 || p.M > 0x7fffffff || p.N > 0x7fffffff) return "bad shape";
  if (p.ldc < p.N || p.ldc > 0x7fffffff) return "row strides must be at least the row length and fit 32 bits";
  const int es = dtype == MLTS_BF16 ? 2 : 4, v = 16 / es;
  const bool a_kc = p.form != FORM_TN, b_kc = p.form == FORM_NT;
  for (int i = 0; i < p.segments; ++i) {
    const int64_t K = p.k[i];
    if (K < 0 || K > 0x7fffffff || p.lda[i] > 0x7fffffff || p.ldb[i] > 0x7fffffff) return "bad shape";
    if (p.lda[i] % v || p.ldb[i] % v) return "operand rows must be 16-byte aligned";
    if ((a_kc || b_kc) && K % v) return "the contraction must be a multiple of 16 bytes";
    if (p.lda[i] < (a_kc ? K : p.M) || p.ldb[i] < (b_kc ? K : p.N)) return "row strides must be at least the row length";
    const int64_t limit = (int64_t{1} << 31) - 4096;
    if ((a_kc ? p.M : K) * p.lda[i] * es >= limit || (b_kc ? p.N : K) * p.ldb[i] * es >= limit) return "operands of 2 GiB or more";
  }
  return nullptr;
}

// Whether two outputs of a call share elements (the column ranges of one buffer interleave, but do not).  Products of a launch run at
// the same time: they must not.
bool outputs_overlap(const mlts_gemm_product& p, const mlts_gemm_product& q, int es) {
  if (p.M == 0 || p.N == 0 || q.M == 0 || q.N == 0) return false;
  const uintptr_t pa = reinterpret_cast<uintptr_t>(p.c), qa = reinterpret_cast<uintptr_t>(q.c);
  if (pa > qa) return outputs_overlap(q, p, es);
  const uintptr_t p_end = pa + static_cast<uintptr_t>((p.M - 1) * p.ldc + p.N) * es;
  if (qa >= p_end) return false;
  if (p.ldc != q.ldc || (qa - pa) % es) return true;  // (row by row they may still miss each other: not worth telling apart)
  const int64_t column = static_cast<int64_t>((qa - pa) / es) % p.ldc;  // of p's row in which q starts
  return column < p.N || column + q.N > p.ldc;
}

mlts_gemm_product single(int32_t form, int64_t M, int64_t N, int64_t K, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
                         int32_t accumulate) {
  mlts_gemm_product p{};
  p.form = form, p.segments = 1, p.accumulate = accumulate;
  p.M = M, p.N = N, p.k[0] = K;
  p.a[0] = a, p.lda[0] = lda, p.b[0] = b, p.ldb[0] = ldb, p.c = c, p.ldc = ldc;
  return p;
}

// rotation: of the outputs (products of the NT form, not split), or null.  activation: of the output of the NN product (small, not split),
// alone or beside one of the TN form, or null.
template <typename T>
int run(const mlts_gemm_product* ps, int count, int dtype, float* workspace, const Rotation* rotation, const Activation* activation, hipStream_t st) {
  const LaunchPlan plan(ps, count, dtype, activation != nullptr, rotation != nullptr);
  MLTS_REQUIRE(plan.workspace == 0 || (workspace && !rotation), "mlts_gemm: a split that the call was not checked for");
  Rotation rot{};
  if (rotation) rot = *rotation;
  Products joint;
  Joins joins{};
  int join_blocks = 0, together, joint_tile = kSmall;
  bool all_nt, all_nn;
  auto clear = [&] {
    joint = {};
    std::fill(joint.first, joint.first + kMaxProducts, 0x7fffffff);
    together = 0, all_nt = all_nn = true;
  };
  auto launch = [&] {  // what `joint` holds
    if (!together) return static_cast<int>(MLTS_OK);
    int64_t tiles[kMaxProducts], at = 0;  // of an XCD
    const int64_t grid = 8 * spread(joint.p, together, joint_tile, dtype, tiles);
    MLTS_REQUIRE(grid < (int64_t{1} << 30), "mlts_gemm: too many tiles");
    for (int i = 0; i < together; ++i) joint.first[i] = static_cast<int>(at), at += 8 * tiles[i];  // (whole rounds over the XCDs, so that each product starts at the first)
    const int blocks = static_cast<int>(grid);
    const int forms = joint.more.count ? FORMS_SEGMENTS : all_nt ? FORMS_NT : all_nn ? FORMS_NN : FORMS_ANY;
    if constexpr (sizeof(T) == 4) {
      if (joint_tile == k32) {
        if (activation) return launch_act_joint<T, 32, 32, 32, 32, 4>(joint, *activation, blocks, st);
        if (rotation) return launch_rope_joint<T, 32, 32, 32, 32, 4>(joint, rot, blocks, st);
        return launch_joint_forms<T, 32, 32, 32, 32, 4>(forms, joint, blocks, st);
      }
    }
    if (joint_tile == k128) {
      if (activation) return launch_act_joint<T, 128, 128, 64, 32, 1>(joint, *activation, blocks, st);
      if (rotation) return launch_rope_joint<T, 128, 128, 64, 32, 1>(joint, rot, blocks, st);
      return launch_joint_forms<T, 128, 128, 64, 32, 1>(forms, joint, blocks, st);
    }
    if (activation) return launch_act_joint<T, 64, 64, 32, 32, kGroups<T>>(joint, *activation, blocks, st);
    if (rotation) return launch_rope_joint<T, 64, 64, 32, 32, kGroups<T>>(joint, rot, blocks, st);
    return launch_joint_forms<T, 64, 64, 32, 32, kGroups<T>>(forms, joint, blocks, st);
  };
  clear();
  MltsKernelTimer timer("gemm", st);
  for (int i = 0; i < count; ++i) {
    const mlts_gemm_product& p = ps[i];
    const int bm = kTileM[plan.tile[i]], bn = kTileN[plan.tile[i]];
    Product g{};
    g.a = p.a[0], g.b = p.b[0], g.c = p.c;
    g.lda = static_cast<int>(p.lda[0]), g.ldb = static_cast<int>(p.ldb[0]), g.ldc = static_cast<int>(p.ldc), g.K = static_cast<int>(p.k[0]);
    g.form = p.form, g.accumulate = p.accumulate != 0;
    g.M = static_cast<int>(p.M), g.N = static_cast<int>(p.N);
    set_tiles(g, p, plan, i, dtype);
    if (g.tiles_m == 0 || g.tiles_n == 0) continue;
    if (p.segments > 1) {
      if (joint.more.count) {  // a launch has room for the segments of one product
        if (int rc = launch(); rc != MLTS_OK) return rc;
        clear();
      }
      for (int k = 1; k < p.segments; ++k) {
        joint.more.a[k - 1] = p.a[k], joint.more.b[k - 1] = p.b[k];
        joint.more.lda[k - 1] = static_cast<int>(p.lda[k]), joint.more.ldb[k - 1] = static_cast<int>(p.ldb[k]), joint.more.K[k - 1] = static_cast<int>(p.k[k]);
      }
      joint.more.count = p.segments - 1, joint.more.product = together;
    }
    if (plan.slices[i] > 1) {
      g.partial = workspace;
      workspace += p.M * p.N * plan.slices[i];
      joins.p[joins.count++] = {p.c, g.partial, g.slices, g.accumulate, join_blocks, p.M * p.N / 4};
      join_blocks += static_cast<int>((p.M * p.N / 4 + 255) / 256);
    }
    if (plan.together[i]) {
      joint_tile = plan.tile[i];
      all_nt = all_nt && p.form == FORM_NT, all_nn = all_nn && p.form == FORM_NN;
      if (rotation) std::copy(rotation->columns[i], rotation->columns[i] + 4, rot.columns[together]);
      joint.p[together++] = g;
      continue;
    }
    int64_t tiles;
    const int64_t grid = 8 * spread(&g, 1, plan.tile[i], dtype, &tiles);
    MLTS_REQUIRE(grid < (int64_t{1} << 30), "mlts_gemm: too many tiles");
    if (rotation) {
      Rotation own = *rotation;
      std::copy(rotation->columns[i], rotation->columns[i] + 4, own.columns[0]);
      if (int rc = launch_rope_alone<T>(plan.tile[i], g, own, static_cast<unsigned>(grid), st); rc != MLTS_OK) return rc;
    } else if (int rc = launch_alone<T>(plan.tile[i], g, static_cast<unsigned>(grid), st); rc != MLTS_OK) {
      return rc;
    }
  }
  if (int rc = launch(); rc != MLTS_OK) return rc;
  if (joins.count) hipLaunchKernelGGL(gemm_join_kernel<T>, dim3(static_cast<unsigned>(join_blocks)), dim3(256), 0, st, joins);
  return mlts_check_launch("mlts_gemm");
}

// The tile that two products of a pair take together, or -1: one after the other
int pair_tile(int64_t M, int64_t N, int64_t K, int dtype) {
  const mlts_gemm_product both = single(FORM_NT, M, 2 * N, K, nullptr, K, nullptr, K, nullptr, 2 * N, 0);
  const LaunchPlan plan(&both, 1, dtype);
  if (plan.slices[0] > 1) return -1;
  const mlts_gemm_product* const one = &both;
  const int64_t whole = 1;
  const auto time = [&](int tile) { return launch_time(dtype, &one, 1, tile, &whole, true) + (dtype == MLTS_BF16 ? pass_time(kPairCost, tile, M, N) : 0); };
  if (dtype == MLTS_BF16) return time(k128) < time(kSmall) ? k128 : kSmall;
  if (plan.tile[0] != k32) return plan.tile[0] == kSmall ? kSmall : k128;  // (these sum in one order: the bits of the product with both weights)
  const double pass = 2.5 + 2.4e-6 * static_cast<double>(M) * static_cast<double>(N);  // (32 x 32 has no pair: the pass over gate and up is then a launch of its own)
  return time(k32) + pass < time(kSmall) ? -1 : kSmall;
}

template <typename T, int BM, int BN, int WM, int WN, int KG = 1>
int launch_pair(Product& g, const Pair& pair, hipStream_t st) {
  typedef TileShape<T, FORM_NT, BM, BN, WM, WN, KG, true> S;
  g.tiles_m = (g.M + BM - 1) / BM, g.tiles_n = (g.N + BN / 2 - 1) / (BN / 2);
  int64_t tiles;
  const int64_t grid = 8 * spread(&g, 1, BM == 128 ? k128 : kSmall, sizeof(T) == 2 ? MLTS_BF16 : MLTS_F32, &tiles);
  MLTS_REQUIRE(grid < (int64_t{1} << 30), "mlts_gemm_swiglu: too many tiles");
  auto kern = gemm_pair_kernel<T, BM, BN, WM, WN, KG>;
  static MltsLdsOptIn once;
  if (int rc = opt_in_lds(once, reinterpret_cast<const void*>(kern), S::LDS, "mlts_gemm_swiglu"); rc != MLTS_OK) return rc;
  MltsKernelTimer timer("gemm_swiglu", st);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(S::THREADS), S::LDS, st, g, pair);
  return mlts_check_launch("mlts_gemm_swiglu");
}
template <typename T>
int run_pair(int tile, Product& g, const Pair& pair, hipStream_t st) {
  if (tile == k128) return launch_pair<T, 128, 128, 64, 32>(g, pair, st);
  return launch_pair<T, 64, 64, 32, 32, kGroups<T>>(g, pair, st);
}

}  // namespace

extern "C" const char* mlts_gemm_supports(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc) {
  if (dtype != MLTS_BF16 && dtype != MLTS_F32) return "dtype must be MLTS_F32 or MLTS_BF16";
  return why_not(single(form, M, N, K, nullptr, lda, nullptr, ldb, nullptr, ldc, 0), dtype);
}

extern "C" int64_t mlts_gemm_workspace_bytes(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K) {
  const mlts_gemm_product p = single(form, M, N, K, nullptr, 0, nullptr, 0, nullptr, N, 0);
  return M <= 0 || N <= 0 ? 0 : LaunchPlan(&p, 1, dtype).workspace;
}

extern "C" int64_t mlts_gemm_multi_workspace_bytes(const mlts_gemm_product* products, int32_t count, int32_t dtype) {
  return count < 1 || count > kMaxProducts ? 0 : LaunchPlan(products, count, dtype).workspace;
}

extern "C" int mlts_gemm_plan(const mlts_gemm_product* products, int32_t count, int32_t dtype, int32_t with, mlts_gemm_tiles* tiles) {
  MLTS_REQUIRE(products && tiles && count >= 1 && count <= kMaxProducts, "mlts_gemm_plan: 1 to %d products in a call", kMaxProducts);
  MLTS_REQUIRE(dtype == MLTS_BF16 || dtype == MLTS_F32, "mlts_gemm_plan: unknown dtype %d", dtype);
  for (int i = 0; i < count; ++i)
    if (const char* why = why_not(products[i], dtype)) MLTS_REQUIRE(false, "mlts_gemm_plan: %s", why);
  if (with == MLTS_GEMM_WITH_GATE_UP) {
    const int tile = pair_tile(products[0].M, products[0].N, products[0].k[0], dtype);
    MLTS_REQUIRE(count == 1 && tile >= 0, "mlts_gemm_plan: gate and up of this size are not made in one launch");
    Product g{};
    int64_t each;
    g.tiles_m = static_cast<int>((products[0].M + kTileM[tile] - 1) / kTileM[tile]), g.tiles_n = static_cast<int>((2 * products[0].N + kTileN[tile] - 1) / kTileN[tile]), g.slices = 1;
    tiles[0] = {kTileM[tile], kTileN[tile], 1, 0, static_cast<int32_t>(std::min<int64_t>(spread(&g, 1, tile, dtype, &each), 0x7fffffff))};
    return MLTS_OK;
  }
  const LaunchPlan plan(products, count, dtype, with == MLTS_GEMM_WITH_ACTIVATION, with == MLTS_GEMM_WITH_ROTATION);
  Product joint[kMaxProducts];
  int64_t each[kMaxProducts];
  int together = 0, joint_tile = kSmall;
  for (int i = 0; i < count; ++i) {
    Product g{};
    set_tiles(g, products[i], plan, i, dtype);
    const int bm = kTileM[plan.tile[i]], bn = kTileN[plan.tile[i]];
    tiles[i] = {bm, bn, static_cast<int32_t>(plan.slices[i]), plan.together[i], static_cast<int32_t>(std::min<int64_t>(spread(&g, 1, plan.tile[i], dtype, each), 0x7fffffff))};
    if (plan.together[i] && g.tiles_m && g.tiles_n) joint[together++] = g, joint_tile = plan.tile[i];
  }
  const int64_t busiest = spread(joint, together, joint_tile, dtype, each);
  for (int i = 0; i < count; ++i)
    if (plan.together[i]) tiles[i].busiest = static_cast<int32_t>(std::min<int64_t>(busiest, 0x7fffffff));
  return MLTS_OK;
}

static int check_products(const mlts_gemm_product* products, int32_t count, int32_t dtype) {
  MLTS_REQUIRE(dtype == MLTS_BF16 || dtype == MLTS_F32, "mlts_gemm: unknown dtype %d", dtype);
  MLTS_REQUIRE(products && count >= 1 && count <= kMaxProducts, "mlts_gemm: 1 to %d products in a call", kMaxProducts);
  for (int i = 0; i < count; ++i) {
    const mlts_gemm_product& p = products[i];
    const char* why = why_not(p, dtype);
    MLTS_REQUIRE(why == nullptr, "mlts_gemm: %s", why);
    if (p.M == 0 || p.N == 0) continue;
    MLTS_REQUIRE(p.c && mlts_aligned16(p.c), "mlts_gemm: pointers must be 16-byte aligned and not null");
    for (int k = 0; k < p.segments; ++k)
      MLTS_REQUIRE(p.k[k] == 0 || (p.a[k] && p.b[k] && mlts_aligned16(p.a[k]) && mlts_aligned16(p.b[k])),
                   "mlts_gemm: pointers must be 16-byte aligned and not null");
    for (int j = 0; j < i; ++j)
      MLTS_REQUIRE(!outputs_overlap(products[j], p, dtype == MLTS_BF16 ? 2 : 4), "mlts_gemm: outputs %d and %d of the call overlap", j, i);
  }
  return MLTS_OK;
}

extern "C" int mlts_gemm_multi(const mlts_gemm_product* products, int32_t count, int32_t dtype, void* workspace, int64_t workspace_bytes,
                               mlts_stream_t stream) {
  if (int rc = check_products(products, count, dtype); rc != MLTS_OK) return rc;
  const int64_t need = mlts_gemm_multi_workspace_bytes(products, count, dtype);
  MLTS_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && mlts_aligned16(workspace)), "mlts_gemm: workspace too small or unaligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* ws = static_cast<float*>(workspace);
  return dtype == MLTS_BF16 ? run<bf16_t>(products, count, dtype, ws, nullptr, nullptr, st) : run<float>(products, count, dtype, ws, nullptr, nullptr, st);
}

extern "C" int mlts_gemm(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K, const void* a, int64_t lda, const void* b, int64_t ldb,
                         void* c, int64_t ldc, int32_t accumulate, void* workspace, int64_t workspace_bytes, mlts_stream_t stream) {
  const mlts_gemm_product p = single(form, M, N, K, a, lda, b, ldb, c, ldc, accumulate);
  return mlts_gemm_multi(&p, 1, dtype, workspace, workspace_bytes, stream);
}

extern "C" const char* mlts_gemm_swiglu_supports(int32_t dtype, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldc, int64_t ldh) {
  if (dtype != MLTS_BF16 && dtype != MLTS_F32) return "dtype must be MLTS_F32 or MLTS_BF16";
  if (const char* why = why_not(single(FORM_NT, M, N, K, nullptr, ldx, nullptr, ldw, nullptr, ldc, 0), dtype)) return why;
  if (M <= 0 || N <= 0 || K <= 0) return "an empty product";
  if (N % 4 || ldc % 4 || ldh % 4 || ldh < N || ldh > 0x7fffffff || 2 * N > 0x7fffffff) return "rows of gate, up and h are written four elements at a time";
  return pair_tile(M, N, K, dtype) < 0 ? "products of this size are not made in one launch" : nullptr;
}

extern "C" int mlts_gemm_swiglu(int32_t dtype, int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx, const void* w_gate, const void* w_up, int64_t ldw,
                                void* gate, void* up, int64_t ldc, void* h, int64_t ldh, mlts_stream_t stream) {
  const char* why = mlts_gemm_swiglu_supports(dtype, M, N, K, ldx, ldw, ldc, ldh);
  MLTS_REQUIRE(why == nullptr, "mlts_gemm_swiglu: %s", why);
  MLTS_REQUIRE(x && w_gate && w_up && h && !gate == !up, "mlts_gemm_swiglu: null pointer");
  for (const void* p : {x, w_gate, w_up, static_cast<const void*>(gate), static_cast<const void*>(up), static_cast<const void*>(h)})
    MLTS_REQUIRE(!p || mlts_aligned16(p), "mlts_gemm_swiglu: pointers must be 16-byte aligned");
  Product g{};
  g.a = x, g.b = w_gate, g.c = gate;
  g.lda = static_cast<int>(ldx), g.ldb = static_cast<int>(ldw), g.ldc = static_cast<int>(ldc);
  g.M = static_cast<int>(M), g.N = static_cast<int>(N), g.K = static_cast<int>(K);
  g.form = FORM_NT, g.slices = 1, g.k_slice = static_cast<int>(K);
  const Pair pair{w_up, up, h, static_cast<int>(ldh), up && M * N * (dtype == MLTS_BF16 ? 2 : 4) > int64_t{32} << 20};
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int tile = pair_tile(M, N, K, dtype);
  return dtype == MLTS_BF16 ? run_pair<bf16_t>(tile, g, pair, st) : run_pair<float>(tile, g, pair, st);
}

extern "C" const char* mlts_gemm_rope_supports(const mlts_gemm_product* products, int32_t count, int32_t dtype, const mlts_gemm_rotation* rotation) {
  if (!products || !rotation || count < 1 || count > kMaxProducts) return "1 to 4 products in a call";
  if (dtype != MLTS_BF16 && dtype != MLTS_F32) return "dtype must be MLTS_F32 or MLTS_BF16";
  if (rotation->head_dim < 4 || rotation->head_dim % 4 || rotation->max_pos < 1 || rotation->seq < 1) return "bad rotation";
  for (int i = 0; i < count; ++i) {
    const mlts_gemm_product& p = products[i];
    if (const char* why = why_not(p, dtype)) return why;
    if (p.form != FORM_NT || p.accumulate || p.M <= 0 || p.N <= 0 || p.k[0] <= 0 || p.N % 4 || p.ldc % 4) return "products whose outputs are not rotated";
    for (int r = 0; r < 4; r += 2) {
      const int64_t a = rotation->columns[i][r], b = rotation->columns[i][r + 1];
      if (a < 0 || b < a || b > p.N || a % 4 || (b - a) % rotation->head_dim) return "columns that are not whole heads";
    }
  }
  return LaunchPlan(products, count, dtype, false, true).workspace ? "products that would be split" : nullptr;
}

extern "C" int mlts_gemm_rope(const mlts_gemm_product* products, int32_t count, int32_t dtype, const mlts_gemm_rotation* rotation, mlts_stream_t stream) {
  const char* why = mlts_gemm_rope_supports(products, count, dtype, rotation);
  MLTS_REQUIRE(why == nullptr, "mlts_gemm_rope: %s", why);
  if (int rc = check_products(products, count, dtype); rc != MLTS_OK) return rc;
  MLTS_REQUIRE(rotation->cos && rotation->sin && ((reinterpret_cast<uintptr_t>(rotation->cos) | reinterpret_cast<uintptr_t>(rotation->sin)) & 7) == 0,
               "mlts_gemm_rope: the cos / sin tables must be 8-byte aligned and not null");
  MLTS_REQUIRE(rotation->positions || (rotation->position_offset >= 0 && rotation->position_offset + static_cast<int64_t>(rotation->seq) <= rotation->max_pos),
               "mlts_gemm_rope: positions exceed the table (%d rows)", rotation->max_pos);
  Rotation r{rotation->cos, rotation->sin, rotation->positions, rotation->max_pos, rotation->position_offset, rotation->seq, rotation->head_dim, {}};
  for (int i = 0; i < count; ++i)
    for (int k = 0; k < 4; ++k) r.columns[i][k] = static_cast<int>(rotation->columns[i][k]);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == MLTS_BF16 ? run<bf16_t>(products, count, dtype, nullptr, &r, nullptr, st) : run<float>(products, count, dtype, nullptr, &r, nullptr, st);
}

// the products of the last projection's backward pass: dW, if it is wanted, then dh
static int swiglu_bwd_products(mlts_gemm_product (&ps)[2], int64_t M, int64_t N, int64_t K, const void* dy, int64_t ldy, const void* w, int64_t ldw,
                               const void* h, int64_t ldh, void* dw, int32_t accumulate, bool weight) {
  int count = 0;
  if (weight) ps[count++] = single(FORM_TN, K, N, M, dy, ldy, h, ldh, dw, N, accumulate);
  ps[count++] = single(FORM_NN, M, N, K, dy, ldy, w, ldw, nullptr, N, 0);
  return count;
}

extern "C" const char* mlts_gemm_swiglu_bwd_supports(int32_t dtype, int32_t weight, int64_t M, int64_t N, int64_t K, int64_t ldy, int64_t ldw, int64_t ldh,
                                                     int64_t ldg, int64_t ldd, int64_t* workspace_bytes) {
  if (dtype != MLTS_BF16 && dtype != MLTS_F32) return "dtype must be MLTS_F32 or MLTS_BF16";
  if (M <= 0 || N <= 0 || K <= 0) return "an empty product";
  mlts_gemm_product ps[2];
  const int count = swiglu_bwd_products(ps, M, N, K, nullptr, ldy, nullptr, ldw, nullptr, ldh, nullptr, 0, weight != 0);
  for (int i = 0; i < count; ++i)
    if (const char* why = why_not(ps[i], dtype)) return why;
  if (N % 4 || ldg % 4 || ldd % 4 || ldg < N || ldd < N || ldg > 0x7fffffff || ldd > 0x7fffffff) return "rows of gate and up are taken four elements at a time";
  if (LaunchPlan(ps, count, dtype).slices[count - 1] > 1) return "a product that would be split";
  const LaunchPlan plan(ps, count, dtype, true);
  if (!std::all_of(plan.together, plan.together + count, [](bool t) { return t; }) || plan.slices[count - 1] > 1) return "products of this size are not made in one launch";
  *workspace_bytes = plan.workspace;
  return nullptr;
}

extern "C" int mlts_gemm_swiglu_bwd(int32_t dtype, int64_t M, int64_t N, int64_t K, const void* dy, int64_t ldy, const void* w, int64_t ldw, const void* h,
                                    int64_t ldh, void* dw, int32_t accumulate, const void* gate, const void* up, int64_t ldg, void* dgate, void* dup,
                                    int64_t ldd, void* workspace, int64_t workspace_bytes, mlts_stream_t stream) {
  int64_t need = 0;
  const char* why = mlts_gemm_swiglu_bwd_supports(dtype, dw != nullptr, M, N, K, ldy, ldw, ldh, ldg, ldd, &need);
  MLTS_REQUIRE(why == nullptr, "mlts_gemm_swiglu_bwd: %s", why);
  for (const void* p : {dy, w, gate, up, static_cast<const void*>(dgate), static_cast<const void*>(dup)})
    MLTS_REQUIRE(p && mlts_aligned16(p), "mlts_gemm_swiglu_bwd: pointers must be 16-byte aligned and not null");
  MLTS_REQUIRE(!dw || (h && mlts_aligned16(h) && mlts_aligned16(dw)), "mlts_gemm_swiglu_bwd: pointers must be 16-byte aligned and not null");
  MLTS_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && mlts_aligned16(workspace)), "mlts_gemm_swiglu_bwd: workspace too small or unaligned");
  mlts_gemm_product ps[2];
  const int count = swiglu_bwd_products(ps, M, N, K, dy, ldy, w, ldw, h, ldh, dw, accumulate, dw != nullptr);
  const Activation act{gate, up, dgate, dup, static_cast<int>(ldg), static_cast<int>(ldd)};
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* ws = static_cast<float*>(workspace);
  return dtype == MLTS_BF16 ? run<bf16_t>(ps, count, dtype, ws, nullptr, &act, st) : run<float>(ps, count, dtype, ws, nullptr, &act, st);
}
