// Types and device helpers shared by the GEMM kernels (gemm.hip: shapes that
// tile exactly and general strides; gemm_edge.hip: any sizes and alignments).
#pragma once

#include "adamw.hpp"
#include "hip_util.hpp"

namespace aicf::hip {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

enum InKind { IN_F32 = 0, IN_F16 = 1, IN_BF16 = 2 };
enum OutKind { OUT_F32 = 0, OUT_F16 = 1, OUT_BF16 = 2 };
// ACT_ADAMW (fp32 accumulators only): the tile is the gradient of a weight
// matrix; the epilogue applies AdamW to that weight instead of storing it.
enum Act { ACT_NONE = 0, ACT_RELU = 1, ACT_GELU = 2, ACT_DGELU = 3, ACT_ADAMW = 4 };

// Optimizer state a fused weight-gradient GEMM updates in place ([M, N]
// row-major like the output, leading dimension ldc).
struct GemmAdamW {
  float* P;             // fp32 master weights
  float* M;             // first moment
  float* V;             // second moment
  uint16_t* Wb;         // bf16 shadow of P
  const int32_t* step;  // device step counter (already incremented)
  AdamWArgs args;
};
enum LoadMode { LD_KCONTIG = 0, LD_MNCONTIG = 1, LD_GATHER = 2 };

struct GemmParams {
  const void* A;
  const void* B;
  void* C;
  const void* bias;  // nullptr = no bias
  void* aux;         // pre-activation out (GELU) or Z in (DGELU); nullptr = none
  int64_t M, N, K;
  int64_t a_rs, a_cs;  // logical A[M,K] strides (elements)
  int64_t b_rs, b_cs;  // logical B[K,N] strides
  int64_t c_rs, c_cs;
  int64_t bias_s;
  int64_t aux_rs;
  int a_mode, b_mode;
  int act;
  int bias_f32;  // bias stored as fp32 (else in the output type)
  int tiles_m, tiles_n;
  GemmAdamW adam;  // ACT_ADAMW only
  float* colsum;   // ACT_DGELU, bf16 out: per-tile column sums of C, row m0/256 of [M/256, N]
  int apart;       // set by run_gemm: gemm_outputs_apart
};

// Whether no byte that the call writes (es, os: bytes of an operand's and an
// output's element) lies in A or B.  A product written over an operand is
// right where one tile spans N (over A) or M (over B): its workgroup has read
// all that it overwrites, and no other one reads it.  Such a call keeps to the
// largest exact tiles, and to the general-stride kernel where none fits; tiles
// that read their neighbours' rows and smaller ones would break it.
inline bool gemm_outputs_apart(const GemmParams& p, int64_t es, int64_t os) {
  struct Range {
    uintptr_t lo, hi;
  };
  auto range = [](const void* d, int64_t r, int64_t rs, int64_t c, int64_t cs, int64_t size) {
    const uintptr_t lo = reinterpret_cast<uintptr_t>(d);
    return Range{lo, lo + (uintptr_t)(((r - 1) * rs + (c - 1) * cs + 1) * size)};
  };
  const Range in[2] = {range(p.A, p.M, p.a_rs, p.K, p.a_cs, es), range(p.B, p.K, p.b_rs, p.N, p.b_cs, es)};
  auto apart = [&](const void* d, int64_t ld, int64_t cs, int64_t size) {
    const Range o = range(d, p.M, ld, p.N, cs, size);
    return !d || ((o.hi <= in[0].lo || in[0].hi <= o.lo) && (o.hi <= in[1].lo || in[1].hi <= o.lo));
  };
  if (!apart(p.C, p.c_rs, p.c_cs, os)) return false;
  if (p.act == ACT_GELU && !apart(p.aux, p.aux_rs, 1, os)) return false;
  if (p.act == ACT_ADAMW)
    return apart(p.adam.M, p.c_rs, 1, 4) && apart(p.adam.V, p.c_rs, 1, 4) && apart(p.adam.Wb, p.c_rs, 1, 2);
  return true;
}

template <int IN>
struct InTraits;
template <>
struct InTraits<IN_F32> {
  typedef float T;
  static constexpr int CE = 4;    // elements per 16-byte chunk
  static constexpr int KPM = 2;   // K per MFMA
  static constexpr int EPL = 1;   // elements per lane per MFMA operand
};
template <>
struct InTraits<IN_F16> {
  typedef uint16_t T;
  static constexpr int CE = 8;
  static constexpr int KPM = 16;
  static constexpr int EPL = 8;
};
template <>
struct InTraits<IN_BF16> {
  typedef uint16_t T;
  static constexpr int CE = 8;
  static constexpr int KPM = 16;
  static constexpr int EPL = 8;
};

template <int OUT>
__device__ __forceinline__ void store_out(void* base, int64_t idx, float v) {
  if constexpr (OUT == OUT_F32) {
    ((float*)base)[idx] = v;
  } else if constexpr (OUT == OUT_F16) {
    ((uint16_t*)base)[idx] = f32_to_f16(v);
  } else {
    ((uint16_t*)base)[idx] = f32_to_bf16(v);
  }
}
template <int OUT>
__device__ __forceinline__ float load_out(const void* base, int64_t idx) {
  if constexpr (OUT == OUT_F32) {
    return ((const float*)base)[idx];
  } else if constexpr (OUT == OUT_F16) {
    return f16_to_f32(((const uint16_t*)base)[idx]);
  } else {
    return bf16_to_f32(((const uint16_t*)base)[idx]);
  }
}

template <int IN>
__device__ __forceinline__ floatx16 mfma32(const typename InTraits<IN>::T* a,
                                          const typename InTraits<IN>::T* b, floatx16 acc);

template <>
__device__ __forceinline__ floatx16 mfma32<IN_F32>(const float* a, const float* b, floatx16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a[0], b[0], acc, 0, 0, 0);
}
template <>
__device__ __forceinline__ floatx16 mfma32<IN_BF16>(const uint16_t* a, const uint16_t* b,
                                                   floatx16 acc) {
  const bf16x8 av = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(a));
  const bf16x8 bv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(b));
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);
}
template <>
__device__ __forceinline__ floatx16 mfma32<IN_F16>(const uint16_t* a, const uint16_t* b,
                                                  floatx16 acc) {
  const f16x8 av = __builtin_bit_cast(f16x8, *reinterpret_cast<const u16x8*>(a));
  const f16x8 bv = __builtin_bit_cast(f16x8, *reinterpret_cast<const u16x8*>(b));
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc, 0, 0, 0);
}

// 16 x 16 x 32 MFMA (16-bit operands): a lane holds 8 consecutive K of one
// row of each operand; the 16 x 16 fp32 result has row (lane & 15) of the
// A operand and 4 consecutive columns 4 (lane >> 4) .. +3 of the B operand.
// Same flops per issue cycle as 32 x 32 x 16 with a quarter of the
// accumulator registers per instruction: it moves half the accumulator bits
// per flop, and on this power-limited part it sustains a ~10% higher clock.
template <int IN>
__device__ __forceinline__ floatx4 mfma16(const uint16_t* a, const uint16_t* b, floatx4 acc) {
  if constexpr (IN == IN_BF16) {
    const bf16x8 av = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(a));
    const bf16x8 bv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(b));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
  } else {
    const f16x8 av = __builtin_bit_cast(f16x8, *reinterpret_cast<const u16x8*>(a));
    const f16x8 bv = __builtin_bit_cast(f16x8, *reinterpret_cast<const u16x8*>(b));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc, 0, 0, 0);
  }
}

// Grouped raster: workgroup w of XCD x (dispatch order w*8+x) gets
// tile (tm, tn) so that each XCD sweeps a contiguous run of tiles and
// GROUP_M consecutive tile rows share B columns in its L2.
__device__ __forceinline__ void tile_coords_of(int id, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  // XCD-aware remap: hardware id i runs on XCD (i % 8); give every XCD a
  // contiguous range of logical ids.
  if ((total & 7) == 0) {
    const int per = total >> 3;
    id = (id & 7) * per + (id >> 3);
  }
  constexpr int GROUP_M = 4;  // measured best on MI355X for 256x256 tiles
  const int group = id / (GROUP_M * tiles_n);
  const int first_m = group * GROUP_M;
  const int gsize = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_group = id % (GROUP_M * tiles_n);
  tm = first_m + in_group % gsize;
  tn = in_group / gsize;
}

// Chunk swizzle of an M/N-contiguous tile in LDS ([k][mn] rows of CPR 16-byte
// chunks, ES bytes an element): row k keeps chunk c at c ^ nt_mn_swizzle(k).
//   16-bit, the 32 lanes of one LDS pass of a transposing fragment read cover 8
//   K-rows, 0-3 and 8-11 of a fragment's 32 (16 x 16 fragments: MS 16) or 0-7
//   (32 x 32: groups 0 and 1 at MN + 0 and + 16):
//     16 chunks or more: with 32 x 32 fragments c ^ 4 (k & 3) keeps the rows on
//       distinct banks; with 16 x 16 fragments both groups read the same 16 MN
//       elements 8 rows apart, and the extra 2 ((k >> 3) & 1) term moves the
//       second group to the other bank half;
//     8 chunks (64-wide tiles): rows of one parity share a 128-byte bank half,
//       so the four of them take its four 32-byte slots: chunk pair XOR (bit 1,
//       bit 3) of k;
//     4 chunks (32-wide, the edge kernel's): rows 0-3 and 8-11 take different
//       halves of their 64 bytes.
//   fp32: a fragment read takes row k and row k + 4 in the two halves of the
//   wave (32 consecutive floats each).  In rows of 16 chunks or more they sit 8
//   chunks (32 banks) apart; a row of 8 chunks is one fragment wide and stays as
//   it is, so the two share their banks.
// Every 16-bit form keeps rows k and k + 4 (k % 8 < 4) alike, as the fragment's
// second read (4 rows on) reuses the first one's column.
template <int MS, int ES = 2, int CPR = 16>
__device__ __forceinline__ int nt_mn_swizzle(int k) {
  if constexpr (ES == 4) return CPR >= 16 ? 8 * ((k >> 2) & 1) : 0;
  if constexpr (CPR == 8) return 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1));
  if constexpr (CPR == 4) return 2 * ((k >> 3) & 1);
  return MS == 16 ? ((4 * (k & 3)) ^ (2 * ((k >> 3) & 1))) : 4 * (k & 3);
}

// gemm_edge.hip: C = epi(op(A) . op(B)) for any M, N, K >= 16 bytes and any
// alignment, operands K- or M/N-contiguous, C with unit column stride.
bool edge_gemm_ok(const GemmParams& p, int in);
// Whether a 16-bit product of whole smaller tiles runs there all the same: at
// most one 32 x 32 tile a CU and long K, which eight groups of waves share
// (64 x 256 x 4096 11.6 -> 9.7 us, 256 x 1024 x 4096 12.0 -> 10.5 against the
// 64 x 64 tiles with 8 stages; M-contiguous A from K = 4096: 256 x 256 x 8192
// 23.1 -> 17.5, 512 x 512 x 4096 equal).  Plain and AdamW products alike: an
// update has the same bits with and without the separate gradient.
bool edge_splits_k(const GemmParams& p, int in);
Status edge_gemm(GemmParams& p, int in, int out, void* stream);

}  // namespace aicf::hip
