// GEMM and GEMM + fused epilogue for gfx950 on the MFMA matrix cores.
//
//   C[M,N] = epi( op(A)[M,K] . op(B)[K,N] )
//
// Reference contracts:
//   Gemm          src/backends/cuda/ops/gemm/launcher.cu:41-70 (attrs <ii> transA,
//                 transB under schema 0 or GEMM), :75-148 (2-D views, checks),
//                 :342-359 (f16 path needs a row-major contiguous C)
//   GemmEpilogue  src/backends/cuda/ops/gemm_epilogue/launcher.cu:49-80 (attrs
//                 <iii> transA, transB, relu under schema 0 or GPEL, relu
//                 default 1), :153-193 (checks: bias rank 1, length N)
//                 plus the executor's GEPI layout <iii> transA, transB, kind
//                 (core_v2/exec.py:211-252), honoured here as documented.
//
// Kernel design (one templated kernel, all dtypes):
//   * workgroup tile BM x BN x BK, WM x WN waves, each wave owns a
//     (BM/WM) x (BN/WN) block of 32x32 MFMA tiles with fp32 accumulators;
//   * 16-bit inputs use v_mfma_f32_32x32x16_{bf16,f16}, fp32 inputs use
//     v_mfma_f32_32x32x2f32 (true fp32 products, no reduced-precision path);
//   * A and B tiles live in LDS as [rows][BK] with K contiguous; 16-byte
//     chunks of a row are XOR-swizzled by (row mod chunks-per-row) so the
//     fragment reads of 32 consecutive rows spread over all banks;
//   * operands whose K stride is 1 are copied with 16-byte loads; operands
//     whose M/N stride is 1 (transposed views) are loaded 16 bytes along
//     M/N and transposed on the LDS write; anything else is gathered per
//     element;
//   * two LDS buffers: the global loads of tile k+1 are in flight while the
//     MFMAs of tile k run, with one barrier per K step;
//   * workgroup ids are remapped so that consecutive tiles of one XCD share
//     A rows (grouped column-major raster per XCD).
#include <type_traits>
#include <utility>

#include "../common/gemm_types.hpp"
#include "../common/smallstep.hpp"

namespace aicf::hip {

namespace {

// XOR swizzle of the 16-byte chunk index inside one LDS row.
template <int NCH>
__device__ __forceinline__ int swz(int row, int chunk) {
  return chunk ^ (row & (NCH - 1));
}

// Loads one operand tile (ROWS x BK, rows along M or N) from global memory
// into registers, then writes it to LDS.  `rs` steps along the tile rows
// (M or N), `cs` along K.
template <int IN, int ROWS, int BK, int THREADS>
struct TileLoader {
  typedef typename InTraits<IN>::T T;
  static constexpr int CE = InTraits<IN>::CE;
  static constexpr int NCH = BK / CE;                    // chunks per LDS row
  static constexpr int CHUNKS = ROWS * BK / CE;          // 16-byte chunks per tile
  static constexpr int PER_THREAD = (CHUNKS + THREADS - 1) / THREADS;
  typedef T vec __attribute__((ext_vector_type(CE)));
  vec r[PER_THREAD];

  // mode LD_KCONTIG: chunk c covers row c / NCH, k chunk c % NCH.
  // mode LD_MNCONTIG: chunk c covers k row c / (ROWS/CE), row chunk c % (ROWS/CE).
  __device__ void load(const T* __restrict__ g, int mode, int64_t row0, int64_t rows_total,
                       int64_t k0, int64_t K, int64_t rs, int64_t cs, bool vec_ok) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int c = t + i * THREADS;
      vec v;
#pragma unroll
      for (int e = 0; e < CE; ++e) v[e] = T(0);
      if (c < CHUNKS) {
        if (mode == LD_KCONTIG) {
          const int row = c / NCH, kc = c % NCH;
          const int64_t gr = row0 + row, gk = k0 + (int64_t)kc * CE;
          if (gr < rows_total) {
            if (vec_ok && gk + CE <= K) {
              v = *reinterpret_cast<const vec*>(g + gr * rs + gk);
            } else {
#pragma unroll
              for (int e = 0; e < CE; ++e)
                if (gk + e < K) v[e] = g[gr * rs + (gk + e) * cs];
            }
          }
        } else {
          constexpr int RCH = ROWS / CE;
          const int kr = c / RCH, rc = c % RCH;
          const int64_t gk = k0 + kr, gr = row0 + (int64_t)rc * CE;
          if (gk < K) {
            if (mode == LD_MNCONTIG && vec_ok && gr + CE <= rows_total) {
              v = *reinterpret_cast<const vec*>(g + gk * cs + gr);
            } else {
#pragma unroll
              for (int e = 0; e < CE; ++e)
                if (gr + e < rows_total) v[e] = g[(gr + e) * rs + gk * cs];
            }
          }
        }
      }
      r[i] = v;
    }
  }

  __device__ void store(T* __restrict__ lds, int mode) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int c = t + i * THREADS;
      if (c >= CHUNKS) continue;
      if (mode == LD_KCONTIG) {
        const int row = c / NCH, kc = c % NCH;
        *reinterpret_cast<vec*>(lds + row * BK + swz<NCH>(row, kc) * CE) = r[i];
      } else {
        constexpr int RCH = ROWS / CE;
        const int kr = c / RCH, rc = c % RCH;
        const int kc = kr / CE, ke = kr % CE;
#pragma unroll
        for (int e = 0; e < CE; ++e) {
          const int row = rc * CE + e;
          lds[row * BK + swz<NCH>(row, kc) * CE + ke] = r[i][e];
        }
      }
    }
  }
};

__device__ __forceinline__ void tile_coords(int tiles_m, int tiles_n, int& tm, int& tn) {
  tile_coords_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
}

template <int IN, int OUT, int BM, int BN, int BK, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mfma_kernel(GemmParams p) {
  typedef typename InTraits<IN>::T T;
  constexpr int THREADS = 64 * WM * WN;
  constexpr int CE = InTraits<IN>::CE;
  constexpr int KPM = InTraits<IN>::KPM;
  constexpr int EPL = InTraits<IN>::EPL;
  constexpr int NCH = BK / CE;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  static_assert(TM >= 1 && TN >= 1, "wave tile must hold a 32x32 block");

  __shared__ __attribute__((aligned(16))) T lds_a[2][BM * BK];
  __shared__ __attribute__((aligned(16))) T lds_b[2][BN * BK];

  int tm_i, tn_i;
  tile_coords(p.tiles_m, p.tiles_n, tm_i, tn_i);
  const int64_t m0 = (int64_t)tm_i * BM, n0 = (int64_t)tn_i * BN;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;

  const T* A = (const T*)p.A;
  const T* B = (const T*)p.B;
  // vector loads need 16-byte aligned rows and base
  const int a_lead = p.a_mode == LD_KCONTIG ? 0 : 1;
  const bool a_vec = (p.a_mode != LD_GATHER) && ((uintptr_t)A % 16 == 0) &&
                     (((a_lead == 0 ? p.a_rs : p.a_cs) * (int64_t)sizeof(T)) % 16 == 0);
  const bool b_vec = (p.b_mode != LD_GATHER) && ((uintptr_t)B % 16 == 0) &&
                     (((p.b_mode == LD_KCONTIG ? p.b_cs : p.b_rs) * (int64_t)sizeof(T)) % 16 == 0);

  TileLoader<IN, BM, BK, THREADS> la;
  TileLoader<IN, BN, BK, THREADS> lb;
  // A tile rows are M (row stride a_rs, k stride a_cs); B tile rows are N
  // (row stride b_cs, k stride b_rs).
  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int nk = (int)((p.K + BK - 1) / BK);
  la.load(A, p.a_mode, m0, p.M, 0, p.K, p.a_rs, p.a_cs, a_vec);
  lb.load(B, p.b_mode, n0, p.N, 0, p.K, p.b_cs, p.b_rs, b_vec);
  la.store(lds_a[0], p.a_mode);
  lb.store(lds_b[0], p.b_mode);
  __syncthreads();

  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) {
      la.load(A, p.a_mode, m0, p.M, (int64_t)(kt + 1) * BK, p.K, p.a_rs, p.a_cs, a_vec);
      lb.load(B, p.b_mode, n0, p.N, (int64_t)(kt + 1) * BK, p.K, p.b_cs, p.b_rs, b_vec);
    }
    const T* sa = lds_a[cur];
    const T* sb = lds_b[cur];
#pragma unroll
    for (int ks = 0; ks < BK / KPM; ++ks) {
      // fragment k position of this lane inside the tile
      const int k = ks * KPM + (lane >> 5) * EPL;
      const int kc = k / CE, ke = k % CE;
      T fa[TM][EPL], fb[TN][EPL];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * WTM + i * 32 + (lane & 31);
        const T* src = sa + row * BK + swz<NCH>(row, kc) * CE + ke;
        if constexpr (EPL == 8) {
          *reinterpret_cast<u16x8*>(fa[i]) = *reinterpret_cast<const u16x8*>(src);
        } else {
          fa[i][0] = src[0];
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn * WTN + j * 32 + (lane & 31);
        const T* src = sb + row * BK + swz<NCH>(row, kc) * CE + ke;
        if constexpr (EPL == 8) {
          *reinterpret_cast<u16x8*>(fb[j]) = *reinterpret_cast<const u16x8*>(src);
        } else {
          fb[j][0] = src[0];
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma32<IN>(fa[i], fb[j], acc[i][j]);
    }
    if (kt + 1 < nk) {
      la.store(lds_a[cur ^ 1], p.a_mode);
      lb.store(lds_b[cur ^ 1], p.b_mode);
    }
    __syncthreads();
  }

  // Epilogue.  Accumulator r of lane l in tile (i, j) holds
  // row 8*(r/4) + 4*(l/32) + r%4 and column l%32 of that 32x32 block.
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t n = n0 + wn * WTN + j * 32 + (lane & 31);
      if (n >= p.N) continue;
      float bv = 0.0f;
      if (p.bias) {
        bv = p.bias_f32 ? ((const float*)p.bias)[n * p.bias_s] : load_out<OUT>(p.bias, n * p.bias_s);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + wm * WTM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (m >= p.M) continue;
        float v = acc[i][j][r];
        if (p.act == ACT_DGELU) {
          v = v * gelu_tanh_grad_f(load_out<OUT>(p.aux, m * p.aux_rs + n));
        } else {
          v += bv;
          if (p.act == ACT_RELU) {
            v = v > 0.0f ? v : 0.0f;
          } else if (p.act == ACT_GELU) {
            if (p.aux) store_out<OUT>(p.aux, m * p.aux_rs + n, v);
            v = gelu_tanh_f(v);
          }
        }
        store_out<OUT>(p.C, m * p.c_rs + n * p.c_cs, v);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Tiled MFMA path for tile-divisible shapes: 16-bit operands (each
// K-contiguous or M/N-contiguous) and fp32 operands (K-contiguous).
//   * BM x BN workgroup tiles; a stage holds 128 bytes of K per row (64
//     16-bit or 32 fp32 elements); WM x WN waves (one or two per SIMD for
//     the 256x256 tile), each owning (BM/WM) x (BN/WN) = TM x TN blocks of
//     32x32 fp32 accumulators (v_mfma_f32_32x32x16_bf16/f16, or 4 x
//     v_mfma_f32_32x32x2f32 per 16-byte fp32 fragment);
//   * global -> LDS with gfx950's direct 16-byte LDS loads
//     (buffer_load_dwordx4 ... lds): lane i of a wave fills bytes
//     [16i, 16i+16) of a 1 KB LDS block, so there is no VGPR staging and no
//     ds_write; the XOR swizzle that keeps the fragment reads bank-conflict
//     free is applied by choosing which global chunk each lane fetches;
//   * two LDS stages and one barrier per K-step, placed before the last
//     sub-step so that no wave waits on LDS after it;
//   * the MFMA fragments of sub-step s+1 are read from LDS while the MFMAs of
//     sub-step s run (two register sets), spread over the MFMAs
//     (sched_group_barrier); with K-contiguous operands the next K-step's
//     loads are spread over two sub-steps as well (all at once, they back up
//     the address queue of the CU and stall the MFMA issue);
//   * MFMA operands swapped (A-operand = W rows, B-operand = X rows) so that
//     each lane holds 4 consecutive output columns of one row;
//   * the epilogue stages the output tile through LDS and stores whole rows;
//   * the activation is a template parameter; bias and the pre-activation
//     output are uniform runtime flags.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void glb_void_t;

// Buffer load straight into LDS (buffer_load_dwordx4 ... lds): lane i's 16
// bytes land at M0 + 16 i.  The LLVM intrinsic has no clang builtin; it is
// bound by name.  A buffer resource = 48-bit base, byte range (loads past it
// return zero), gfx9 format word.  Per-lane 32-bit offsets stay fixed for the
// whole K loop; the K advance is the scalar offset.
typedef int i32x4_t __attribute__((ext_vector_type(4)));
__device__ void raw_buffer_load_lds(i32x4_t rsrc, __attribute__((address_space(3))) unsigned* lds,
                                    int size, int voffset, int soffset, int offset,
                                    int aux) __asm("llvm.amdgcn.raw.buffer.load.lds");
// The same load written as inline asm (M0 = LDS address, set by the
// compiler through the constraint).  The compiler's hazard recognizer does
// not see the vector-memory instruction inside the asm, so the asm covers the
// hazards of its scalar operands itself: a VMEM read of an SGPR that a VALU
// instruction wrote (v_readfirstlane / v_readlane into the resource words or
// the scalar offset) needs 5 wait states, and the M0 write one; s_nop 4
// provides 5.  (With s_nop 0 a build whose scheduler placed a
// v_readfirstlane of the resource base right before the asm ended in a GPU
// memory fault.)  PAD: the loads of a tile's first stages, which follow the
// resource set-up; the K loop's loads (scalar offsets from SALU adds) keep
// s_nop 0 for the M0 write, and a codegen test checks every asm load's wait
// states against the VALU writes before it.
// The compiler does not know that it writes LDS, so it adds no vmcnt wait in
// front of the LDS reads that follow it: it cannot prove that a transposing
// ds_read_b64_tr_b16 does not alias an in-flight direct-to-LDS load, and
// with the intrinsic it waits for all loads before every such read.  The
// kernel orders every LDS read of a stage after that stage's loads itself
// (s_waitcnt 0 + barrier at the top of each K-step).  The memory clobber
// keeps the loads in program order with the LDS reads.
template <bool PAD>
__device__ __forceinline__ void asm_buffer_load_lds(i32x4_t rsrc, uint32_t lds_addr, int voffset,
                                                    int soffset) {
  if constexpr (PAD)
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voffset), "s"(rsrc), "s"(soffset), "{m0}"(lds_addr)
                 : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voffset), "s"(rsrc), "s"(soffset), "{m0}"(lds_addr)
                 : "memory");
}
__device__ __forceinline__ i32x4_t buffer_rsrc(const void* base, uint32_t bytes) {
  struct __attribute__((packed)) Rsrc {
    const void* ptr;
    uint32_t range;
    uint32_t config;
  } r{base, bytes, 0x00020000u};
  i32x4_t v = __builtin_bit_cast(i32x4_t, r);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_readfirstlane(v[i]);
  return v;
}

struct NTParams {
  const void* A;      // K-contiguous [M, K] or M-contiguous [K, M], row stride lda (elements)
  const void* B;      // K-contiguous [N, K] or N-contiguous [K, N], row stride ldb (elements)
  void* C;            // [M, N], row stride ldc
  const void* bias;
  void* aux;
  int64_t lda, ldb, ldc, aux_ld;
  int M, N, K;
  int bias_f32;
  int tiles_m, tiles_n;
  GemmAdamW adam;  // ACT_ADAMW only
  float* colsum;   // see GemmParams::colsum
};

// Epilogue of the NT kernels.  Block (i, j) of the accumulators holds D[n][m]
// (MS x MS, see col_of below for the lane's elements).  The fragments go
// through LDS (`smem`, at least
// STAGE_BYTES, free when this is called) so that every global store, and the
// load of the dGELU pre-activation, moves whole 512-1024 byte rows.  LDS rows
// hold 16-byte chunks XOR-swizzled by row, which keeps both the fragment
// writes (32 rows, one chunk each) and the row reads bank-balanced.  A tile
// that does not fit (fp32 256x256) is done in passes over the wave's MS-row
// fragment groups.
template <int MS>
using nt_acc_t = typename std::conditional<MS == 16, floatx4, floatx16>::type;

template <int OUT, int ACT, int BM, int BN, int WM, int WN, int STAGE_BYTES, int MS>
__device__ __forceinline__ void nt_epilogue_staged(const NTParams& p,
                                                   nt_acc_t<MS> (&acc)[BN / WN / MS][BM / WM / MS],
                                                   uint8_t* smem, int m0, int n0) {
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / MS, TN = WTN / MS;
  // 32 x 32 blocks: lane (fr, fh) holds row fr, columns 8 g + 4 fh + {0..3}
  // in acc[..][4 g .. 4 g + 3] (g = 0..3); 16 x 16 blocks: row fr, columns
  // 4 fh + {0..3} in acc[0..3].
  constexpr int G = MS == 32 ? 4 : 1;
  // The lane's coordinates come from a thread index the compiler cannot see
  // through (see opaque_tid below): the LDS slots derived from them are then
  // computed here rather than hoisted out of the persistent tile loop and
  // spilled across the K loop.
  int tid_e = threadIdx.x;
  asm volatile("" : "+v"(tid_e));
  const int lane = tid_e & 63, wave = tid_e >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int fr = lane % MS, fh = lane / MS;
  auto col_of = [&](int i, int g) -> int { return wn * WTN + i * MS + (MS == 32 ? 8 * g + 4 * fh : 4 * fh); };
  constexpr int NT = 64 * NW;
  constexpr int OB = OUT == OUT_F32 ? 4 : 2;
  // Output stores with the nontemporal hint (no L2 allocation), except on
  // the persistent 8-wave 256 x 256 tiles.  Elsewhere workgroups reach their
  // epilogues at different times, and 128-256 KB of cached output per CU
  // evicts the operand panels the other workgroups of the XCD are still
  // streaming (8192 x 4096 x 11008: 506 -> 469 us, x 256: 24.9 -> 23.0 us,
  // 8192^3: 702 -> 688 us).  The persistent tiles finish their K loops
  // together, and there the train step's next GEMM finds the cached output
  // (its step ran 1.2% slower with nontemporal stores).
  constexpr bool NT_STORE = !(BM == 256 && BN == 256 && NW == 8);
  auto store16 = [&](void* dst, const u16x8& x) {
    if constexpr (NT_STORE)
      __builtin_nontemporal_store(x, reinterpret_cast<u16x8*>(dst));
    else
      *reinterpret_cast<u16x8*>(dst) = x;
  };
  constexpr int ROWB = BN * OB;    // bytes per staged row
  constexpr int CPR = ROWB / 16;   // 16-byte chunks per row
  // GELU stages the pre-activation z and the activation side by side (two
  // regions of half the staging bytes, so half the rows per pass): the
  // accumulators of a pass are dead once both are staged, and none are live
  // beside the copies of the other outputs.
  constexpr bool GELU_DUAL = ACT == ACT_GELU;
  constexpr int REGION = GELU_DUAL ? STAGE_BYTES / 2 : STAGE_BYTES;
  constexpr int ROWS_PASS = REGION / ROWB < BM ? REGION / ROWB : BM;
  constexpr int NPASS = BM / ROWS_PASS;
  constexpr int JP = TM / NPASS;   // MS-row fragment groups per wave per pass
  constexpr int WROWS = JP * MS;   // rows per wave per pass
  static_assert(NPASS * ROWS_PASS == BM && JP * NPASS == TM, "pass split");
  static_assert((CPR & (CPR - 1)) == 0 && (ROWS_PASS * CPR) % NT == 0, "chunk split");
  uint8_t* const tile = smem;

  // Bias of the lane's columns.  32 x 32 blocks: added to the accumulators
  // in place (8 floats per block).  16 x 16 blocks: the lane's 4 x TN bias
  // values are loaded once and added where each fragment is staged; an
  // in-place pass over 32 small accumulator blocks behind the runtime bias
  // test makes the compiler materialise all of them a second time and spill.
  constexpr bool HAS_BIAS_ACT = ACT != ACT_DGELU && ACT != ACT_ADAMW;
  const bool with_bias = HAS_BIAS_ACT && p.bias != nullptr;
  auto bias4 = [&](int i, int g, float* b) {
    const int n = n0 + col_of(i, g);
    if (p.bias_f32) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>((const float*)p.bias + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = bv[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = load_out<OUT>(p.bias, n + e);
    }
  };
  constexpr int BI = MS == 16 ? TN : 1;
  float bias_v[BI][4];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) bias_v[i][e] = 0.0f;
  if constexpr (HAS_BIAS_ACT) {
    if (with_bias) {
      if constexpr (MS == 16) {
#pragma unroll
        for (int i = 0; i < TN; ++i) bias4(i, 0, bias_v[i]);
      } else {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int g = 0; g < G; ++g) {
            float b[4];
            bias4(i, g, b);
#pragma unroll
            for (int j = 0; j < TM; ++j)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] += b[e];
          }
      }
    }
  }
  // accumulators of fragment (j, i, g), plus the bias for 16 x 16 blocks
  auto frag4 = [&](int j, int i, int g, float* v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e];
    if constexpr (MS == 16) {
      if (with_bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += bias_v[i][e];
      }
    }
  };

  // byte offset of this lane's 4 outputs of fragment (jj, i, g) in the tile
  auto slot = [&](int jj, int i, int g) -> int {
    const int pr = wm * WROWS + jj * MS + fr;
    const int cb = col_of(i, g) * OB;  // byte of the 4 outputs in the row
    const int c = cb / 16, half = cb % 16;
    return pr * ROWB + ((c ^ (pr & (CPR - 1))) * 16) + half;
  };
  auto put4 = [&](int off, const float* v) {
    if constexpr (OB == 4) {
      *reinterpret_cast<f32x4*>(tile + off) = f32x4{v[0], v[1], v[2], v[3]};
    } else if constexpr (OUT == OUT_BF16) {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      *reinterpret_cast<u32x2*>(tile + off) = u32x2{f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3])};
    } else {
      u16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = f32_to_f16(v[e]);
      *reinterpret_cast<u16x4*>(tile + off) = o;
    }
  };
  auto get4 = [&](int off, float* v) {
    if constexpr (OB == 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(tile + off);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = x[e];
    } else {
      const u16x4 x = *reinterpret_cast<const u16x4*>(tile + off);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = OUT == OUT_BF16 ? bf16_to_f32(x[e]) : f16_to_f32(x[e]);
    }
  };
  // global row of staged row pr in pass `pass`
  auto grow = [&](int pass, int pr) -> int64_t {
    return (int64_t)m0 + (pr / WROWS) * WTM + pass * WROWS + (pr % WROWS);
  };
  // The thread index as a value the compiler cannot see through: the
  // per-chunk offsets below are then computed here, in the epilogue.
  // Otherwise they are loop-invariant for the persistent tile loop, get
  // hoisted to the kernel start and spilled across the K loop, and each
  // reload's vmcnt(0) wait also waits for the memory operation issued just
  // before it, which serialises the epilogue's loads.
  auto opaque_tid = [&]() -> int {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  // tile rows of this pass -> global matrix (row stride ld elements)
  // (at most four 16-byte chunks in flight: the GELU epilogue calls this
  // with all accumulators live, and more in flight spill them)
  auto copy_out = [&](int pass, void* dst, int64_t ld, const uint8_t* src = nullptr) {
    const uint8_t* from = src ? src : tile;
    const int tid = opaque_tid();
#pragma unroll 4
    for (int k = 0; k < ROWS_PASS * CPR / NT; ++k) {
      const int idx = tid + k * NT;
      const int pr = idx / CPR, c = idx % CPR;
      const u16x8 x = *reinterpret_cast<const u16x8*>(from + pr * ROWB + ((c ^ (pr & (CPR - 1))) * 16));
      store16((uint8_t*)dst + (grow(pass, pr) * ld + n0) * OB + c * 16, x);
    }
  };
  // copy_out of the whole tile (bf16, 256 x 256, 8 waves) that also writes
  // the tile's column sums of the stored (bf16-rounded) values to row m0/256
  // of p.colsum.  A lane always handles the same 8-column chunk c = tid % 32,
  // rows tid / 32 + 16 k (k = 0..15, summed in that order); lanes l and l + 32
  // of a wave hold the same chunk and are added, then the 8 waves in order
  // through LDS.
  auto copy_out_colsum = [&]() {
    const int tid = opaque_tid();
    float cs[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) cs[e] = 0.0f;
#pragma unroll
    for (int k = 0; k < ROWS_PASS * CPR / NT; ++k) {
      const int idx = tid + k * NT;
      const int pr = idx / CPR, c = idx % CPR;
      const u16x8 x = *reinterpret_cast<const u16x8*>(tile + pr * ROWB + ((c ^ (pr & (CPR - 1))) * 16));
      store16((uint8_t*)p.C + (grow(0, pr) * p.ldc + n0) * OB + c * 16, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) cs[e] += bf16_to_f32(x[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) cs[e] += __shfl_xor(cs[e], 32, 64);
    __syncthreads();  // every lane has read its rows of the tile
    float* red = reinterpret_cast<float*>(tile);  // [8 waves][256 columns]
    const int w = tid >> 6, l = tid & 63;
    if (l < 32) {
#pragma unroll
      for (int e = 0; e < 8; ++e) red[w * BN + l * 8 + e] = cs[e];
    }
    __syncthreads();
    if (tid < BN) {
      float s = red[tid];
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) s += red[ww * BN + tid];
      p.colsum[(int64_t)(m0 / BM) * p.N + n0 + tid] = s;
    }
  };
  // global matrix -> tile rows of this pass, straight into LDS (no VGPRs:
  // the accumulators are live).  Wave instruction q fills the 1 KB at
  // tile + 1024 q, i.e. physical chunks idx = 64 q + lane; the lane fetches
  // the logical chunk stored there.
  auto copy_in = [&](int pass, const void* src, int64_t ld) {
    const int tid = opaque_tid();
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6), ln = tid & 63;
#pragma unroll
    for (int k = 0; k < ROWS_PASS * CPR / NT; ++k) {
      const int q = wave_id + k * NW;
      const int idx = q * 64 + ln;
      const int pr = idx / CPR, c = (idx % CPR) ^ (pr & (CPR - 1));
      __builtin_amdgcn_global_load_lds(
          (glb_void_t*)((const uint8_t*)src + (grow(pass, pr) * ld + n0) * OB + c * 16),
          (lds_void_t*)(tile + q * 1024), 16, 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0);
  };

  // ACT_ADAMW: the staged rows of this pass are the weight gradient; each
  // 16-byte chunk updates 4 weights (P, M, V read and written, bf16 shadow
  // written), row-contiguous like copy_out.
  auto adam_out = [&](int pass) {
    if constexpr (ACT == ACT_ADAMW) {
      const AdamWScalars sc = adamw_scalars(p.adam.step, p.adam.args);
      const int tid = opaque_tid();
#pragma unroll 4
      for (int k = 0; k < ROWS_PASS * CPR / NT; ++k) {
        const int idx = tid + k * NT;
        const int pr = idx / CPR, c = idx % CPR;
        const f32x4 g = *reinterpret_cast<const f32x4*>(tile + pr * ROWB + ((c ^ (pr & (CPR - 1))) * 16));
        const int64_t e = grow(pass, pr) * p.ldc + n0 + c * 4;
        f32x4 pp = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.adam.P + e));
        f32x4 mm = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.adam.M + e));
        f32x4 vv = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.adam.V + e));
        u16x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float pj = pp[j], mj = mm[j], vj = vv[j];
          adamw_elem(pj, g[j], mj, vj, sc, p.adam.args);
          pp[j] = pj;
          mm[j] = mj;
          vv[j] = vj;
          w[j] = f32_to_bf16(pj);
        }
        __builtin_nontemporal_store(pp, reinterpret_cast<f32x4*>(p.adam.P + e));
        __builtin_nontemporal_store(mm, reinterpret_cast<f32x4*>(p.adam.M + e));
        __builtin_nontemporal_store(vv, reinterpret_cast<f32x4*>(p.adam.V + e));
        __builtin_nontemporal_store(w, reinterpret_cast<u16x4*>(p.adam.Wb + e));
      }
    }
  };

#pragma unroll
  for (int pass = 0; pass < NPASS; ++pass) {
    if constexpr (ACT == ACT_DGELU) {
      copy_in(pass, p.aux, p.aux_ld);
      __syncthreads();
    }
    if constexpr (ACT == ACT_GELU && !GELU_DUAL) {
      if (p.aux) {  // pre-activation z
#pragma unroll
        for (int jj = 0; jj < JP; ++jj)
#pragma unroll
          for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int g = 0; g < G; ++g) {
              float v[4];
              frag4(pass * JP + jj, i, g, v);
              put4(slot(jj, i, g), v);
            }
        __syncthreads();
        copy_out(pass, p.aux, p.aux_ld);
        __syncthreads();
      }
    }
#pragma unroll
    for (int jj = 0; jj < JP; ++jj)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int off = slot(jj, i, g);
          float v[4];
          frag4(pass * JP + jj, i, g, v);
          if constexpr (ACT == ACT_DGELU) {
            float z[4];
            get4(off, z);  // this lane's own slot: no barrier between read and write
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= gelu_tanh_grad_f(z[e]);
          } else if constexpr (ACT == ACT_RELU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
          } else if constexpr (ACT == ACT_GELU) {
            if constexpr (GELU_DUAL) {
              if (p.aux) put4(REGION + off, v);  // pre-activation z
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f(v[e]);
          }
          put4(off, v);
        }
    __syncthreads();
    if constexpr (GELU_DUAL) {
      if (p.aux) copy_out(pass, p.aux, p.aux_ld, tile + REGION);
      copy_out(pass, p.C, p.ldc);
    } else if constexpr (ACT == ACT_ADAMW) {
      adam_out(pass);
    } else if constexpr (ACT == ACT_DGELU && OUT == OUT_BF16 && NPASS == 1 && CPR == 32 && NT == 512) {
      if (p.colsum)
        copy_out_colsum();
      else
        copy_out(pass, p.C, p.ldc);
    } else {  // (run_gemm sends column-sum launches to the branch above only)
      copy_out(pass, p.C, p.ldc);
    }
    if (pass + 1 < NPASS) __syncthreads();
  }
}

template <int V>
using template_int_t = std::integral_constant<int, V>;

// Schedule of one MFMA sub-step of the NT kernel: MFMA t is followed by its
// FPER fragments' LDS reads (front-loaded, so the last reads still have
// several MFMAs to land before the next sub-step needs them) and by its
// share of the NV loads, spread over the first LSPAN MFMAs (load u after
// MFMA t when t*NV/LSPAN <= u < (t+1)*NV/LSPAN).  sched_group_barrier masks:
// 0x008 MFMA, 0x100 DS read, 0x020 VMEM read.
template <int TM, int TN, int ES, bool AKC, bool BKC, int MS, int LSPAN>
struct NTSched {
  static constexpr int NMF = TM * TN * (ES == 4 ? 4 : 1);  // MFMAs per sub-step
  static_assert(LSPAN >= 1 && LSPAN <= NMF, "loads spread over the sub-step's MFMAs");
  static constexpr int load_lo(int t, int nv) { return t < LSPAN ? t * nv / LSPAN : nv; }
  static constexpr int NFR = TM + TN;                      // fragments per sub-step
  static constexpr int FPER = (NFR + NMF - 1) / NMF;       // fragments per MFMA
  // 16 x 16 blocks (RECYCLE): the MFMAs run A-fragment-major (t -> block
  // (t % TN, t / TN)) and the next sub-step's A fragment j is read into the
  // same registers right after its last MFMA (t = j TN + TN - 1), so only
  // the B fragments are double-buffered; the next B fragment t is read after
  // MFMA t.  Otherwise fragment r (A for r < TM, else B) after MFMA r / FPER.
  static constexpr bool RECYCLE = MS == 16;
  static constexpr int ds_instrs(int lo, int hi) {
    int n = 0;
    constexpr int MN_READS = ES == 4 ? 4 : 2;  // LDS reads of an M/N-contiguous fragment
    for (int r = lo; r < hi && r < NFR; ++r) n += r < TM ? (AKC ? 1 : MN_READS) : (BKC ? 1 : MN_READS);
    return n;
  }
  static constexpr int ds_after(int t) {
    if (!RECYCLE) return ds_instrs(t * FPER, (t + 1) * FPER);
    return (t < TN ? (BKC ? 1 : 2) : 0) + (t % TN == TN - 1 ? (AKC ? 1 : 2) : 0);
  }
  template <bool R, int NV, int T>
  static __device__ __forceinline__ void step() {
    constexpr int nds = R ? ds_after(T) : 0;
    constexpr int vlo = load_lo(T, NV), vhi = load_lo(T + 1, NV);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (nds > 0) __builtin_amdgcn_sched_group_barrier(0x100, nds, 0);
    if constexpr (vhi > vlo) __builtin_amdgcn_sched_group_barrier(0x020, vhi - vlo, 0);
  }
  template <bool R, int NV, int... T>
  static __device__ __forceinline__ void seq(std::integer_sequence<int, T...>) {
    (step<R, NV, T>(), ...);
  }
  template <bool R, int NV>
  static __device__ __forceinline__ void pin() {
    seq<R, NV>(std::make_integer_sequence<int, NMF>{});
  }
};

// One operand of the NT kernel: BMN rows (the M or N dimension) x BK = 64
// K-elements per stage.
//   KC (K-contiguous, memory [MN][K] with row stride ld): 1 KB LDS blocks of
//     8 MN-rows x 64 K (128 B per row); row r keeps logical 16-byte chunk c
//     at physical chunk c ^ ((r >> 1) & 7), so the 32-row ds_read_b128
//     fragment reads hit all 64 banks.  Slot `lane` of block j is row
//     8j + lane/8, physical chunk lane%8.
//   MN-contiguous (memory [K][MN] with row stride ld): 64 K-rows of BMN
//     elements; row k keeps logical chunk c (8 MN-elements) at physical chunk
//     c ^ nt_mn_swizzle(k).  A fragment (MS MN x 16 or 32 K) is two
//     ds_read_b64_tr_b16 per 16-lane group: lane j points at row k0 + j/4,
//     elements m + 4 (j%4) .. +3, and the transposing read hands lane i the
//     four K values of element m + i.
//   K-contiguous rows are 128 B: the chunk c ^ ((r >> 1) & 7) keeps the 32
//     (or 16) rows of one fragment read on all 64 banks.
// Loads are buffer loads straight into LDS with per-lane offsets fixed for
// the whole K loop (the K advance is the scalar offset); the host checks that
// the bytes a resource spans fit a signed 32-bit offset.
template <bool KC, int BMN, int NW, int ES>
struct NTOperand {
  static constexpr int BYTES = BMN * 128;            // a stage holds 128 B of K per row
  static constexpr int BLOCKS = BYTES / 1024 / NW;   // 1 KB load blocks per wave
  static constexpr int ROWB = BMN * ES;              // MN-contiguous row bytes
  static constexpr int CPR = ROWB / 16;              // chunks per MN-contiguous row
  static_assert(BYTES % (1024 * NW) == 0, "load blocks must split evenly over waves");
  static_assert(KC || CPR >= 16 || (ES == 2 && CPR == 8), "MN-contiguous tiles: >= 16 chunks per row, or 8 (16-bit)");

  i32x4_t rsrc;
  int voff[BLOCKS];
  int soff_step;  // scalar byte offset per K-step
};

template <bool KC, int BMN, int NW, int ES, int MS>
__device__ __forceinline__ void nt_operand_init(NTOperand<KC, BMN, NW, ES>& o, const void* X, int64_t ld,
                                                int mn0, int K, int lane, int wave) {
  const uint8_t* Xb = static_cast<const uint8_t*>(X);
  if constexpr (KC) {
    o.rsrc = buffer_rsrc(Xb + (int64_t)mn0 * ld * ES, (uint32_t)((int64_t)BMN * ld * ES));
    const int r_in = lane >> 3;
    const int cl_even = (lane & 7) ^ (r_in >> 1);
    const int cl_odd = (lane & 7) ^ ((4 + (r_in >> 1)) & 7);
#pragma unroll
    for (int t = 0; t < o.BLOCKS; ++t) {
      const int j = wave + t * NW;
      o.voff[t] = (j * 8 + r_in) * (int)ld * ES + ((j & 1) ? cl_odd : cl_even) * 16;
    }
    o.soff_step = 128;
  } else {
    constexpr int CPR = NTOperand<KC, BMN, NW, ES>::CPR;
    constexpr int RPB = 64 / CPR;  // rows per 1 KB block
    o.rsrc = buffer_rsrc(Xb + (int64_t)mn0 * ES, (uint32_t)((int64_t)K * ld * ES));
#pragma unroll
    for (int t = 0; t < o.BLOCKS; ++t) {
      const int q = wave + t * NW;
      const int k = q * RPB + lane / CPR;
      const int c = (lane % CPR) ^ nt_mn_swizzle<MS, ES, CPR>(k);
      o.voff[t] = k * (int)ld * ES + c * 16;
    }
    o.soff_step = 128 * (int)ld;  // 128 / ES K-rows per stage
  }
}

// Persistent tiles (one workgroup per CU looping over tiles) for the 8-wave
// 256 x 256 configuration; the 4-wave one keeps one tile per workgroup: its
// 256 accumulators per lane leave no room for the registers that a tile loop
// carries through the epilogue (they spill to scratch and cost more than the
// overlap gains).
constexpr bool nt_persistent(int BM, int BN, int WM, int WN) {
  return BM == 256 && BN == 256 && WM * WN == 8;
}

// s_waitcnt immediate for vmcnt(n), lgkmcnt(0), expcnt left alone (gfx9
// layout: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (((N >> 4) & 0x3) << 14));
}

// Workgroup barrier without the vmcnt(0) the compiler puts in front of
// __syncthreads (its release fence waits for every load in flight, which
// would drain a pipeline of more than two stages); the "memory" clobber
// keeps the compiler from moving memory accesses across it.  The caller
// waits right before for what the barrier publishes (its own loads of the
// next stage, its LDS reads of the stage about to be refilled).
__device__ __forceinline__ void barrier_keep_loads() { asm volatile("s_barrier" ::: "memory"); }

// S: LDS stages.  Two for the large tiles (their K-step's MFMA work covers a
// load's latency); small tiles, whose K-step is a few hundred cycles of MFMA
// work, keep S - 1 K-steps of loads in flight.
template <int IN, int OUT, int ACT, int BM, int BN, int WM, int WN, bool AKC, bool BKC, int S = 2>
__global__ __launch_bounds__(64 * WM * WN) void gemm_nt_kernel(NTParams p) {
  static_assert(S == 2 || S == 4 || S == 8, "stages: 2, 4 or 8");
  constexpr int ES = IN == IN_F32 ? 4 : 2;  // element bytes
  // MFMA block: 16 x 16 x 32 for 16-bit operands, 32 x 32 x 2 for fp32
  constexpr int MS = ES == 2 ? 16 : 32;
  constexpr int KS = MS == 16 ? 2 : 4;  // MFMA sub-steps per K-step
  constexpr int CPS = 64 / MS;          // 16-byte chunks of a 128-byte K-row per sub-step
  constexpr int KPS = ES == 4 ? 8 : 16 * CPS / 2;  // K-rows of an MN-contiguous stage per sub-step
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / MS, TN = WTN / MS;
  constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128;  // 128 B of K per row and stage
  constexpr int STAGE = A_BYTES + B_BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[S * STAGE];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  int m0 = 0, n0 = 0;
  NTOperand<AKC, BM, NW, ES> opa;
  NTOperand<BKC, BN, NW, ES> opb;

  // Load u of the wave for K-step kt into stage `stage`: 1 KB direct-to-LDS
  // block u (A blocks first).  With an M/N-contiguous operand the loads are
  // issued as inline asm (no compiler waits in front of the transposing
  // reads); K-contiguous kernels use the intrinsic, which the scheduler
  // places by itself.
  constexpr bool ASM_LDS = !(AKC && BKC);
  constexpr int NVM = opa.BLOCKS + opb.BLOCKS;  // loads per wave and K-step
  auto load_one = [&](int kt, int stage, int u, auto PAD) {
    uint8_t* base = smem + stage * STAGE;
    const bool is_a = u < opa.BLOCKS;
    uint8_t* dst = is_a ? base + (wave_s + u * NW) * 1024 : base + A_BYTES + (wave_s + (u - opa.BLOCKS) * NW) * 1024;
    const i32x4_t rsrc = is_a ? opa.rsrc : opb.rsrc;
    const int voff = is_a ? opa.voff[u] : opb.voff[u - opa.BLOCKS];
    const int soff = kt * (is_a ? opa.soff_step : opb.soff_step);
    if constexpr (ASM_LDS)
      asm_buffer_load_lds<decltype(PAD)::value>(rsrc, (uint32_t)(uintptr_t)dst, voff, soff);
    else
      raw_buffer_load_lds(rsrc, (__attribute__((address_space(3))) unsigned*)dst, 16, voff, soff, 0, 0);
  };
  auto issue_loads = [&](int kt, int stage) {
#pragma unroll
    for (int u = 0; u < NVM; ++u) load_one(kt, stage, u, std::true_type{});
  };

  nt_acc_t<MS> acc[TN][TM];

  // Fragment addresses.  K-contiguous: row offset of the lane's MN-row plus
  // the swizzled chunk of (sub-step, lane group).  MN-contiguous: the lane's
  // K-row within a sub-step and its swizzled column bytes (loop invariant).
  // A lane of an MS x MS block holds MN-row fr and K chunk fh of the
  // sub-step (8 K per 16-byte chunk).
  const int fr = lane % MS, fh = lane / MS;
  const int rsw = (fr >> 1) & 7;  // fragment rows start at multiples of MS
  const int g16 = (lane >> 4) & 3, i16 = lane & 15;
  // 32 x 32: groups 0/1 take MN + 0/16 of K-rows 0-7, groups 2/3 K-rows
  // 8-15; 16 x 16: group g takes K-rows 8 g .. 8 g + 7 of the same 16 MN
  const int tr_row = MS == 32 ? (8 * (g16 >> 1) + (i16 >> 2)) : (8 * g16 + (i16 >> 2));
  // byte offset of the lane's 8-byte piece in a K-row of `cpr` chunks
  auto tr_col = [&](int mb, auto CPR_) {
    constexpr int cpr = decltype(CPR_)::value;
    if constexpr (MS == 32)
      return ((((mb >> 3) ^ (4 * ((i16 >> 2) & 3))) + 2 * (g16 & 1) + ((i16 >> 1) & 1)) * 16) + 8 * (i16 & 1);
    else
      return ((((mb >> 3) ^ nt_mn_swizzle<MS, 2, cpr>(tr_row)) + ((i16 >> 1) & 1)) * 16) + 8 * (i16 & 1);
  };
  // fp32 M/N-contiguous: lane (fr, fh) holds element mb + fr of K-rows
  // 4 fh .. 4 fh + 3 of the sub-step (four 4-byte reads, one per K-row);
  // the row swizzle of those rows is 8 fh
  auto mn32_off = [&](int mb, int rowb) {
    const int m = mb + fr;
    return 4 * fh * rowb + (((m >> 2) ^ (8 * fh)) * 16) + (m & 3) * 4;
  };
  int a_off[TM], b_off[TN];
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int mb = wm * WTM + j * MS;
    if constexpr (AKC) a_off[j] = (mb + fr) * 128;
    else a_off[j] = ES == 4 ? mn32_off(mb, BM * ES) : tr_row * (BM * 2) + tr_col(mb, template_int_t<BM * 2 / 16>{});
  }
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int nb = wn * WTN + i * MS;
    if constexpr (BKC) b_off[i] = A_BYTES + (nb + fr) * 128;
    else b_off[i] = A_BYTES + (ES == 4 ? mn32_off(nb, BN * ES) : tr_row * (BN * 2) + tr_col(nb, template_int_t<BN * 2 / 16>{}));
  }

  typedef short v4i16 __attribute__((ext_vector_type(4)));
  auto tr_frag = [&](const uint8_t* addr, int rowb) -> u16x8 {
    if constexpr (ES == 4) {  // fp32: four K-rows, one float each
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const float*>(addr + e * rowb);
      return __builtin_bit_cast(u16x8, v);
    } else {
      const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)addr);
      const v4i16 hi =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)(addr + 4 * rowb));
      u16x8 f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[e] = (uint16_t)lo[e];
        f[e + 4] = (uint16_t)hi[e];
      }
      return f;
    }
  };

  u16x8 fa[2][TM], fb[2][TN];
  auto read_frags = [&](const uint8_t* st, int kk, int buf) {
    const int chunk = ((kk * CPS + fh) ^ rsw) * 16;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int ab = MS == 16 ? 0 : buf;
      if constexpr (AKC) fa[ab][j] = *reinterpret_cast<const u16x8*>(st + a_off[j] + chunk);
      else fa[ab][j] = tr_frag(st + a_off[j] + kk * KPS * (BM * ES), BM * ES);
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      if constexpr (BKC) fb[buf][i] = *reinterpret_cast<const u16x8*>(st + b_off[i] + chunk);
      else fb[buf][i] = tr_frag(st + b_off[i] + kk * KPS * (BN * ES), BN * ES);
    }
  };
  // Single operations of the pipeline, emitted one by one in the order the
  // schedule below pins (the compiler keeps LDS-writing loads and LDS reads
  // in program order, so the order has to be written out).
  //   fragment f: f < TM is A fragment f, else B fragment f - TM (one
  //     ds_read_b128, or two ds_read_b64_tr_b16 for an M/N-contiguous tile);
  //     with RECYCLE (NTSched) the A fragments use register set 0 only;
  //   MFMA t: block (i, j) = (t / TM % TN, t % TM), or (t % TN, t / TN) with
  //     RECYCLE; fp32 runs 4 MFMAs per block and sub-step, t / (TM * TN)
  //     selecting the fragment element;
  //   load u: 1 KB direct-to-LDS block u of the wave (A blocks first).
  // The 8-wave tiles with 16-bit operands spread a K-step's loads over the
  // first 3/4 of the first sub-step's MFMAs, the others over all of them
  // (step 2.85 -> 2.79 ms, same bits; spans of 5/8 and 7/8, a later start,
  // or loads in both sub-steps were slower, and 3/4 on the 4-wave tiles
  // slowed 8192^3).
  constexpr int NMF_ = TM * TN * (ES == 4 ? 4 : 1);
  using Sched = NTSched<TM, TN, ES, AKC, BKC, MS, NW == 8 && ES == 2 ? NMF_ * 3 / 4 : NMF_>;
  constexpr bool RECYCLE = Sched::RECYCLE;
  auto read_one = [&](const uint8_t* st, int kk, int buf, int f) {
    const int chunk = ((kk * CPS + fh) ^ rsw) * 16;
    if (f < TM) {
      const int ab = RECYCLE ? 0 : buf;
      if constexpr (AKC) fa[ab][f] = *reinterpret_cast<const u16x8*>(st + a_off[f] + chunk);
      else fa[ab][f] = tr_frag(st + a_off[f] + kk * KPS * (BM * ES), BM * ES);
    } else {
      const int i = f - TM;
      if constexpr (BKC) fb[buf][i] = *reinterpret_cast<const u16x8*>(st + b_off[i] + chunk);
      else fb[buf][i] = tr_frag(st + b_off[i] + kk * KPS * (BN * ES), BN * ES);
    }
  };
  auto mfma_one = [&](int buf, int t) {
    const int i = RECYCLE ? t % TN : (t / TM) % TN, j = RECYCLE ? t / TN : t % TM;
    if constexpr (MS == 16) {
      acc[i][j] = mfma16<IN>(reinterpret_cast<const uint16_t*>(&fb[buf][i]),
                             reinterpret_cast<const uint16_t*>(&fa[0][j]), acc[i][j]);
    } else if constexpr (ES == 2) {
      acc[i][j] = mfma32<IN>(reinterpret_cast<const uint16_t*>(&fb[buf][i]),
                             reinterpret_cast<const uint16_t*>(&fa[buf][j]), acc[i][j]);
    } else {
      const int e = t / (TM * TN);
      const float a = reinterpret_cast<const float*>(&fb[buf][i])[e];
      const float b = reinterpret_cast<const float*>(&fa[buf][j])[e];
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i][j], 0, 0, 0);
    }
  };
  constexpr int NMF = Sched::NMF, NFR = Sched::NFR, FPER = Sched::FPER;
  // One sub-step: the MFMAs on fragment buffer `buf`; when R, the fragments
  // of sub-step rkk of stage `rst` into buffer rbuf (front-loaded, FPER per
  // MFMA); loads [VLO, VHI) of K-step lkt into stage lst, spread evenly.
  auto substep = [&](auto R, auto VLO, auto VHI, int buf, const uint8_t* rst, int rkk, int rbuf, int lkt,
                     int lst) {
    constexpr int vlo = decltype(VLO)::value, vhi = decltype(VHI)::value, nv = vhi - vlo;
#pragma unroll
    for (int t = 0; t < NMF; ++t) {
      mfma_one(buf, t);
      if constexpr (decltype(R)::value) {
        if constexpr (RECYCLE) {
          if (t < TN) read_one(rst, rkk, rbuf, TM + t);
          if (t % TN == TN - 1) read_one(rst, rkk, rbuf, t / TN);
        } else {
#pragma unroll
          for (int q = 0; q < FPER; ++q)
            if (t * FPER + q < NFR) read_one(rst, rkk, rbuf, t * FPER + q);
        }
      }
      if constexpr (nv > 0) {
#pragma unroll
        for (int u = vlo + Sched::load_lo(t, nv); u < vlo + Sched::load_lo(t + 1, nv); ++u)
          load_one(lkt, lst, u, std::false_type{});
      }
    }
    Sched::template pin<decltype(R)::value, ASM_LDS ? 0 : nv>();  // asm loads are in no sched group
  };
  using Rd = std::true_type;
  using NoRd = std::false_type;
  template_int_t<0> z;

  // Pipeline.  A K-step (128 bytes of K per row) has KS sub-steps (four of
  // 32 x 32 x 16 or 32 x 32 x 2 MFMAs, or two of 16 x 16 x 32); the
  // fragments of sub-step s+1 are read during the MFMAs of sub-step s, from
  // two register sets.  The body of the K loop starts with the K-step's only
  // barrier: after it the stage of K-step kt+1 is visible to every wave and
  // the stage of K-step kt is read by none, so the loads of K-step kt+2
  // refill it.  The body then runs the last sub-step of kt (its fragments are
  // already in registers) and the other sub-steps of kt+1, with the loads of
  // kt+2 spread over the first half of the body: issued all at once after the
  // barrier they back up the address queue and stall the MFMA issue, and
  // issued later they have too little time left before the next wait.
  // Tiles: the grid covers all tiles (one per workgroup), or, persistent,
  // one workgroup per CU loops over tiles blockIdx.x + q * gridDim.x, so that
  // the global stores of a tile's epilogue drain while the next tile's loads
  // and MFMAs run.  With a grid that is a multiple of 8, tile % 8 is the
  // workgroup's XCD, as the remap in tile_coords_of assumes.
  const int total_tiles = p.tiles_m * p.tiles_n;
  constexpr bool PERSIST = nt_persistent(BM, BN, WM, WN);
  for (int tile = blockIdx.x; tile < total_tiles; tile += gridDim.x) {
  {
    int tm_i, tn_i;
    tile_coords_of(tile, p.tiles_m, p.tiles_n, tm_i, tn_i);
    m0 = tm_i * BM;
    n0 = tn_i * BN;
    if constexpr (ACT != ACT_ADAMW) {
      // A last tile that would pass M or N is moved back to end there: it
      // computes rows or columns of its neighbour again, with the same bits
      // (an output's K order does not depend on its place in a tile).
      m0 = m0 < p.M - BM ? m0 : p.M - BM;
      n0 = n0 < p.N - BN ? n0 : p.N - BN;
    }
  }
  nt_operand_init<AKC, BM, NW, ES, MS>(opa, p.A, p.lda, m0, p.K, lane, wave);
  nt_operand_init<BKC, BN, NW, ES, MS>(opb, p.B, p.ldb, n0, p.K, lane, wave);
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int r = 0; r < (MS == 16 ? 4 : 16); ++r) acc[i][j][r] = 0.0f;

  const int nk = p.K / (128 / ES);
  constexpr int L1 = NVM / 2;  // with four sub-steps: loads in the first of the two
  // Wait until at most n K-steps of this wave's loads are in flight (and its
  // fragment reads are done); n < S - 1.
  auto wait_steps = [&](int n) {
    if constexpr (S > 2) {
      if (n >= 6) { wait_vm_lgkm0<6 * NVM>(); return; }
      if (n == 5) { wait_vm_lgkm0<5 * NVM>(); return; }
      if (n == 4) { wait_vm_lgkm0<4 * NVM>(); return; }
      if (n == 3) { wait_vm_lgkm0<3 * NVM>(); return; }
      if (n == 2) { wait_vm_lgkm0<2 * NVM>(); return; }
      if (n == 1) { wait_vm_lgkm0<NVM>(); return; }
    }
    __builtin_amdgcn_s_waitcnt(0);
  };
  issue_loads(0, 0);
  if constexpr (S > 2) {
    // K-steps 1 .. S - 2 go out before the first wait
    for (int q = 1; q < S - 1 && q < nk; ++q) issue_loads(q, q);
    wait_steps((nk - 1 < S - 2 ? nk - 1 : S - 2));
    barrier_keep_loads();
  } else {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (S - 1 < nk) issue_loads(S - 1, S - 1);
  read_frags(smem, 0, 0);
  if constexpr (KS == 4) {
    substep(Rd{}, z, z, 0, smem, 1, 1, 0, 0);
    substep(Rd{}, z, z, 1, smem, 2, 0, 0, 0);
    substep(Rd{}, z, z, 0, smem, 3, 1, 0, 0);
  } else {
    substep(Rd{}, z, z, 0, smem, 1, 1, 0, 0);
  }
  int kt = 0;
  for (; kt + S < nk; ++kt) {
    // own loads of K-step kt+1 and fragment reads done; K-steps kt+2 ..
    // kt+S-1 may still be in flight
    if constexpr (S > 2) {
      wait_vm_lgkm0<(S - 2) * NVM>();
      barrier_keep_loads();
    } else {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
    const uint8_t* nx = smem + ((kt + 1) % S) * STAGE;
    const int ls = kt % S;  // the stage of K-step kt, free after the barrier, takes K-step kt+S
    if constexpr (KS == 4) {
      substep(Rd{}, z, template_int_t<L1>{}, 1, nx, 0, 0, kt + S, ls);
      substep(Rd{}, template_int_t<L1>{}, template_int_t<NVM>{}, 0, nx, 1, 1, kt + S, ls);
      substep(Rd{}, z, z, 1, nx, 2, 0, 0, 0);
      substep(Rd{}, z, z, 0, nx, 3, 1, 0, 0);
    } else {
      // two sub-steps of twice the MFMAs: the loads of K-step kt+S over the first
      substep(Rd{}, z, template_int_t<NVM>{}, 1, nx, 0, 0, kt + S, ls);
      substep(Rd{}, z, z, 0, nx, 1, 1, 0, 0);
    }
  }
  if constexpr (S > 2) {
    for (; kt + 2 < nk; ++kt) {  // nothing left to load: K-steps kt+2 .. nk-1 in flight
      wait_steps(nk - 2 - kt);
      barrier_keep_loads();
      const uint8_t* nx = smem + ((kt + 1) % S) * STAGE;
      if constexpr (KS == 4) {
        substep(Rd{}, z, z, 1, nx, 0, 0, 0, 0);
        substep(Rd{}, z, z, 0, nx, 1, 1, 0, 0);
        substep(Rd{}, z, z, 1, nx, 2, 0, 0, 0);
        substep(Rd{}, z, z, 0, nx, 3, 1, 0, 0);
      } else {
        substep(Rd{}, z, z, 1, nx, 0, 0, 0, 0);
        substep(Rd{}, z, z, 0, nx, 1, 1, 0, 0);
      }
    }
  }
  if constexpr (ASM_LDS) {
    // The asm loads are hidden from the compiler's hazard tracking: once the
    // loop has issued its last one, their lane offsets are dead to it and
    // their registers could be reused while those loads are in flight.  Wait
    // for them here and keep the offsets live up to this point.
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int t = 0; t < opa.BLOCKS; ++t) asm volatile("" ::"v"(opa.voff[t]));
#pragma unroll
    for (int t = 0; t < opb.BLOCKS; ++t) asm volatile("" ::"v"(opb.voff[t]));
  }
  if (kt + 1 < nk) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const uint8_t* nx = smem + ((kt + 1) % S) * STAGE;
    if constexpr (KS == 4) {
      substep(Rd{}, z, z, 1, nx, 0, 0, 0, 0);
      substep(Rd{}, z, z, 0, nx, 1, 1, 0, 0);
      substep(Rd{}, z, z, 1, nx, 2, 0, 0, 0);
      substep(Rd{}, z, z, 0, nx, 3, 1, 0, 0);
    } else {
      substep(Rd{}, z, z, 1, nx, 0, 0, 0, 0);
      substep(Rd{}, z, z, 0, nx, 1, 1, 0, 0);
    }
  }
  substep(NoRd{}, z, z, 1, nullptr, 0, 0, 0, 0);

  __syncthreads();  // every wave is done reading the last stage
  nt_epilogue_staged<OUT, ACT, BM, BN, WM, WN, 2 * STAGE, MS>(p, acc, smem, m0, n0);
  if constexpr (!PERSIST) break;  // one tile per workgroup: no loop-carried registers
  __syncthreads();  // the staged tile is read out before the next tile's loads refill the stages
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct View2D {
  const void* data;
  int64_t rows, cols, rs, cs;
};

View2D view2d(const TensorDesc& t, bool trans) {
  if (!trans) return {t.data, t.shape[0], t.shape[1], t.stride[0], t.stride[1]};
  return {t.data, t.shape[1], t.shape[0], t.stride[1], t.stride[0]};
}

bool stride_valid_2d(const TensorDesc& t) {
  return t.rank == 2 && t.stride[0] > 0 && t.stride[1] > 0;
}

// gemm/launcher.cu:48-70
void read_gemm_attr(const void* attr, bool* ta, bool* tb) {
  *ta = *tb = false;
  const AttrBlob& a = blob(attr);
  if (!attr) return;
  if (a.schema_id != 0 && a.schema_id != AICF_SCHEMA_GEMM) return;
  if (!payload_ok(a, 8)) return;
  *ta = field<int32_t>(a, 0) != 0;
  *tb = field<int32_t>(a, 4) != 0;
}

// Epilogue attributes: GPEL <iii> (transA, transB, relu; relu default 1,
// gemm_epilogue/launcher.cu:57-80) or GEPI <iii> (transA, transB, kind).
struct EpiAttr {
  bool ta = false, tb = false;
  int kind = AICF_EPI_BIAS_RELU;
};
EpiAttr read_epi_attr(const void* attr) {
  EpiAttr e;
  const AttrBlob& a = blob(attr);
  if (!attr) return e;
  if (a.schema_id == AICF_SCHEMA_GEPI) {
    if (!payload_ok(a, 12)) return e;
    e.ta = field<int32_t>(a, 0) != 0;
    e.tb = field<int32_t>(a, 4) != 0;
    e.kind = field<int32_t>(a, 8);
    return e;
  }
  if (a.schema_id != 0 && a.schema_id != AICF_SCHEMA_GPEL) return e;
  if (!payload_ok(a, 12)) return e;
  e.ta = field<int32_t>(a, 0) != 0;
  e.tb = field<int32_t>(a, 4) != 0;
  e.kind = field<int32_t>(a, 8) != 0 ? AICF_EPI_BIAS_RELU : AICF_EPI_BIAS;
  return e;
}

bool epi_kind_valid(int k) { return k >= AICF_EPI_BIAS_RELU && k <= AICF_EPI_DGELU_PARTIALS; }

// gemm/launcher.cu:116-148: A[M,K] . B[K,N] -> C[M,N] with positive strides.
bool gemm_views_ok(const TensorDesc& A0, const TensorDesc& B0, const TensorDesc& C0, bool ta,
                   bool tb) {
  if (A0.rank != 2 || B0.rank != 2 || C0.rank != 2) return false;
  if (!stride_valid_2d(A0) || !stride_valid_2d(B0) || !stride_valid_2d(C0)) return false;
  const View2D A = view2d(A0, ta), B = view2d(B0, tb), C = view2d(C0, false);
  const int64_t M = A.rows, K = A.cols, N = B.cols;
  if (M <= 0 || N <= 0 || K <= 0) return false;
  if (B.rows != K || C.rows != M || C.cols != N) return false;
  if (M > INT32_MAX / 2 || N > INT32_MAX / 2) return false;
  return true;
}

int load_mode(int64_t rs_rows, int64_t cs_k) {
  if (cs_k == 1) return LD_KCONTIG;
  if (rs_rows == 1) return LD_MNCONTIG;
  return LD_GATHER;
}

template <int IN, int OUT, int BM, int BN, int BK, int WM, int WN>
Status run_cfg(GemmParams& p, hipStream_t s) {
  p.tiles_m = (int)((p.M + BM - 1) / BM);
  p.tiles_n = (int)((p.N + BN - 1) / BN);
  const int64_t total = (int64_t)p.tiles_m * p.tiles_n;
  if (total > INT32_MAX) return Status::InvalidArgument;
  gemm_mfma_kernel<IN, OUT, BM, BN, BK, WM, WN><<<(unsigned)total, 64 * WM * WN, 0, s>>>(p);
  return launch_status("gemm_mfma");
}

// Compute units of the current device (cached per device; 0 if unknown).
int device_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cached[dev] = n;
  }
  return cached[dev];
}

template <int IN, int OUT, int ACT, int BM, int BN, int WM, int WN, bool AKC, bool BKC, int S = 2>
Status run_nt_act(const GemmParams& g, hipStream_t s) {
  NTParams p{};
  p.A = g.A;
  p.B = g.B;
  p.C = g.C;
  p.bias = g.bias;
  p.aux = g.aux;
  p.lda = AKC ? g.a_rs : g.a_cs;  // memory row stride of A ([M][K] or [K][M])
  p.ldb = BKC ? g.b_cs : g.b_rs;  // memory row stride of B ([N][K] or [K][N])
  p.ldc = g.c_rs;
  p.aux_ld = g.aux_rs;
  p.M = (int)g.M;
  p.N = (int)g.N;
  p.K = (int)g.K;
  p.bias_f32 = g.bias_f32;
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  p.adam = g.adam;
  p.colsum = g.colsum;
  // 256 x 256 tiles hold one workgroup per CU: with more tiles than CUs, the
  // persistent configuration launches one workgroup per CU (a multiple of 8,
  // one per XCD slot) that loops over its tiles.
  unsigned grid = (unsigned)(p.tiles_m * p.tiles_n);
  if constexpr (nt_persistent(BM, BN, WM, WN)) {
    const int ncu = device_cu_count();
    if (ncu > 0 && ncu % 8 == 0 && grid > (unsigned)ncu) grid = (unsigned)ncu;
  }
  gemm_nt_kernel<IN, OUT, ACT, BM, BN, WM, WN, AKC, BKC, S><<<grid, 64 * WM * WN, 0, s>>>(p);
  return launch_status("gemm_nt");
}

template <int IN, int OUT, int BM, int BN, int WM, int WN, bool AKC, bool BKC, int S = 2>
Status run_nt_layout(const GemmParams& g, hipStream_t s) {
  switch (g.act) {
    case ACT_RELU: return run_nt_act<IN, OUT, ACT_RELU, BM, BN, WM, WN, AKC, BKC, S>(g, s);
    case ACT_GELU: return run_nt_act<IN, OUT, ACT_GELU, BM, BN, WM, WN, AKC, BKC, S>(g, s);
    case ACT_DGELU: return run_nt_act<IN, OUT, ACT_DGELU, BM, BN, WM, WN, AKC, BKC, S>(g, s);
    case ACT_ADAMW:
      if constexpr (IN == IN_BF16 && OUT == OUT_F32)
        return run_nt_act<IN, OUT, ACT_ADAMW, BM, BN, WM, WN, AKC, BKC, S>(g, s);
      return Status::Internal;  // fused AdamW takes bf16 operands and an fp32 gradient
    default: return run_nt_act<IN, OUT, ACT_NONE, BM, BN, WM, WN, AKC, BKC, S>(g, s);
  }
}

// Operand layouts: K-contiguous ([MN][K]) on every tile configuration;
// MN-contiguous ([K][MN], read through the transposing LDS loads for 16-bit
// operands, one 4-byte read per K-row for fp32) where MN_OK (rows of at
// least 16 chunks: 256 x 256 and 128 x 128, and 64 x 64 for fp32).
template <int IN, int OUT, int BM, int BN, int WM, int WN, bool MN_OK, int S = 2>
Status run_nt(const GemmParams& g, hipStream_t s) {
  const bool akc = g.a_mode == LD_KCONTIG, bkc = g.b_mode == LD_KCONTIG;
  if (akc && bkc) return run_nt_layout<IN, OUT, BM, BN, WM, WN, true, true, S>(g, s);
  if constexpr (MN_OK) {
    if (akc) return run_nt_layout<IN, OUT, BM, BN, WM, WN, true, false, S>(g, s);
    if (bkc) return run_nt_layout<IN, OUT, BM, BN, WM, WN, false, true, S>(g, s);
    return run_nt_layout<IN, OUT, BM, BN, WM, WN, false, false, S>(g, s);
  }
  return Status::Internal;  // excluded by nt_eligible
}

// 256 x 256 tiles.  bf16 with K-contiguous operands and a one-output
// epilogue (none, ReLU, GELU): four waves of 128 x 128, one per SIMD, which
// issue the MFMAs back to back.  Everything else: eight waves of 128 x 64; the
// GELU (two outputs) and dGELU (pre-activation read) epilogues move twice
// the bytes per wave with four waves.  f16 keeps eight: four take 4% less on
// several rounds of long K (8192^3 770 us, 740) but 6-9% more at K <= 1024
// (8192 x 4096 x 1024 61.2, 65.1, with GELU 69.6, 75.0).
template <int IN, int OUT>
Status run_nt256(const GemmParams& g, hipStream_t s) {
  if constexpr (IN == IN_BF16) {
    if (g.a_mode == LD_KCONTIG && g.b_mode == LD_KCONTIG) {
      if (g.act == ACT_NONE) return run_nt_act<IN, OUT, ACT_NONE, 256, 256, 2, 2, true, true>(g, s);
      if (g.act == ACT_RELU) return run_nt_act<IN, OUT, ACT_RELU, 256, 256, 2, 2, true, true>(g, s);
      // bias+GELU without the pre-activation output: 8192^3 757 vs 810 us,
      // 8192 x 4096 x 11008 535 vs 559 (same bits); with it the two
      // configurations are equal and the step keeps eight waves
      if (g.act == ACT_GELU && !g.aux)
        return run_nt_act<IN, OUT, ACT_GELU, 256, 256, 2, 2, true, true>(g, s);
    }
  }
  return run_nt<IN, OUT, 256, 256, 2, 4, true>(g, s);
}

// The NT fast path applies to 16-bit and fp32 operands that are each
// K-contiguous ([MN][K]) or, where the caller allows it (mn_ok: the 256 x 256
// and 128 x 128 tiles, and fp32 64 x 64), MN-contiguous ([K][MN]), with 16-byte
// aligned bases and rows; C (and the aux matrix) have unit column stride with
// 16-byte aligned rows, and bias is contiguous.  K is whole K-steps, and the
// shape tiles exactly or, where the output is only written (no update in
// place, no column sums, no operand or pre-activation in the output's memory),
// the last tiles are moved back to end at M and N: columns, and rows of an
// M-contiguous A, then have to be whole 16-byte chunks, and the tiles may hold
// a quarter more than the output (above that the next smaller tile or the edge
// kernel does less work).  bf16 against the edge kernel: 8190 x 4096 x 4096 NT
// 233 -> 184 us, NN 238 -> 190; 1000 x 1000 x 1024 9.5 -> 6.5.
template <int IN, int OUT>
bool nt_eligible(const GemmParams& p, int BM, int BN, bool mn_ok) {
  constexpr int ES = IN == IN_F32 ? 4 : 2;
  auto operand_ok = [&](int mode, int64_t ld_k, int64_t ld_mn, int64_t rows_mn) {
    if (mode == LD_KCONTIG) return (ld_k * ES) % 16 == 0 && rows_mn * ld_k * ES < INT32_MAX;
    if (mode == LD_MNCONTIG && mn_ok) return (ld_mn * ES) % 16 == 0 && p.K * ld_mn * ES < INT32_MAX;
    return false;
  };
  // A view [M, K]: K-contiguous row stride a_rs, MN-contiguous row stride a_cs.
  // B view [K, N]: K-contiguous row stride b_cs, MN-contiguous row stride b_rs.
  if (!operand_ok(p.a_mode, p.a_rs, p.a_cs, BM) || !operand_ok(p.b_mode, p.b_cs, p.b_rs, BN)) return false;
  if (p.K % (128 / ES)) return false;
  if (p.M % BM || p.N % BN) {
    constexpr int64_t CE = 16 / ES, CO = OUT == OUT_F32 ? 4 : 8;
    if (p.act == ACT_ADAMW || p.colsum || !p.apart || p.M < BM || p.N < BN) return false;
    if (p.M % BM && p.a_mode != LD_KCONTIG && p.M % CE) return false;
    if (p.N % BN && (p.N % CO || (p.b_mode != LD_KCONTIG && p.N % CE))) return false;
    if (p.M % 64 == 0 && p.N % 64 == 0) {
      // exact smaller tiles exist: fp32 is bound by its MFMAs and loses by
      // every row computed twice (4160 x 4160 x 512 NN 141 us on 64 x 64, 242
      // here); 16-bit from K = 1024 on, or 768 with one output and a 128 x 128
      // tile a CU (bf16 2048 x 2880 x 1024 NN 29.7 us on 64 x 64, 15.6 here, x 768
      // 17.0, 12.9, but 1600 x 1600 x 768 7.6, 8.4), or 512 with eight of them
      // (5824 x 5824 x 512 76, 46; 6464 x 3136 x 512 with both GELU outputs loses
      // 20%); and 256 x 256 only while they take one round of the CUs (2944 x 2944
      // x 1024 NN 28.6 on 128 x 128, 24.7; 4224 x 4224 x 1024 47.2, 49.4) and,
      // beside 128 x 128 ones, with two outputs or a pre-activation from K = 1536
      // on (8192 x 1152 x 1024 NT with both GELU outputs 30.3, 32.1)
      const int64_t tiles128 = ((p.M + 127) / 128) * ((p.N + 127) / 128);
      const bool one_out = p.act == ACT_NONE || p.act == ACT_RELU || (p.act == ACT_GELU && !p.aux);
      const int64_t from = tiles128 >= 2048 ? 512 : one_out && tiles128 >= 256 ? 768 : 1024;
      if (IN == IN_F32 || p.K < from) return false;
      if (BM == 256 && (((p.M + 255) / 256) * ((p.N + 255) / 256) > 256 ||
                        (!one_out && p.M % 128 == 0 && p.N % 128 == 0 && p.K < 1536)))
        return false;
    }
    const int64_t rows = (p.M + BM - 1) / BM * BM, cols = (p.N + BN - 1) / BN * BN;
    if ((double)rows * cols > 1.25 * (double)p.M * p.N) return false;
    if (p.act == ACT_DGELU) {  // Z read again after a neighbour stored its tile
      const uintptr_t c = (uintptr_t)p.C, z = (uintptr_t)p.aux, osz = OUT == OUT_F32 ? 4 : 2;
      if (c < z + (uintptr_t)(p.M * p.aux_rs) * osz && z < c + (uintptr_t)(p.M * p.c_rs) * osz) return false;
    }
  }
  if ((uintptr_t)p.A % 16 || (uintptr_t)p.B % 16) return false;
  const int osz = OUT == OUT_F32 ? 4 : 2;
  if (p.c_cs != 1 || (uintptr_t)p.C % 16 || (p.c_rs * osz) % 16) return false;
  if (p.aux && (((uintptr_t)p.aux % 16) || (p.aux_rs * osz) % 16)) return false;
  if (p.bias && (p.bias_s != 1 || (uintptr_t)p.bias % 16)) return false;
  if (p.M > INT32_MAX / 2 || p.N > INT32_MAX / 2 || p.K > INT32_MAX / 2) return false;
  return true;
}

// Column sums of a 256 x 256 block of a stored bf16 matrix, row t of
// out [M/256, N] for block row t, in the order of the epilogue's
// copy_out_colsum: a lane takes one 8-column chunk and every 16th row, lanes
// l and l + 32 are added, then the 8 waves in order.
__global__ __launch_bounds__(512) void tile_colsum_kernel(const uint16_t* __restrict__ c, int64_t ldc,
                                                          float* __restrict__ out, int N) {
  __shared__ float red[8][256];
  const int tid = threadIdx.x, n0 = blockIdx.x * 256;
  const uint16_t* src = c + ((int64_t)blockIdx.y * 256 + (tid >> 5)) * ldc + n0 + (tid & 31) * 8;
  u16x8 x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) x[k] = *reinterpret_cast<const u16x8*>(src + (int64_t)k * 16 * ldc);
  float cs[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) cs[e] = 0.0f;
#pragma unroll
  for (int k = 0; k < 16; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) cs[e] += bf16_to_f32(x[k][e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) cs[e] += __shfl_xor(cs[e], 32, 64);
  const int w = tid >> 6, l = tid & 63;
  if (l < 32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[w][l * 8 + e] = cs[e];
  }
  __syncthreads();
  if (tid < 256) {
    float s = red[0][tid];
#pragma unroll
    for (int k = 1; k < 8; ++k) s += red[k][tid];
    out[(int64_t)blockIdx.y * N + n0 + tid] = s;
  }
}

template <int IN, int OUT>
Status run_gemm(GemmParams& p, hipStream_t s) {
  p.apart = gemm_outputs_apart(p, IN == IN_F32 ? 4 : 2, OUT == OUT_F32 ? 4 : 2);
  if (p.colsum) {  // dGELU with column sums, bf16 output, M and N multiples of 256
    if constexpr (OUT == OUT_BF16 && IN != IN_F32) {
      if (p.act == ACT_DGELU && nt_eligible<IN, OUT>(p, 256, 256, true)) {
        // the column sums live in the 8-wave 256 x 256 configuration's
        // epilogue (whole tile in one pass): dispatch to it directly
        if ((p.M / 256) * (p.N / 256) >= 128 || !p.apart) return run_nt<IN, OUT, 256, 256, 2, 4, true>(p, s);
        // fewer of those tiles than half the CUs: smaller ones, then the sums
        // from the stored output, in the same order (256 x 3584 x 3584: 72 ->
        // 21 us, 2048^3 49 -> 28; same bits)
        float* colsum = p.colsum;
        p.colsum = nullptr;
        const Status st = run_gemm<IN, OUT>(p, s);
        p.colsum = colsum;
        if (st != Status::Ok) return st;
        tile_colsum_kernel<<<dim3((unsigned)(p.N / 256), (unsigned)(p.M / 256)), 512, 0, s>>>(
            (const uint16_t*)p.C, p.c_rs, colsum, (int)p.N);
        return launch_status("gemm_tile_colsum");
      }
    }
    return Status::NotImplemented;
  }
  if (p.act == ACT_ADAMW) {  // the fused optimizer epilogue: M and N multiples of 256
    if constexpr (OUT == OUT_F32 && IN == IN_BF16) {
      if (nt_eligible<IN, OUT>(p, 256, 256, true)) {
        // the largest tiles that give every other CU one, as for the other
        // epilogues: 1024 x 1024 x 8192 174 -> 37 us, 2048 x 2048 x 8192 181 ->
        // 85, 2560 x 2560 x 4096 122 -> 87 (400 tiles of 128 x 128).  The
        // gradient has the plain product's bits: K order does not depend on the
        // tile, and K is split where the plain product splits it.
        if (edge_splits_k(p, IN)) return edge_gemm(p, IN, OUT, s);
        const int64_t tiles128 = (p.M / 128) * (p.N / 128);
        const bool deep = p.K >= 16 * 64;
        if (tiles128 >= 512 || !p.apart) return run_nt256<IN, OUT>(p, s);
        if (tiles128 >= 128) {
          if (deep && tiles128 <= 256) return run_nt<IN, OUT, 128, 128, 2, 2, true, 4>(p, s);
          return run_nt<IN, OUT, 128, 128, 2, 2, true>(p, s);
        }
        if (deep) return run_nt<IN, OUT, 64, 64, 2, 2, true, 8>(p, s);
        return run_nt<IN, OUT, 64, 64, 2, 2, true>(p, s);
      }
    }
    return Status::NotImplemented;
  }
  if constexpr (IN == IN_F32 && OUT == OUT_F32) {
    // fewer than 128 tiles of 64 x 64: one 16 x 16 tile per wave with K split
    // over the waves of a workgroup reaches more CUs than any tiled
    // configuration, and reads every operand layout in place.  Above 512
    // such tiles (two workgroups a CU) it re-reads the operands from L2 often
    // and long K goes to the edge kernel's K-split tiles: 512 x 512 x 1024 NN
    // 15.8 us, 10.1 there, NT 20.2, 9.4; 300 x 1001 x 2000 NN 45.7, 31.5.  Short
    // K stays, with whole 16 x 16 tiles to K = 511 (512 x 512 x 384 NN 6.5, 8.2;
    // NT 8.0, 8.3), else to 319 (1000 x 200 x 256 NN 5.1, 5.3, NT 6.2, 5.2, x 384
    // 6.6, 6.2; 4096 x 60 x 384 TN 14.4, 6.3), and to 255 from 1408 tiles on (768
    // x 512 x 256 NN 6.7, 6.4, NT 8.0, 6.4).
    const int64_t tiles64 = ((p.M + 63) / 64) * ((p.N + 63) / 64);
    const int64_t tiles16 = ((p.M + 15) / 16) * ((p.N + 15) / 16);
    const bool whole = p.M % 16 == 0 && p.N % 16 == 0 && p.N >= 64;
    const bool split = tiles16 > 512 && p.K >= (tiles16 >= 1408 ? 256 : whole ? 512 : 320) && edge_gemm_ok(p, IN);
    if (tiles64 < kSmallGemmMaxTiles64 && !split && (p.act == ACT_NONE || p.act == ACT_RELU) && p.c_cs == 1 && !p.aux) {
      SmallGemm g{};
      g.A = (const float*)p.A;
      g.B = (const float*)p.B;
      g.C = (float*)p.C;
      g.bias = (const float*)p.bias;
      g.a_m = p.a_rs;
      g.a_k = p.a_cs;
      g.b_k = p.b_rs;
      g.b_n = p.b_cs;
      g.c_m = p.c_rs;
      g.bias_s = p.bias_s;
      g.M = p.M;
      g.N = p.N;
      g.K = p.K;
      g.relu = p.act == ACT_RELU;
      if (small_gemm_ok(g)) return small_gemm_f32(g, s);
    }
    // at most half a 64 x 64 tile a CU: K split over groups of waves (512 x
    // 1024 x 4096 67 -> 46 us, 1856 x 184 x 3392 TN 54 -> 40)
    const int64_t tiles64x32 = ((p.M + 63) / 64) * ((p.N + 31) / 32);
    if (tiles64x32 <= 256 && p.K >= 512 && edge_gemm_ok(p, IN)) return edge_gemm(p, IN, OUT, s);
  }
  {
    constexpr bool MN = true;
    const int64_t tiles256 = ((p.M + 255) / 256) * ((p.N + 255) / 256);
    const int64_t tiles128 = ((p.M + 127) / 128) * ((p.N + 127) / 128);
    // K <= 512 (at most 8 K-steps) with a one-output epilogue (none, bias,
    // ReLU): a 256 x 256 tile's loads and stores are no longer covered by its
    // MFMA work, and 128 x 128 tiles, two workgroups per CU, overlap one
    // tile's epilogue with another's K loop (8192 x 4096 x 256: 30.5 vs 36
    // us, x 512: 42.7 vs 46).  16-bit bias+GELU without the pre-activation
    // output too at K <= 256 (x 256: 33.4 vs 36.5 us on the 8-wave 256 x 256
    // tiles); at K = 512 GELU stays on 256 x 256 (45 vs 48-50 us).
    // K-contiguous operands only; the others keep 256.
    const bool one_out = p.act == ACT_NONE || p.act == ACT_RELU ||
                         (IN != IN_F32 && p.act == ACT_GELU && !p.aux && p.K <= 256);
    if (p.K <= 512 && one_out && tiles128 >= 256 && (p.K <= 256 || IN == IN_F32) &&
        nt_eligible<IN, OUT>(p, 128, 128, false)) {
      // 16-bit: 8 waves of 64 x 32 (8192 x 4096 x 256: 28.3 vs 29.4-31.3 us
      // none, 33.7 vs 35.2-36.0 GELU against 4 waves of 64 x 64)
      if constexpr (IN != IN_F32) return run_nt<IN, OUT, 128, 128, 2, 4, false>(p, s);
      return run_nt<IN, OUT, 128, 128, 2, 2, false>(p, s);
    }
    // Other 16-bit GEMMs with K <= 512 and at least one 256 x 256 tile per
    // CU: the 8-wave persistent tiles (8192 x 4096 x 512: 41.4 vs 46.0 us
    // none, 48.0 vs 52.5 GELU; x 256 with GELU: 38.4 vs 42.2 us against the
    // 4-wave 256 x 256 tiles, same bits).
    if constexpr (IN != IN_F32) {
      if (p.K <= 512 && tiles256 >= 256 && nt_eligible<IN, OUT>(p, 256, 256, MN))
        return run_nt<IN, OUT, 256, 256, 2, 4, MN>(p, s);
    }
    if (tiles256 >= 128 && nt_eligible<IN, OUT>(p, 256, 256, MN)) return run_nt256<IN, OUT>(p, s);
    // 16-bit operands with at least 16 K-steps: small tiles take deeper
    // pipelines (a K-step is a few hundred cycles of MFMA work per wave, less
    // than a load's latency).  128 x 128 with 4 stages needs all of LDS, so
    // only where one workgroup per CU is all the grid gives anyway.
    const bool deep = IN != IN_F32 && p.K >= 16 * (128 / (IN == IN_F32 ? 4 : 2));
    // 128 x 128 and 64 x 64 tiles read every operand layout (2048^3 bf16 NN
    // 112.6 -> 19.8 us, fp32 1024^3 NN 53.8 -> 19.7 us against the
    // general-stride kernel)
    constexpr bool MN64 = true;
    // fp32 is bound by its MFMAs, so by the work of the fullest CU, counted here
    // in 64 x 64 tiles: 2048 x 1024 x 512 takes 33.5 us as one 128 x 128 tile on
    // each of 128 CUs, 17.9 as two 64 x 64 tiles each; 2048 x 2176 x 2048 233,
    // 151.  Where both load it alike, short K gains from the finer tiles (2048 x
    // 1792 x 128 12.1, 11.0), long K from reading half the operand bytes (2048 x
    // 2048 x 4096 NT 236, 254).  From 384 tiles of 128 x 128 on, 128 x 128.
    const int64_t round64 = (((p.M + 63) / 64) * ((p.N + 63) / 64) + 255) / 256, round128 = 4 * ((tiles128 + 255) / 256);
    const bool smaller = IN == IN_F32 && p.apart && tiles128 < 384 &&
                         (round64 < round128 || (round64 == round128 && p.K <= 512));
    if (tiles128 >= 128 && !smaller && nt_eligible<IN, OUT>(p, 128, 128, true)) {
      if constexpr (IN != IN_F32) {
        if (deep && tiles128 <= 256) return run_nt<IN, OUT, 128, 128, 2, 2, true, 4>(p, s);
      }
      return run_nt<IN, OUT, 128, 128, 2, 2, true>(p, s);
    }
    if constexpr (IN != IN_F32) {
      if (edge_splits_k(p, IN)) return edge_gemm(p, IN, OUT, s);
    }
    // fewer tiles than CUs at 128x128: 64x64 tiles (4 waves of 32x32)
    if (nt_eligible<IN, OUT>(p, 64, 64, MN64)) {
      if constexpr (IN != IN_F32) {
        if (deep) return run_nt<IN, OUT, 64, 64, 2, 2, MN64, 8>(p, s);
      }
      return run_nt<IN, OUT, 64, 64, 2, 2, MN64>(p, s);
    }
    if (nt_eligible<IN, OUT>(p, 128, 128, true)) {
      if constexpr (IN != IN_F32) {
        if (deep) return run_nt<IN, OUT, 128, 128, 2, 2, true, 4>(p, s);
      }
      return run_nt<IN, OUT, 128, 128, 2, 2, true>(p, s);
    }
  }
  // shapes no tile divides, unaligned rows
  if (edge_gemm_ok(p, IN)) return edge_gemm(p, IN, OUT, s);
  // What is left: strides with no contiguous dimension, a strided output, K
  // or a contiguous extent of less than 16 bytes.  Large problems: 128x128
  // workgroup tiles (4 waves, 64x64 per wave).  Smaller ones: 64x64 tiles so
  // that enough workgroups exist.
  const int64_t big_tiles = ((p.M + 127) / 128) * ((p.N + 127) / 128);
  if (big_tiles >= 512) return run_cfg<IN, OUT, 128, 128, (IN == IN_F32 ? 32 : 64), 2, 2>(p, s);
  return run_cfg<IN, OUT, 64, 64, (IN == IN_F32 ? 32 : 64), 2, 2>(p, s);
}

int in_kind(DType d) {
  return d == DType::kF32 ? IN_F32 : d == DType::kF16 ? IN_F16 : IN_BF16;
}

Status dispatch_gemm(GemmParams& p, DType din, DType dout, hipStream_t s) {
  const int ik = in_kind(din);
  if (ik == IN_F32 && dout == DType::kF32) return run_gemm<IN_F32, OUT_F32>(p, s);
  if (ik == IN_F16 && dout == DType::kF16) return run_gemm<IN_F16, OUT_F16>(p, s);
  if (ik == IN_F16 && dout == DType::kF32) return run_gemm<IN_F16, OUT_F32>(p, s);
  if (ik == IN_BF16 && dout == DType::kBF16) return run_gemm<IN_BF16, OUT_BF16>(p, s);
  if (ik == IN_BF16 && dout == DType::kF32) return run_gemm<IN_BF16, OUT_F32>(p, s);
  return Status::InvalidArgument;
}

void fill_operands(GemmParams& p, const TensorDesc& A0, const TensorDesc& B0, const TensorDesc& C0,
                   bool ta, bool tb) {
  const View2D A = view2d(A0, ta), B = view2d(B0, tb), C = view2d(C0, false);
  p.A = A.data;
  p.B = B.data;
  p.C = const_cast<void*>(C.data);
  p.M = A.rows;
  p.K = A.cols;
  p.N = B.cols;
  p.a_rs = A.rs;
  p.a_cs = A.cs;
  p.b_rs = B.rs;
  p.b_cs = B.cs;
  p.c_rs = C.rs;
  p.c_cs = C.cs;
  p.a_mode = load_mode(A.rs, A.cs);
  p.b_mode = load_mode(B.cs, B.rs);  // B tile rows are N, K stride is b_rs
  p.bias = nullptr;
  p.aux = nullptr;
  p.act = ACT_NONE;
}

// ---- Gemm variants --------------------------------------------------------
bool gemm_check(const TensorDesc* in, int ni, const TensorDesc* out, int no, const void* attr,
                DType din, DType dout, bool c_rowmajor) {
  if (!in || !out || ni != 2 || no != 1) return false;
  if (dt(in[0]) != din || dt(in[1]) != din || dt(out[0]) != dout) return false;
  bool ta, tb;
  read_gemm_attr(attr, &ta, &tb);
  if (!gemm_views_ok(in[0], in[1], out[0], ta, tb)) return false;
  return !c_rowmajor || is_contig_2d_rowmajor(out[0]);
}

Status gemm_launch_common(const TensorDesc* in, TensorDesc* out, const void* attr, DType din,
                          DType dout, void* stream) {
  bool ta, tb;
  read_gemm_attr(attr, &ta, &tb);
  GemmParams p{};
  fill_operands(p, in[0], in[1], out[0], ta, tb);
  return dispatch_gemm(p, din, dout, as_stream(stream));
}

#define GEMM_VARIANT(NAME, DIN, DOUT, CROW)                                                       \
  bool NAME##_sup(const TensorDesc* i, int ni, const TensorDesc* o, int no, const void* a) {     \
    return gemm_check(i, ni, o, no, a, DIN, DOUT, CROW);                                          \
  }                                                                                               \
  Status NAME##_launch(const TensorDesc* i, int ni, TensorDesc* o, int no, const void* a, void*, \
                       size_t, void* s) {                                                         \
    if (!NAME##_sup(i, ni, o, no, a)) return Status::InvalidArgument;                            \
    return gemm_launch_common(i, o, a, DIN, DOUT, s);                                             \
  }

GEMM_VARIANT(gemm_f32, DType::kF32, DType::kF32, false)
GEMM_VARIANT(gemm_f16, DType::kF16, DType::kF16, true)
GEMM_VARIANT(gemm_bf16, DType::kBF16, DType::kBF16, false)
GEMM_VARIANT(gemm_bf16_f32out, DType::kBF16, DType::kF32, false)

// ---- GemmEpilogue variants ------------------------------------------------
// inputs (A, B, X): X is the bias [N] (kinds 0..4) or Z [M,N] (kind 5).
// outputs (C) or (C, Zaux) for BIAS_GELU.
bool epi_check(const TensorDesc* in, int ni, const TensorDesc* out, int no, const void* attr,
               DType din, DType dout, bool c_rowmajor) {
  if (!in || !out || ni != 3 || no < 1 || no > 3) return false;
  if (dt(in[0]) != din || dt(in[1]) != din || dt(out[0]) != dout) return false;
  const EpiAttr e = read_epi_attr(attr);
  if (!epi_kind_valid(e.kind)) return false;
  if (!gemm_views_ok(in[0], in[1], out[0], e.ta, e.tb)) return false;
  if (c_rowmajor && !is_contig_2d_rowmajor(out[0])) return false;
  const View2D C = view2d(out[0], false);
  const TensorDesc& X = in[2];
  if (e.kind == AICF_EPI_DGELU_COLSUM || e.kind == AICF_EPI_DGELU_PARTIALS) {
    // outputs (C, db [N] f32, workspace [P >= M/256, N] f32), or (C,
    // partials [P >= M/256, N] f32); bf16 output
    const bool fin = e.kind == AICF_EPI_DGELU_COLSUM;
    if (no != (fin ? 3 : 2) || dout != DType::kBF16 || !is_contig_2d_rowmajor(out[0])) return false;
    if (dt(X) != dout || X.rank != 2 || X.shape[0] != C.rows || X.shape[1] != C.cols) return false;
    if (X.stride[1] != 1 || X.stride[0] <= 0) return false;
    const TensorDesc &D = out[1], &W = out[fin ? 2 : 1];
    if (fin && (dt(D) != DType::kF32 || !D.contiguous || D.rank != 1 || D.shape[0] != C.cols)) return false;
    if (dt(W) != DType::kF32 || !W.contiguous || W.rank != 2 || W.shape[1] != C.cols ||
        W.shape[0] < C.rows / 256)
      return false;
    if (!fin && W.shape[0] != C.rows / 256) return false;  // its reader sums every row
    // the column sums are kept per 256-row block: accept exactly the shapes
    // that run_gemm takes with them (M, N multiples of 256, so the workspace
    // has at least one row; K of 64; aligned operands), also of a descriptor
    // whose workspace has no memory yet
    if (din != DType::kBF16 || C.rows % 256 || C.cols % 256) return false;
    GemmParams p{};
    fill_operands(p, in[0], in[1], out[0], e.ta, e.tb);
    p.act = ACT_DGELU;
    p.aux = const_cast<void*>(X.data);
    p.aux_rs = X.stride[0];
    return nt_eligible<IN_BF16, OUT_BF16>(p, 256, 256, true);
  }
  if (no > 2) return false;
  if (e.kind == AICF_EPI_DGELU) {
    if (no != 1) return false;
    if (dt(X) != dout || X.rank != 2 || X.shape[0] != C.rows || X.shape[1] != C.cols) return false;
    if (X.stride[1] != 1 || X.stride[0] <= 0) return false;
  } else {
    // bias: rank 1, length N, positive stride; dtype = input dtype, or fp32
    if (X.rank != 1 || X.stride[0] <= 0 || X.shape[0] != C.cols) return false;
    if (dt(X) != din && dt(X) != DType::kF32) return false;
    if (dt(X) != dout && dt(X) != DType::kF32) return false;
  }
  if (no == 2) {
    if (e.kind != AICF_EPI_BIAS_GELU) return false;
    const TensorDesc& Z = out[1];
    if (dt(Z) != dout || Z.rank != 2 || Z.shape[0] != C.rows || Z.shape[1] != C.cols) return false;
    if (Z.stride[1] != 1 || Z.stride[0] <= 0) return false;
  }
  return true;
}

Status epi_launch_common(const TensorDesc* in, int no, TensorDesc* out, const void* attr, DType din,
                         DType dout, void* stream) {
  const EpiAttr e = read_epi_attr(attr);
  GemmParams p{};
  fill_operands(p, in[0], in[1], out[0], e.ta, e.tb);
  const TensorDesc& X = in[2];
  switch (e.kind) {
    case AICF_EPI_BIAS_RELU: p.act = ACT_RELU; break;
    case AICF_EPI_BIAS: p.act = ACT_NONE; break;
    case AICF_EPI_RELU: p.act = ACT_RELU; break;
    case AICF_EPI_BIAS_GELU: p.act = ACT_GELU; break;
    case AICF_EPI_GELU: p.act = ACT_GELU; break;
    case AICF_EPI_DGELU: p.act = ACT_DGELU; break;
    case AICF_EPI_DGELU_COLSUM: p.act = ACT_DGELU; break;
    case AICF_EPI_DGELU_PARTIALS: p.act = ACT_DGELU; break;
  }
  const bool with_bias = e.kind == AICF_EPI_BIAS_RELU || e.kind == AICF_EPI_BIAS ||
                         e.kind == AICF_EPI_BIAS_GELU;
  if (with_bias) {
    p.bias = X.data;
    p.bias_s = X.stride[0];
    p.bias_f32 = dt(X) == DType::kF32 ? 1 : 0;
  }
  if (e.kind == AICF_EPI_DGELU || e.kind == AICF_EPI_DGELU_COLSUM || e.kind == AICF_EPI_DGELU_PARTIALS) {
    p.aux = const_cast<void*>(X.data);
    p.aux_rs = X.stride[0];
  } else if (no == 2) {
    p.aux = out[1].data;
    p.aux_rs = out[1].stride[0];
  }
  if (e.kind == AICF_EPI_DGELU_PARTIALS) {  // the column sums are finished by a later op
    p.colsum = (float*)out[1].data;
    return dispatch_gemm(p, din, dout, as_stream(stream));
  }
  if (e.kind == AICF_EPI_DGELU_COLSUM) {
    if (!out[2].data) return Status::InvalidArgument;
    p.colsum = (float*)out[2].data;
    const Status st = dispatch_gemm(p, din, dout, as_stream(stream));
    if (st != Status::Ok) return st;
    return colsum_finish(p.colsum, (float*)out[1].data, p.M / 256, p.N, stream);
  }
  return dispatch_gemm(p, din, dout, as_stream(stream));
}

#define EPI_VARIANT(NAME, DIN, DOUT, CROW)                                                        \
  bool NAME##_sup(const TensorDesc* i, int ni, const TensorDesc* o, int no, const void* a) {     \
    return epi_check(i, ni, o, no, a, DIN, DOUT, CROW);                                           \
  }                                                                                               \
  Status NAME##_launch(const TensorDesc* i, int ni, TensorDesc* o, int no, const void* a, void*, \
                       size_t, void* s) {                                                         \
    if (!NAME##_sup(i, ni, o, no, a)) return Status::InvalidArgument;                            \
    return epi_launch_common(i, no, o, a, DIN, DOUT, s);                                          \
  }

EPI_VARIANT(epi_f32, DType::kF32, DType::kF32, false)
EPI_VARIANT(epi_f16, DType::kF16, DType::kF16, true)
EPI_VARIANT(epi_bf16, DType::kBF16, DType::kBF16, false)
EPI_VARIANT(epi_bf16_f32out, DType::kBF16, DType::kF32, false)

// ---------------------------------------------------------------------------
// GemmAdamW (no reference counterpart): the weight-gradient GEMM of a Linear
// layer with AdamW applied in its epilogue, so the fp32 gradient never goes
// to memory.  inputs (A bf16, B bf16, P f32, M f32, V f32, step i32 scalar),
// outputs (P, M, V in place, Wb bf16 shadow of P); P, M, V, Wb are [M, N]
// row-major views; grad = op(A) . op(B).  Attr schema GADW
// <ii fffff>: transA, transB, lr, beta1, beta2, eps, weight_decay.  M and N
// multiples of 256, K of 64, 16-byte aligned rows; other shapes are not
// supported.
// ---------------------------------------------------------------------------
struct GadwAttr {
  bool ta = false, tb = false;
  AdamWArgs args{};
  bool ok = false;
};
GadwAttr read_gadw(const void* attr) {
  GadwAttr g;
  const AttrBlob& a = blob(attr);
  if (!attr || a.schema_id != AICF_SCHEMA_GADW || !payload_ok(a, 28)) return g;
  g.ta = field<int32_t>(a, 0) != 0;
  g.tb = field<int32_t>(a, 4) != 0;
  const float lr = field<float>(a, 8), b1 = field<float>(a, 12), b2 = field<float>(a, 16);
  const float eps = field<float>(a, 20), wd = field<float>(a, 24);
  if (lr != lr || b1 != b1 || b2 != b2 || eps != eps || wd != wd) return g;
  g.args = AdamWArgs{lr, b1, b2, eps, wd, 1.0f - b1, 1.0f - b2, 1.0f - lr * wd};
  g.ok = true;
  return g;
}

bool gadw_fill(const TensorDesc* in, int ni, const TensorDesc* out, int no, const void* attr,
               GemmParams* pp) {
  if (!in || !out || ni != 6 || no != 4) return false;
  const GadwAttr at = read_gadw(attr);
  if (!at.ok) return false;
  if (dt(in[0]) != DType::kBF16 || dt(in[1]) != DType::kBF16) return false;
  for (int k = 2; k < 5; ++k)
    if (dt(in[k]) != DType::kF32 || !is_contig_2d_rowmajor(in[k])) return false;
  if (dt(in[5]) != DType::kI32 || !in[5].contiguous || numel_of(in[5]) != 1) return false;
  for (int k = 0; k < 3; ++k)  // P, M, V updated in place
    if (dt(out[k]) != DType::kF32 || out[k].data != in[k + 2].data || !same_shape(out[k], in[k + 2]))
      return false;
  if (dt(out[3]) != DType::kBF16 || !is_contig_2d_rowmajor(out[3]) || !same_shape(out[3], in[2])) return false;
  if (!same_shape(in[2], in[3]) || !same_shape(in[2], in[4])) return false;
  if (!gemm_views_ok(in[0], in[1], in[2], at.ta, at.tb)) return false;
  GemmParams p{};
  fill_operands(p, in[0], in[1], in[2], at.ta, at.tb);
  p.act = ACT_ADAMW;
  p.adam = GemmAdamW{(float*)in[2].data, (float*)in[3].data, (float*)in[4].data, (uint16_t*)out[3].data,
                     (const int32_t*)in[5].data, at.args};
  if ((uintptr_t)p.adam.M % 16 || (uintptr_t)p.adam.V % 16 || (uintptr_t)p.adam.Wb % 8) return false;
  if (!nt_eligible<IN_BF16, OUT_F32>(p, 256, 256, true)) return false;
  if (pp) *pp = p;
  return true;
}
bool gadw_sup(const TensorDesc* i, int ni, const TensorDesc* o, int no, const void* a) {
  return gadw_fill(i, ni, o, no, a, nullptr);
}
Status gadw_launch(const TensorDesc* i, int ni, TensorDesc* o, int no, const void* a, void*, size_t,
                   void* s) {
  GemmParams p{};
  if (!gadw_fill(i, ni, o, no, a, &p)) return Status::InvalidArgument;
  return run_gemm<IN_BF16, OUT_F32>(p, as_stream(s));
}

size_t no_workspace(const TensorDesc*, int, const void*) { return 0; }

KernelVariant make(const char* name, LaunchFn l, SupportedFn s) {
  KernelVariant v;
  v.name = name;
  v.launch = l;
  v.supported = s;
  v.query_workspace = no_workspace;
  return v;
}

}  // namespace

KernelVariant make_gemm_f32_naive_variant() {
  return make("gemm_f32_mfma", gemm_f32_launch, gemm_f32_sup);
}
KernelVariant make_gemm_f16_tc_wmma_out_f16_variant() {
  return make("gemm_f16_mfma", gemm_f16_launch, gemm_f16_sup);
}
KernelVariant make_gemm_bf16_variant() {
  return make("gemm_bf16_mfma", gemm_bf16_launch, gemm_bf16_sup);
}
KernelVariant make_gemm_bf16_f32out_variant() {
  return make("gemm_bf16_mfma_f32out", gemm_bf16_f32out_launch, gemm_bf16_f32out_sup);
}
KernelVariant make_gemm_bias_relu_f32_naive_variant() {
  return make("gemm_epilogue_f32_mfma", epi_f32_launch, epi_f32_sup);
}
KernelVariant make_gemm_bias_relu_f16_tc_wmma_out_f16_variant() {
  return make("gemm_epilogue_f16_mfma", epi_f16_launch, epi_f16_sup);
}
KernelVariant make_gemm_epilogue_bf16_variant() {
  return make("gemm_epilogue_bf16_mfma", epi_bf16_launch, epi_bf16_sup);
}
KernelVariant make_gemm_epilogue_bf16_f32out_variant() {
  return make("gemm_epilogue_bf16_mfma_f32out", epi_bf16_f32out_launch, epi_bf16_f32out_sup);
}
KernelVariant make_gemm_adamw_bf16_variant() {
  KernelVariant v = make("gemm_adamw_bf16_mfma", gadw_launch, gadw_sup);
  v.expected_attr_schema_id = AICF_SCHEMA_GADW;
  return v;
}

}  // namespace aicf::hip
