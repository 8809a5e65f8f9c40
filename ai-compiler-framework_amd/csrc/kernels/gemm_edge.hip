// GEMM on MFMA for sizes that no exact tiling covers: any M, N and K, any
// element alignment, operands K-contiguous ([MN][K] in memory) or
// M/N-contiguous ([K][MN]), every epilogue of gemm.hip except the column sums
// (AdamW on whole tiles with K split, for the weights that a plain product
// would compute there).
//
//   C[M,N] = epi( op(A)[M,K] . op(B)[K,N] )
//
// The tiles of gemm.hip load straight into LDS, which needs 16-byte aligned
// rows and leaves nothing between memory and the MFMAs to mend a ragged edge
// with.  Here a tile goes through registers: a lane loads 16 bytes (gfx950
// takes them at any element address), and only the chunks that meet an edge
// are mended before they are written to LDS:
//   * rows past M or N read the last row again (their outputs are not stored);
//   * a chunk that would run past the end of its contiguous dimension is
//     moved back to end there, so no load leaves the matrix, and shifted into
//     place; how far is the same for the whole launch, so the shift is scalar;
//   * K past the end is zero in both operands (a NaN beside the matrix, or in
//     another row, reaches no output).
// The LDS layouts, the transposing fragment reads and the operand order (the
// B rows are the MFMA's A operand, so a lane holds 4 consecutive columns of
// one output row) are those of gemm.hip.  One barrier a K-step (128 bytes of K
// per row): two LDS buffers, and the loads of PD further K-steps in flight in
// registers.  PD is 1 throughout: two measured the same, and the loop written
// for one register set without the parameter compiles to slower code (bf16 512
// x 512 x 8192 NT 16.8 us, 20.6).  KSPL groups of waves share a tile's K-steps
// and add up in LDS in a fixed order, for problems with too few tiles for the
// chip.
#include <type_traits>

#include "../common/gemm_types.hpp"

namespace aicf::hip {

namespace {

struct EdgeParams {
  const void* A;
  const void* B;
  void* C;
  const void* bias;
  void* aux;
  int64_t lda, ldb, ldc, aux_ld, bias_s;  // memory row strides (elements)
  int M, N, K;
  int bias_f32, act;
  int tiles_m, tiles_n;
  GemmAdamW adam;  // ADAM only
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <int ES>
struct Chunk;
template <>
struct Chunk<4> {
  typedef uint32_t type __attribute__((ext_vector_type(4), aligned(4)));
};
template <>
struct Chunk<2> {
  typedef uint16_t type __attribute__((ext_vector_type(8), aligned(2)));
};

// Elements s.. of a 16-byte chunk moved to the front, zeros behind (s is
// uniform, 0 <= s < 16 / ES).
template <int ES>
__device__ __forceinline__ u32x4 shift_down(u32x4 d, int s) {
  const int w = ES == 4 ? s : s >> 1;
  if (w & 2) d = u32x4{d[2], d[3], 0, 0};
  if (w & 1) d = u32x4{d[1], d[2], d[3], 0};
  if (ES == 2 && (s & 1))
    d = u32x4{(d[0] >> 16) | (d[1] << 16), (d[1] >> 16) | (d[2] << 16), (d[2] >> 16) | (d[3] << 16), d[3] >> 16};
  return d;
}

// One operand's share of a thread: NCH 16-byte chunks of a BMN x 128 byte
// stage, chunk i at LDS bytes lds + i T 16.
template <int IN, bool KC, int BMN, int T>
struct EdgeOperand {
  static constexpr int ES = IN == IN_F32 ? 4 : 2, CE = 16 / ES;
  static constexpr int MS = ES == 2 ? 16 : 32;       // MFMA block edge
  static constexpr int KB = 128 / ES;                // K of a stage
  static constexpr int NCH = BMN * 8 / T;
  static constexpr int CPR = BMN * ES / 16;          // chunks of an M/N-contiguous row
  static constexpr int DK = KC ? 0 : T / CPR;        // K-rows from a chunk to the thread's next
  // chunk i's LDS place is chunk 0's plus i T 16 (store): its swizzle must not
  // depend on i beyond what store() mends
  static_assert(KC ? T % 64 == 0 : DK % 8 == 0 && (ES == 4 || DK % 16 == 0 || NCH == 1), "swizzle period");
  static_assert(BMN * 8 % T == 0 && (KC || T % CPR == 0), "chunks split evenly over the threads");

  const uint8_t* base;  // uniform.  K-contiguous: the tile's first row; M/N-contiguous: its first column of K-row 0
  int64_t step;         // bytes from a K-step to the next
  int off[KC ? NCH : 1];  // K-contiguous: bytes of each chunk from base; else of the chunk's column
  int kpos;             // first K of the thread's chunk 0 within a K-step
  int ldb;              // M/N-contiguous: bytes of a K-row
  int mn_shift;         // M/N-contiguous: elements the edge chunk was moved back by, 0 elsewhere
  int mn_mod;           // M/N-contiguous, uniform: extent % CE where the tile has such a chunk, else 0
  int lds;

  __device__ __forceinline__ void init(const void* X, int64_t ld, int mn0, int mn_total, int t) {
    const uint8_t* Xb = static_cast<const uint8_t*>(X);
    if constexpr (KC) {
      const int row = t >> 3, c = t & 7, last = mn_total - mn0 - 1;
      base = Xb + (int64_t)mn0 * ld * ES;
      step = 128;
      kpos = c * CE;
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int r = row + i * (T / 8);
        off[i] = (r < last ? r : last) * (int)(ld * ES) + kpos * ES;
      }
      lds = row * 128 + ((c ^ ((row >> 1) & 7)) << 4);
    } else {
      const int k = t / CPR, c = t % CPR, last = mn_total - mn0 - CE, want = c * CE;
      // a tile of fewer than CE columns reads from up to CE - 1 before them
      const int back = last < 0 ? -last : 0;
      base = Xb + (int64_t)(mn0 - back) * ES;
      ldb = (int)(ld * ES);
      step = (int64_t)KB * ldb;
      kpos = k;
      off[0] = ((want < last ? want : last) + back) * ES;
      mn_shift = want > last && want < last + CE ? want - last : 0;
      mn_mod = mn_total - mn0 < BMN ? mn_total % CE : 0;
      lds = k * (CPR * 16) + ((c ^ nt_mn_swizzle<MS, ES, CPR>(k)) << 4);
    }
  }

  // uniform base + unsigned lane offset: one scalar-base load, no 64-bit lane address
  __device__ __forceinline__ static u32x4 get(const uint8_t* b, uint32_t at) {
    return __builtin_bit_cast(u32x4, *reinterpret_cast<const typename Chunk<ES>::type*>(b + at));
  }

  // The thread's chunks of K-step kt.
  __device__ __forceinline__ void load(u32x4 (&r)[NCH], int kt, int K) const {
    const uint8_t* b = base + kt * step;
    const int left = K - kt * KB;  // K from this step on (> 0)
    if constexpr (KC) {
      if (left >= KB) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) r[i] = get(b, (uint32_t)off[i]);
      } else {  // last, partial K-step; K >= CE
        const int last = left - CE, at = kpos < last ? kpos : last;
        const int s = CE - (left & (CE - 1));  // of the one chunk that K ends in
        const bool part = kpos > last && kpos < left, none = kpos >= left;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
          const u32x4 v = get(b - 128, (uint32_t)(off[i] + (at - kpos) * ES + 128));  // at > -CE
          const u32x4 m = shift_down<ES>(v, s & (CE - 1));
#pragma unroll
          for (int d = 0; d < 4; ++d) r[i][d] = none ? 0 : part ? m[d] : v[d];
        }
      }
    } else {
      const int kmax = left - 1;  // K-rows past it read it again and become zero
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int k = kpos + i * DK;
        r[i] = get(b, (uint32_t)(off[0] + (left >= KB ? k : k < kmax ? k : kmax) * ldb));
      }
      if (mn_mod) {
        const int s = CE - mn_mod;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
          const u32x4 m = shift_down<ES>(r[i], s);
#pragma unroll
          for (int d = 0; d < 4; ++d) r[i][d] = mn_shift ? m[d] : r[i][d];
        }
      }
      if (left < KB) {
#pragma unroll
        for (int i = 0; i < NCH; ++i)
          if (kpos + i * DK > kmax) r[i] = u32x4{0, 0, 0, 0};
      }
    }
  }
  __device__ __forceinline__ void store(uint8_t* stage, const u32x4 (&r)[NCH]) const {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      // a K-contiguous row's chunk swizzle has a period of 16 rows: 8 rows on
      // (64 threads), its bit 2 is the other one
      const int at = KC && T == 64 && (i & 1) ? lds ^ 64 : lds;
      *reinterpret_cast<u32x4*>(stage + at + i * (T * 16)) = r[i];
    }
  }
};

// ADAM: the tile is the gradient of a weight matrix; AdamW is applied to it
// instead of storing it (whole tiles, 16-byte aligned rows).
template <int IN, int OUT, int BM, int BN, int WM, int WN, int KSPL, int PD, bool AKC, bool BKC, bool ADAM>
__global__ __launch_bounds__(64 * WM * WN * KSPL) void gemm_edge_kernel(EdgeParams p) {
  constexpr int ES = IN == IN_F32 ? 4 : 2;
  constexpr int MS = ES == 2 ? 16 : 32;             // 16 x 16 x 32, or fp32 32 x 32 x 2
  constexpr int CPS = 64 / MS;                      // 16-byte chunks of K a sub-step
  constexpr int KS = 8 / CPS;                       // sub-steps of a K-step
  constexpr int KPS = CPS * 16 / ES;                // K of a sub-step
  constexpr int KB = 128 / ES;
  constexpr int NW = WM * WN, T = 64 * NW;          // waves and threads of one K group
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / MS, TN = WTN / MS;
  constexpr int A_BYTES = BM * 128, STAGE = (BM + BN) * 128;
  typedef typename std::conditional<MS == 16, floatx4, floatx16>::type acc_t;
  __shared__ __attribute__((aligned(16))) uint8_t smem[KSPL * 2 * STAGE];
  static_assert((KSPL - 1) * BM * BN * 4 <= (int)sizeof(smem), "the K groups' sums fit");

  int tm_i, tn_i;
  tile_coords_of(blockIdx.x, p.tiles_m, p.tiles_n, tm_i, tn_i);
  const int m0 = tm_i * BM, n0 = tn_i * BN;
  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave_all / NW, wave = wave_all % NW;
  const int wm = wave / WN, wn = wave % WN;
  const int t = KSPL == 1 ? (int)threadIdx.x : (int)threadIdx.x - grp * T;
  uint8_t* const mine = smem + grp * (2 * STAGE);

  EdgeOperand<IN, AKC, BM, T> opa;
  EdgeOperand<IN, BKC, BN, T> opb;
  opa.init(p.A, p.lda, m0, p.M, t);
  opb.init(p.B, p.ldb, n0, p.N, t);

  acc_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int r = 0; r < (MS == 16 ? 4 : 16); ++r) acc[i][j][r] = 0.0f;

  // Fragment addresses (as in gemm.hip): the lane holds MN-row fr and K
  // chunk kk CPS + fh of sub-step kk.
  const int fr = lane % MS, fh = lane / MS, rsw = (fr >> 1) & 7;
  const int g16 = (lane >> 4) & 3, i16 = lane & 15;
  const int tr_row = 8 * g16 + (i16 >> 2);
  auto frag_off = [&](int mb, auto KC_, auto BMN_) -> int {
    constexpr int BMN = decltype(BMN_)::value;
    if constexpr (decltype(KC_)::value) {
      return (mb + fr) * 128;
    } else if constexpr (ES == 4) {
      const int m = mb + fr;
      return 4 * fh * (BMN * 4) + (((m >> 2) ^ nt_mn_swizzle<MS, 4, BMN / 4>(4 * fh)) * 16) + (m & 3) * 4;
    } else {
      return tr_row * (BMN * 2) + ((((mb >> 3) ^ nt_mn_swizzle<MS, 2, BMN / 8>(tr_row)) + ((i16 >> 1) & 1)) * 16) +
             8 * (i16 & 1);
    }
  };
  using akc_t = std::integral_constant<bool, AKC>;
  using bkc_t = std::integral_constant<bool, BKC>;
  int a_off[TM], b_off[TN];
#pragma unroll
  for (int j = 0; j < TM; ++j) a_off[j] = frag_off(wm * WTM + j * MS, akc_t{}, std::integral_constant<int, BM>{});
#pragma unroll
  for (int i = 0; i < TN; ++i)
    b_off[i] = A_BYTES + frag_off(wn * WTN + i * MS, bkc_t{}, std::integral_constant<int, BN>{});
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  auto frag = [&](const uint8_t* st, int off, int kk, auto KC_, auto BMN_) -> u16x8 {
    constexpr int ROWB = decltype(BMN_)::value * ES;
    if constexpr (decltype(KC_)::value) {
      return *reinterpret_cast<const u16x8*>(st + off + (((kk * CPS + fh) ^ rsw) * 16));
    } else {
      const uint8_t* a = st + off + kk * KPS * ROWB;
      if constexpr (ES == 4) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const float*>(a + e * ROWB);
        return __builtin_bit_cast(u16x8, v);
      } else {
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)a);
        const v4i16 hi =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)(a + 4 * ROWB));
        u16x8 f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[e] = (uint16_t)lo[e];
          f[e + 4] = (uint16_t)hi[e];
        }
        return f;
      }
    }
  };
  // Fragments of two sub-steps, so that the reads of the next one run during
  // the MFMAs of this one; the 128 x 64 wave tiles have registers for one.
  constexpr int FB = TM * TN >= 32 ? 1 : 2;
  u16x8 fa[FB][TM], fb[FB][TN];
  auto read = [&](const uint8_t* st, int kk) {
    const int s = kk % FB;
#pragma unroll
    for (int j = 0; j < TM; ++j) fa[s][j] = frag(st, a_off[j], kk, akc_t{}, std::integral_constant<int, BM>{});
#pragma unroll
    for (int i = 0; i < TN; ++i) fb[s][i] = frag(st, b_off[i], kk, bkc_t{}, std::integral_constant<int, BN>{});
  };
  auto mfma = [&](int kk) {
    const int s = kk % FB;
    if constexpr (MS == 16) {
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int i = 0; i < TN; ++i)
          acc[i][j] = mfma16<IN>(reinterpret_cast<const uint16_t*>(&fb[s][i]),
                                 reinterpret_cast<const uint16_t*>(&fa[s][j]), acc[i][j]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int i = 0; i < TN; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(reinterpret_cast<const float*>(&fb[s][i])[e],
                                                             reinterpret_cast<const float*>(&fa[s][j])[e], acc[i][j],
                                                             0, 0, 0);
    }
  };

  // K-step `it` of this group is step it KSPL + grp of the tile.  At the top
  // of an iteration its stage is in LDS buffer it & 1 and the loads of the
  // next PD steps are in flight, step it + 1 + j in register set
  // (it + 1 + j) % PD.  Step it + 1 goes to the other buffer after the first
  // sub-step; every wave left that buffer before the last barrier.
  const int nk = (p.K + KB - 1) / KB, iters = (nk + KSPL - 1) / KSPL;
  u32x4 ra[PD][decltype(opa)::NCH], rb[PD][decltype(opb)::NCH];
  auto gload = [&](int it, u32x4 (&xa)[decltype(opa)::NCH], u32x4 (&xb)[decltype(opb)::NCH]) {
    const int kt = it * KSPL + grp;
    if (kt < nk) {
      opa.load(xa, kt, p.K);
      opb.load(xb, kt, p.K);
    }
  };
  auto publish = [&]() {  // own LDS writes done, then the workgroup's; loads stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  gload(0, ra[0], rb[0]);
  opa.store(mine, ra[0]);
  opb.store(mine + A_BYTES, rb[0]);
#pragma unroll
  for (int d = 1; d <= PD; ++d) gload(d, ra[d % PD], rb[d % PD]);
  publish();
  for (int it0 = 0; it0 < iters; it0 += 2 * PD) {
#pragma unroll
    for (int u = 0; u < 2 * PD; ++u) {
      const int it = it0 + u;
      if (it >= iters) break;
      const uint8_t* st = mine + (u & 1) * STAGE;
      const bool here = KSPL == 1 || it * KSPL + grp < nk;
      if (here) {
        read(st, 0);
        if constexpr (FB == 2) read(st, 1);
        mfma(0);
      }
      if (it + 1 < iters) {
        uint8_t* nx = mine + ((u & 1) ^ 1) * STAGE;
        if (KSPL == 1 || (it + 1) * KSPL + grp < nk) {
          opa.store(nx, ra[(u + 1) % PD]);
          opb.store(nx + A_BYTES, rb[(u + 1) % PD]);
        }
        gload(it + 1 + PD, ra[(u + 1) % PD], rb[(u + 1) % PD]);
      }
      if (here) {
#pragma unroll
        for (int kk = 1; kk < KS; ++kk) {
          if constexpr (FB == 1) read(st, kk);
          else if (kk + 1 < KS) read(st, kk + 1);
          mfma(kk);
        }
      }
      publish();
    }
  }

  if constexpr (KSPL > 1) {  // the groups' sums, added in order by group 0
    constexpr int AE = MS == 16 ? 4 : 16;
    float* red = reinterpret_cast<float*>(smem);
    auto slot = [&](int g, int i, int j, int r) {
      return ((((g - 1) * NW + wave) * (TN * TM) + i * TM + j) * AE + r) * 64 + lane;
    };
    if (grp > 0) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int r = 0; r < AE; ++r) red[slot(grp, i, j, r)] = acc[i][j][r];
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 1; g < KSPL; ++g)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int r = 0; r < AE; ++r) acc[i][j][r] += red[slot(g, i, j, r)];
  }

  // Epilogue from the registers: lane (fr, fh) holds 4 consecutive columns of
  // one row per accumulator quad.
  constexpr int G = MS == 32 ? 4 : 1;
  if constexpr (ADAM) {  // 512 x 512 x 4096 NT 12.2 us, 15.7 on the 64 x 64 tiles without the split
    static_assert(G == 1 && OUT == OUT_F32, "bf16 operands, fp32 gradient");
    const AdamWScalars sc = adamw_scalars(p.adam.step, p.adam.args);
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int64_t e = (m0 + wm * WTM + j * MS + fr) * p.ldc + n0 + wn * WTN + i * MS + 4 * fh;
        f32x4 pp = *reinterpret_cast<const f32x4*>(p.adam.P + e);
        f32x4 mm = *reinterpret_cast<const f32x4*>(p.adam.M + e);
        f32x4 vv = *reinterpret_cast<const f32x4*>(p.adam.V + e);
        u16x4 w;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float pk = pp[k], mk = mm[k], vk = vv[k];
          adamw_elem(pk, acc[i][j][k], mk, vk, sc, p.adam.args);
          pp[k] = pk;
          mm[k] = mk;
          vv[k] = vk;
          w[k] = f32_to_bf16(pk);
        }
        *reinterpret_cast<f32x4*>(p.adam.P + e) = pp;
        *reinterpret_cast<f32x4*>(p.adam.M + e) = mm;
        *reinterpret_cast<f32x4*>(p.adam.V + e) = vv;
        *reinterpret_cast<u16x4*>(p.adam.Wb + e) = w;
      }
    return;
  }
  constexpr int OB = OUT == OUT_F32 ? 4 : 2;
  typedef typename std::conditional<OB == 4, float, uint16_t>::type out_t;
  typedef out_t out4 __attribute__((ext_vector_type(4), aligned(OB)));
  auto pack = [&](const float* v) -> out4 {
    if constexpr (OUT == OUT_F32) return out4{v[0], v[1], v[2], v[3]};
    else if constexpr (OUT == OUT_F16) return out4{f32_to_f16(v[0]), f32_to_f16(v[1]), f32_to_f16(v[2]), f32_to_f16(v[3])};
    else return out4{f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]), f32_to_bf16(v[3])};
  };
  auto put = [&](void* base, int64_t row, int n, const float* v) {
    out_t* q = (out_t*)base + row + n;
    const out4 o = pack(v);
    if (n + 4 <= p.N) {
      *reinterpret_cast<out4*>(q) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (n + e < p.N) q[e] = o[e];
    }
  };
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int n = n0 + wn * WTN + i * MS + (MS == 32 ? 8 * g : 0) + 4 * fh;
      if (n >= p.N) continue;
      float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (p.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t at = (n + e < p.N ? n + e : p.N - 1) * p.bias_s;
          b[e] = p.bias_f32 ? ((const float*)p.bias)[at] : load_out<OUT>(p.bias, at);
        }
      }
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int m = m0 + wm * WTM + j * MS + fr;
        if (m >= p.M) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e];
        if (p.act == ACT_DGELU) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] *= gelu_tanh_grad_f(load_out<OUT>(p.aux, m * p.aux_ld + (n + e < p.N ? n + e : p.N - 1)));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += b[e];
          if (p.act == ACT_RELU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
          } else if (p.act == ACT_GELU) {
            if (p.aux) put(p.aux, m * p.aux_ld, n, v);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f(v[e]);
          }
        }
        put(p.C, m * p.ldc, n, v);
      }
    }
}

template <int IN, int OUT, int BM, int BN, int WM, int WN, int KSPL, int PD, bool ADAM = false>
Status run_edge(const GemmParams& g, hipStream_t s) {
  EdgeParams p{};
  const bool akc = g.a_mode == LD_KCONTIG, bkc = g.b_mode == LD_KCONTIG;
  p.A = g.A;
  p.B = g.B;
  p.C = g.C;
  p.bias = g.bias;
  p.aux = g.aux;
  p.lda = akc ? g.a_rs : g.a_cs;
  p.ldb = bkc ? g.b_cs : g.b_rs;
  p.ldc = g.c_rs;
  p.aux_ld = g.aux_rs;
  p.bias_s = g.bias_s;
  p.M = (int)g.M;
  p.N = (int)g.N;
  p.K = (int)g.K;
  p.bias_f32 = g.bias_f32;
  p.act = g.act;
  p.adam = g.adam;
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  const unsigned grid = (unsigned)p.tiles_m * (unsigned)p.tiles_n;
  constexpr int threads = 64 * WM * WN * KSPL;
#define EDGE(A_, B_) gemm_edge_kernel<IN, OUT, BM, BN, WM, WN, KSPL, PD, A_, B_, ADAM><<<grid, threads, 0, s>>>(p)
  if (akc && bkc) EDGE(true, true);
  else if (akc) EDGE(true, false);
  else if (bkc) EDGE(false, true);
  else EDGE(false, false);
#undef EDGE
  return launch_status("gemm_edge");
}

// Tiles by how far the shape fills the chip; us for these sizes, 16-bit unless
// f32 is said:
//   256 x 256, from 3/4 of the CUs on and 8 K-steps: 8190 x 4096 x 4096 NT 233
//     against 286 on 128 x 128 (LDS reads a byte of tile fall with its edge);
//   128 x 128, from 1.5 tiles a CU: 2000 x 3000 x 1000 24.9, 25.9 on 128 x 64;
//   128 x 64, from 7/8 of the CUs: 640 x 3128 x 1405 17.9, 20.7 on 64 x 64;
//   fewer: the K-steps of a tile split over groups of waves.  Eight groups
//     on 32 x 32 (18 x 6464 x 6377 24.6, 40.2 with four on 64 x 64, 53.6
//     without), four on 64 x 32 (f32 777 x 523 x 1000 15.5, 24.0), four on
//     64 x 64 (640 x 1405 x 3128 NN 28.3, 46.7 without), each while it is at
//     most one workgroup a CU;
//   short K: 64 x 128 from 7/8 of the CUs (4096 x 4394 x 64 15.1, 17.1 on 64 x
//     64; 6464 x 6377 x 18 37.7, 39.9, 41.7 on 128 x 64, 65 on 256 x 256), else
//     64 x 64.
template <int IN, int OUT>
Status run_edge_tiles(const GemmParams& g, hipStream_t s) {
  const int64_t nk = (g.K * (IN == IN_F32 ? 4 : 2) + 127) / 128;
  auto tiles = [&](int64_t bm, int64_t bn) { return ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn); };
  if constexpr (IN != IN_F32) {  // fp32 is bound by its MFMAs at 128 x 64 already
    if (nk >= 8 && tiles(256, 256) >= 192) return run_edge<IN, OUT, 256, 256, 2, 4, 1, 1>(g, s);
    if (nk >= 4 && tiles(128, 128) >= 384) return run_edge<IN, OUT, 128, 128, 2, 4, 1, 1>(g, s);
  }
  if (nk >= 4 && tiles(128, 64) >= 224) return run_edge<IN, OUT, 128, 64, 4, 2, 1, 1>(g, s);
  if (nk >= 8) {
    if (tiles(32, 32) <= 256) return run_edge<IN, OUT, 32, 32, 1, 1, 8, 1>(g, s);
    if (tiles(64, 32) <= 256) return run_edge<IN, OUT, 64, 32, 2, 1, 4, 1>(g, s);
    if (tiles(64, 64) <= 256) return run_edge<IN, OUT, 64, 64, 2, 2, 4, 1>(g, s);
  }
  if (nk < 4 && tiles(64, 128) >= 224) return run_edge<IN, OUT, 64, 128, 2, 4, 1, 1>(g, s);
  return run_edge<IN, OUT, 64, 64, 2, 2, 1, 1>(g, s);
}

}  // namespace

bool edge_gemm_ok(const GemmParams& p, int in) {
  const int64_t es = in == IN_F32 ? 4 : 2, ce = 16 / es;
  if (p.colsum || p.c_cs != 1 || !p.apart) return false;
  if (p.M > INT32_MAX / 2 || p.N > INT32_MAX / 2 || p.K > INT32_MAX / 2 || p.K < ce) return false;
  // 32-bit offsets from a tile's first row, for the up to 256 rows of it
  auto operand_ok = [&](int mode, int64_t ld_k, int64_t ld_mn, int64_t mn) {
    if (mode == LD_KCONTIG) return 256 * ld_k * es < INT32_MAX;
    return mode == LD_MNCONTIG && mn >= ce && 128 * ld_mn * es < INT32_MAX;
  };
  if (!operand_ok(p.a_mode, p.a_rs, p.a_cs, p.M) || !operand_ok(p.b_mode, p.b_cs, p.b_rs, p.N)) return false;
  return ((p.M + 63) / 64) * ((p.N + 63) / 64) <= INT32_MAX;
}

bool edge_splits_k(const GemmParams& p, int in) {
  const int64_t tiles32 = ((p.M + 31) / 32) * ((p.N + 31) / 32);
  return tiles32 <= 256 && p.K >= (p.a_mode == LD_KCONTIG ? 2048 : 4096) && edge_gemm_ok(p, in);
}

Status edge_gemm(GemmParams& p, int in, int out, void* stream) {
  hipStream_t s = as_stream(stream);
  if (p.act == ACT_ADAMW) {  // edge_splits_k: the configuration of the plain product
    if (in != IN_BF16 || out != OUT_F32 || p.M % 32 || p.N % 32) return Status::Internal;
    return run_edge<IN_BF16, OUT_F32, 32, 32, 1, 1, 8, 1, true>(p, s);
  }
  if (in == IN_F32 && out == OUT_F32) return run_edge_tiles<IN_F32, OUT_F32>(p, s);
  if (in == IN_F16 && out == OUT_F16) return run_edge_tiles<IN_F16, OUT_F16>(p, s);
  if (in == IN_F16 && out == OUT_F32) return run_edge_tiles<IN_F16, OUT_F32>(p, s);
  if (in == IN_BF16 && out == OUT_BF16) return run_edge_tiles<IN_BF16, OUT_BF16>(p, s);
  if (in == IN_BF16 && out == OUT_F32) return run_edge_tiles<IN_BF16, OUT_F32>(p, s);
  return Status::InvalidArgument;
}

}  // namespace aicf::hip
