// Normalisation kernels for gfx950: LayerNorm forward/backward (f32, f16)
// and BatchNorm forward/backward (f16 NCHW).
//
// Reference contracts:
//   LayerNorm  src/backends/cuda/ops/layernorm/launcher.cu:1-10 (I/O),
//              :41-58 (LNEP eps, default 1e-5), :399-429 (fwd checks),
//              :538-573 (bwd checks); 2-D contiguous row-major x[M,N],
//              normalised over N; mean/rstd f32 [M]; dgamma/dbeta f32 [N].
//   BatchNorm  src/backends/cuda/ops/batchnorm/launcher.cu:1-20 (I/O),
//              :51-84 (BNEP eps + flags), :295-345 (fwd checks),
//              :364-366 (training requires batch statistics), :483-526 (bwd
//              checks, affine only); f16 NCHW contiguous, statistics f32 [C].
//
// Design: memory-bound, so each kernel reads its inputs in 16-byte vectors
// and as few times as its reductions allow.
//   * A LayerNorm row is held in registers by 64 to 1024 lanes, for any
//     row length and alignment (RowVec below).  The affine backward of a
//     large matrix reads x and dy once: the lanes that compute dx also
//     accumulate their columns' dgamma and dbeta over the rows of their
//     workgroup.
//   * A BatchNorm channel of up to 64K elements is held in the registers of
//     one workgroup; larger channels are split over workgroups, with a
//     second pass for the output.
//   * Partial sums between two kernels of one call live in that call's own
//     output (dx or y), which a later kernel of the call overwrites: the ops
//     have no workspace argument, and nothing is shared between calls.
// Every reduction has a fixed order (wave64 butterflies, LDS combines, no
// atomics, no memsets): results are reproducible and the ops are safe under
// graph capture.  Variances are centred (sum of squared deviations from the
// mean), the accurate form of the reference's E[x^2] - mean^2.
#include "../common/hip_util.hpp"

namespace aicf::hip {

namespace {

size_t no_workspace(const TensorDesc*, int, const void*) { return 0; }

KernelVariant make(const char* name, LaunchFn l, SupportedFn s, uint32_t schema = 0) {
  KernelVariant v;
  v.name = name;
  v.launch = l;
  v.supported = s;
  v.query_workspace = no_workspace;
  v.expected_attr_schema_id = schema;
  return v;
}

template <typename T>
__device__ __forceinline__ float ld_as_f32(const T* p, int64_t i) {
  if constexpr (sizeof(T) == 4) {
    return p[i];
  } else {
    return f16_to_f32(p[i]);
  }
}
template <typename T>
__device__ __forceinline__ void st_from_f32(T* p, int64_t i, float v) {
  if constexpr (sizeof(T) == 4) {
    p[i] = v;
  } else {
    p[i] = f32_to_f16(v);
  }
}

// ===========================================================================
// LayerNorm
// ===========================================================================
// Rows of at most 64 columns, one a lane, a wave per row.  In vectors such a
// row leaves most lanes without one and pays for the masks of the last: f32
// [4024, 49] 2.6 us against 3.0, f16 [4024, 64] without affine, backward, 2.4
// against 3.0.
template <typename T>
__global__ __launch_bounds__(256) void ln_fwd_narrow_kernel(const T* x, const T* gamma, const T* beta, T* y,
                                                            float* mean, float* rstd, int M, int N, float eps) {
  const int c = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;  // whole wave
  const int64_t at = (int64_t)row * N + c;
  const float invN = 1.0f / (float)N;
  const float v = c < N ? ld_as_f32(x, at) : 0.0f;
  const float mu = wave_sum(v) * invN;
  const float t = c < N ? v - mu : 0.0f;
  const float rs = 1.0f / sqrtf(wave_sum(t * t) * invN + eps);
  if (c < N) {
    float o = (v - mu) * rs;
    if (gamma) o = fmaf(o, ld_as_f32(gamma, c), ld_as_f32(beta, c));
    st_from_f32(y, at, o);
  }
  if (c == 0) {
    mean[row] = mu;
    rstd[row] = rs;
  }
}
template <typename T>
__global__ __launch_bounds__(256) void ln_bwd_dx_narrow_kernel(const T* x, const T* dy, const T* gamma,
                                                               const float* mean, const float* rstd, T* dx, int M,
                                                               int N) {
  const int c = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const int64_t at = (int64_t)row * N + c;
  const float mu = mean[row], rs = rstd[row];
  const float fN = (float)N, scale = rs / fN;
  float xh = 0.0f, g = 0.0f;
  if (c < N) {
    xh = (ld_as_f32(x, at) - mu) * rs;
    g = ld_as_f32(dy, at);
    if (gamma) g *= ld_as_f32(gamma, c);
  }
  const float s1 = wave_sum(g), s2 = wave_sum(g * xh);
  if (c < N) st_from_f32(dx, at, (fN * g - s1 - xh * s2) * scale);
}

// Any N, one wave per row, the row read two or three times: rows longer than
// the register-resident kernels hold.
template <typename T>
__global__ __launch_bounds__(256) void ln_fwd_loop_kernel(const T* x, const T* gamma,
                                                          const T* beta, T* y,
                                                          float* mean, float* rstd,
                                                          int M, int N, float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;  // whole wave
  const T* xr = x + (int64_t)row * N;
  T* yr = y + (int64_t)row * N;
  const float invN = 1.0f / (float)N;
  float s = 0.0f;
  for (int c = lane; c < N; c += 64) s += ld_as_f32(xr, c);
  const float mu = wave_sum(s) * invN;
  float d = 0.0f;
  for (int c = lane; c < N; c += 64) {
    const float t = ld_as_f32(xr, c) - mu;
    d = fmaf(t, t, d);
  }
  const float rs = 1.0f / sqrtf(wave_sum(d) * invN + eps);
  for (int c = lane; c < N; c += 64) {
    float o = (ld_as_f32(xr, c) - mu) * rs;
    if (gamma) o = fmaf(o, ld_as_f32(gamma, c), ld_as_f32(beta, c));
    st_from_f32(yr, c, o);
  }
  if (lane == 0) {
    mean[row] = mu;
    rstd[row] = rs;
  }
}

// Backward dx: dyh = dy * gamma (gamma null => 1), xhat = (x - mean) rstd,
// dx = (N dyh - sum(dyh) - xhat sum(dyh xhat)) * rstd / N.
template <typename T>
__global__ __launch_bounds__(256) void ln_bwd_dx_loop_kernel(const T* x, const T* dy,
                                                             const T* gamma,
                                                             const float* mean,
                                                             const float* rstd, T* dx,
                                                             int M, int N) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const T* xr = x + (int64_t)row * N;
  const T* dyr = dy + (int64_t)row * N;
  T* dxr = dx + (int64_t)row * N;
  const float mu = mean[row], rs = rstd[row];
  const float fN = (float)N, scale = rs / fN;
  float s1 = 0.0f, s2 = 0.0f;
  for (int c = lane; c < N; c += 64) {
    const float xh = (ld_as_f32(xr, c) - mu) * rs;
    float g = ld_as_f32(dyr, c);
    if (gamma) g *= ld_as_f32(gamma, c);
    s1 += g;
    s2 = fmaf(g, xh, s2);
  }
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  for (int c = lane; c < N; c += 64) {
    const float xh = (ld_as_f32(xr, c) - mu) * rs;
    float g = ld_as_f32(dyr, c);
    if (gamma) g *= ld_as_f32(gamma, c);
    st_from_f32(dxr, c, (fN * g - s1 - xh * s2) * scale);
  }
}

// Backward dgamma[c] = sum_m dy xhat, dbeta[c] = sum_m dy: lane per column,
// the 4 waves take every fourth row, combined in LDS in a fixed order.
template <typename T>
__global__ __launch_bounds__(256) void ln_bwd_dgdb_loop_kernel(const T* __restrict__ x, const T* __restrict__ dy,
                                                               const float* __restrict__ mean,
                                                               const float* __restrict__ rstd,
                                                               float* __restrict__ dgamma,
                                                               float* __restrict__ dbeta, int M, int N) {
  __shared__ float red[2][4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float sg = 0.0f, sb = 0.0f;
  if (c < N) {
    for (int64_t r = w; r < M; r += 4) {
      const float xh = (ld_as_f32(x, r * N + c) - mean[r]) * rstd[r];
      const float d = ld_as_f32(dy, r * N + c);
      sb += d;
      sg = fmaf(d, xh, sg);
    }
  }
  red[0][w][lane] = sg;
  red[1][w][lane] = sb;
  __syncthreads();
  if (w == 0 && c < N) {
    dgamma[c] = (red[0][0][lane] + red[0][1][lane]) + (red[0][2][lane] + red[0][3][lane]);
    dbeta[c] = (red[1][0][lane] + red[1][1][lane]) + (red[1][2][lane] + red[1][3][lane]);
  }
}

// 16-byte vectors of elements at any element address (gfx950 loads and stores
// them unaligned).
template <typename T>
constexpr int kVec = 16 / (int)sizeof(T);
template <typename T>
struct RowVecType {
  typedef T type __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};
template <typename T>
__device__ __forceinline__ float cvt_f32(T v) {
  if constexpr (sizeof(T) == 4) return v;
  else return f16_to_f32(v);
}

// A row of N >= V columns as V-column vectors over the lanes of its group:
// vector k of lane l covers columns col(k) .. col(k) + V - 1.  The vectors
// past the last whole one are moved back to end at column N - 1, so every
// load and store is a whole vector inside the row; first(k) is the first of
// its elements that no earlier vector holds (V: none), and only those count
// in a sum.  A column that two vectors hold is stored by both, with the same
// bits, since both compute it from the same values.
template <typename T, int LPR>
struct RowVec {
  static constexpr int V = kVec<T>;
  int N, l;
  __device__ __forceinline__ int col(int k) const {
    const int c = (k * LPR + l) * V;
    return c < N - V ? c : N - V;
  }
  __device__ __forceinline__ int first(int k) const {
    const int c = (k * LPR + l) * V - (N - V);
    return c < 0 ? 0 : c < V ? c : V;
  }
  __device__ __forceinline__ bool any(int k) const { return (k * LPR + l) * V < N; }
};
template <typename T>
__device__ __forceinline__ void load_f32(const T* p, float* o) {
  const typename RowVecType<T>::type v = *reinterpret_cast<const typename RowVecType<T>::type*>(p);
#pragma unroll
  for (int e = 0; e < kVec<T>; ++e) o[e] = cvt_f32<T>(v[e]);
}
// Nontemporal: the output is not read again by this op.
template <typename T>
__device__ __forceinline__ void store_f32(T* p, const float* o) {
  typename RowVecType<T>::type v;
#pragma unroll
  for (int e = 0; e < kVec<T>; ++e) {
    if constexpr (sizeof(T) == 4) v[e] = o[e];
    else v[e] = f32_to_f16(o[e]);
  }
  __builtin_nontemporal_store(v, reinterpret_cast<typename RowVecType<T>::type*>(p));
}

// Sums of two values over the LPR lanes of a row (LPR >= 64): butterfly in
// each wave, then the waves of the row through LDS in a fixed order.  One
// barrier; a call may follow another one only with the other half of `lds`
// (a wave can be at most one barrier ahead, so it never writes a half that a
// slower wave still reads).
template <int LPR>
__device__ __forceinline__ void row_sum2(float& a, float& b, f32x2_t* lds) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  if constexpr (LPR > 64) {
    constexpr int NW = LPR / 64;
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds[w] = f32x2_t{a, b};
    __syncthreads();
    const f32x2_t* r = lds + w / NW * NW;
    a = r[0][0];
    b = r[0][1];
#pragma unroll
    for (int k = 1; k < NW; ++k) {
      a += r[k][0];
      b += r[k][1];
    }
  }
}

constexpr int ln_threads(int lpr) { return lpr > 512 ? lpr : 512; }

// Forward, row in registers: one read of x, one write of y; bound by HBM.
// f32 [8192, 4096]: 46 us (5.8 TB/s) against 115 on the looping kernel, which
// reads x three times, 4 bytes a lane; f16 [1500, 1000]: 4.2 against 14.3.
template <typename T, int LPR, int VPT>
__global__ __launch_bounds__(ln_threads(LPR)) void ln_fwd_kernel(const T* x, const T* gamma,
                                                                const T* beta, T* y,
                                                                float* mean, float* rstd,
                                                                int M, int N, float eps) {
  constexpr int V = kVec<T>, RPB = ln_threads(LPR) / LPR;
  __shared__ f32x2_t lds[2][ln_threads(LPR) / 64];
  const RowVec<T, LPR> rv{N, (int)threadIdx.x % LPR};
  const int row0 = blockIdx.x * RPB + threadIdx.x / LPR;
  const int row = row0 < M ? row0 : M - 1;  // every wave takes part in the barriers
  const T* xr = x + (int64_t)row * N;
  float v[VPT][V];
#pragma unroll
  for (int k = 0; k < VPT; ++k) load_f32<T>(xr + rv.col(k), v[k]);
  float s = 0.0f, z = 0.0f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int f = rv.first(k);
#pragma unroll
    for (int e = 0; e < V; ++e) s += e >= f ? v[k][e] : 0.0f;
  }
  row_sum2<LPR>(s, z, lds[0]);
  const float invN = 1.0f / (float)N;
  const float mu = s * invN;
  float d = 0.0f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int f = rv.first(k);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float t = e >= f ? v[k][e] - mu : 0.0f;
      d = fmaf(t, t, d);
    }
  }
  row_sum2<LPR>(d, z, lds[1]);
  const float rs = 1.0f / sqrtf(d * invN + eps);
  if (row0 >= M) return;
  T* yr = y + (int64_t)row * N;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    if (!rv.any(k)) continue;
    const int c = rv.col(k);
    float o[V];
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = (v[k][e] - mu) * rs;
    if (gamma) {
      float g[V], b[V];
      load_f32<T>(gamma + c, g);
      load_f32<T>(beta + c, b);
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = fmaf(o[e], g[e], b[e]);
    }
    store_f32<T>(yr + c, o);
  }
  if (rv.l == 0) {
    mean[row] = mu;
    rstd[row] = rs;
  }
}

template <typename T>
struct LnBwd {
  const T* x;
  const T* dy;
  const T* gamma;
  const float* mean;
  const float* rstd;
  T* dx;
  float* dgamma;
  float* dbeta;
  int M, N;
  // Fused backward: the rows are cut into P chunks, one workgroup each.  A
  // chunk's last RS rows of dx hold its partial sums (2 N floats) until the
  // finish kernel has added them up; their dx is computed after that.
  int P, RS;
  int q, r;  // M / P, M % P
  __device__ __forceinline__ int chunk(int w) const { return w * q + (w < r ? w : r); }  // its first row
  __device__ float* partial(int w) const {
    const uintptr_t a = reinterpret_cast<uintptr_t>(dx + (int64_t)(chunk(w + 1) - RS) * N);
    return reinterpret_cast<float*>((a + 3) & ~(uintptr_t)3);
  }
};

// dx of one row from its x and dy in registers (x is replaced by xhat, dy by
// dy gamma); gamma null => 1.
template <typename T, int LPR, int VPT>
__device__ __forceinline__ void ln_bwd_row(const LnBwd<T>& a, const RowVec<T, LPR>& rv, int row, bool store,
                                          float (&xh)[VPT][kVec<T>], float (&g)[VPT][kVec<T>], f32x2_t* lds) {
  constexpr int V = kVec<T>;
  const float rs = a.rstd[row];
  const float fN = (float)a.N, scale = rs / fN;
  float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    if (a.gamma) {
      float w[V];
      load_f32<T>(a.gamma + rv.col(k), w);
#pragma unroll
      for (int e = 0; e < V; ++e) g[k][e] *= w[e];
    }
    const int f = rv.first(k);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float ge = e >= f ? g[k][e] : 0.0f;
      s1 += ge;
      s2 = e >= f ? fmaf(ge, xh[k][e], s2) : s2;
    }
  }
  row_sum2<LPR>(s1, s2, lds);
  if (!store) return;
  T* dxr = a.dx + (int64_t)row * a.N;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    if (!rv.any(k)) continue;
    float o[V];
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = (fN * g[k][e] - s1 - xh[k][e] * s2) * scale;
    store_f32<T>(dxr + rv.col(k), o);
  }
}

template <typename T, int LPR, int VPT>
__device__ __forceinline__ void ln_bwd_load(const LnBwd<T>& a, const RowVec<T, LPR>& rv, int row,
                                           float (&xh)[VPT][kVec<T>], float (&g)[VPT][kVec<T>]) {
  const T* xr = a.x + (int64_t)row * a.N;
  const T* dyr = a.dy + (int64_t)row * a.N;
#pragma unroll
  for (int k = 0; k < VPT; ++k) {
    load_f32<T>(xr + rv.col(k), xh[k]);
    load_f32<T>(dyr + rv.col(k), g[k]);
  }
  const float mu = a.mean[row], rs = a.rstd[row];
#pragma unroll
  for (int k = 0; k < VPT; ++k)
#pragma unroll
    for (int e = 0; e < kVec<T>; ++e) xh[k][e] = (xh[k][e] - mu) * rs;
}

// dgamma and dbeta of 2 V columns over all rows (one workgroup of 512): 256
// row slots of two lanes, four rows in flight a slot, the slots added in LDS
// by a fixed-order tree.
constexpr int kLnColThreads = 512, kLnColLanes = 2, kLnColSlots = kLnColThreads / kLnColLanes;
template <typename T>
constexpr int ln_col_lds() { return kLnColSlots * (2 * kLnColLanes * kVec<T> + 1); }  // floats
template <typename T>
__device__ __forceinline__ void ln_bwd_columns(const LnBwd<T>& a, int block, float* red) {
  constexpr int V = kVec<T>, W = 2 * kLnColLanes * V, STRIDE = W + 1, UNROLL = 4;
  const int slot = (int)threadIdx.x / kLnColLanes, v = (int)threadIdx.x % kLnColLanes;
  const int c = (block * kLnColLanes + v) * V;
  const int c0 = c < a.N - V ? c : a.N - V;
  float sg[V], sb[V];
#pragma unroll
  for (int e = 0; e < V; ++e) sg[e] = sb[e] = 0.0f;
  typedef typename RowVecType<T>::type vec;
  auto add = [&](const vec& xv, const vec& dv, float mu, float rs) {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float d = cvt_f32<T>(dv[e]);
      sb[e] += d;
      sg[e] = fmaf(d, (cvt_f32<T>(xv[e]) - mu) * rs, sg[e]);
    }
  };
  int r = slot;
  for (; r + (UNROLL - 1) * kLnColSlots < a.M; r += UNROLL * kLnColSlots) {
    vec xv[UNROLL], dv[UNROLL];
    float mu[UNROLL], rs[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int64_t at = (int64_t)(r + u * kLnColSlots) * a.N + c0;
      xv[u] = *reinterpret_cast<const vec*>(a.x + at);
      dv[u] = *reinterpret_cast<const vec*>(a.dy + at);
      mu[u] = a.mean[r + u * kLnColSlots];
      rs[u] = a.rstd[r + u * kLnColSlots];
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) add(xv[u], dv[u], mu[u], rs[u]);
  }
  if (r < a.M) {  // the rest in one batch too; rows past M read the last one and add zeros
    vec xv[UNROLL - 1], dv[UNROLL - 1];
    float mu[UNROLL - 1], rs[UNROLL - 1];
#pragma unroll
    for (int u = 0; u < UNROLL - 1; ++u) {
      const bool on = r + u * kLnColSlots < a.M;
      const int row = on ? r + u * kLnColSlots : a.M - 1;
      const int64_t at = (int64_t)row * a.N + c0;
      xv[u] = *reinterpret_cast<const vec*>(a.x + at);
      dv[u] = *reinterpret_cast<const vec*>(a.dy + at);
      mu[u] = a.mean[row];
      rs[u] = a.rstd[row];
      if (!on) xv[u] = dv[u] = vec{}, mu[u] = rs[u] = 0.0f;
    }
#pragma unroll
    for (int u = 0; u < UNROLL - 1; ++u) add(xv[u], dv[u], mu[u], rs[u]);
  }
#pragma unroll
  for (int e = 0; e < V; ++e) {
    red[slot * STRIDE + 2 * v * V + e] = sg[e];
    red[slot * STRIDE + (2 * v + 1) * V + e] = sb[e];
  }
  __syncthreads();
  for (int half = kLnColSlots / 2; half > 0; half >>= 1) {  // slot i += slot i + half
    for (int t = (int)threadIdx.x; t < half * W; t += kLnColThreads) {
      const int i = t / W, q = t % W;
      red[i * STRIDE + q] += red[(i + half) * STRIDE + q];
    }
    __syncthreads();
  }
  if ((int)threadIdx.x < W) {
    const int lane = (int)threadIdx.x / (2 * V), q = (int)threadIdx.x % (2 * V);
    const int cl = (block * kLnColLanes + lane) * V;
    if (cl < a.N) {
      const int at = (cl < a.N - V ? cl : a.N - V) + q % V;
      (q < V ? a.dgamma : a.dbeta)[at] = red[threadIdx.x];
    }
  }
}

// Backward in one launch: the first `row_blocks` workgroups compute dx, a row
// per LPR lanes; the others dgamma and dbeta, reading x and dy a second time,
// which comes from the caches for the sizes this kernel is used at.  reserved
// (see LnBwd): dx of the last RS rows of each chunk instead of all rows.  f16
// [1500, 1000]: 8.0 us against 146 for a dx kernel and a column kernel of N / 64
// workgroups that walk all rows.
template <typename T, int LPR, int VPT>
__global__ __launch_bounds__(ln_threads(LPR)) void ln_bwd_kernel(LnBwd<T> a, int row_blocks, bool reserved) {
  constexpr int RPB = ln_threads(LPR) / LPR;
  __shared__ union {
    f32x2_t row[ln_threads(LPR) / 64];
    float col[ln_threads(LPR) == kLnColThreads ? ln_col_lds<T>() : 1];
  } lds;
  if (ln_threads(LPR) == kLnColThreads && (int)blockIdx.x >= row_blocks) {  // whole workgroup
    ln_bwd_columns<T>(a, (int)blockIdx.x - row_blocks, lds.col);
    return;
  }
  const RowVec<T, LPR> rv{a.N, (int)threadIdx.x % LPR};
  int row = blockIdx.x * RPB + threadIdx.x / LPR;
  const int rows = reserved ? a.P * a.RS : a.M;
  const bool on = row < rows;
  if (!on) row = rows - 1;
  if (reserved) row = a.chunk(row / a.RS + 1) - a.RS + row % a.RS;
  float xh[VPT][kVec<T>], g[VPT][kVec<T>];
  ln_bwd_load<T, LPR, VPT>(a, rv, row, xh, g);
  ln_bwd_row<T, LPR, VPT>(a, rv, row, on, xh, g, lds.row);
}
template <typename T>
__global__ __launch_bounds__(kLnColThreads) void ln_bwd_columns_kernel(LnBwd<T> a) {
  __shared__ float red[ln_col_lds<T>()];
  ln_bwd_columns<T>(a, blockIdx.x, red);
}

// Fused backward: workgroup w owns the rows of chunk w, G = 1024 / LPR groups
// of lanes taking every G-th of them, and a lane keeps the dgamma and dbeta
// sums of its columns in registers over all its rows.  The groups' sums are
// added in LDS by a fixed-order tree and written to the chunk's reserved rows
// of dx.  f32 [8192, 4096]: 66 us (6.1 TB/s of x, dy and dx), 78 with the finish
// and the reserved rows, against 1040 for the two separate kernels; bound by HBM.
template <typename T, int LPR, int VPT>
__global__ __launch_bounds__(1024) void ln_bwd_fused_kernel(LnBwd<T> a) {
  constexpr int V = kVec<T>, G = 1024 / LPR, COLS = LPR * VPT * V;
  __shared__ f32x2_t lds[2][16];
  __shared__ float red[G > 1 ? G / 2 * COLS : 1];
  const int grp = threadIdx.x / LPR;
  const RowVec<T, LPR> rv{a.N, (int)threadIdx.x % LPR};
  const int r0 = a.chunk(blockIdx.x), r1 = a.chunk(blockIdx.x + 1);
  float sg[VPT][V], sb[VPT][V];
#pragma unroll
  for (int k = 0; k < VPT; ++k)
#pragma unroll
    for (int e = 0; e < V; ++e) sg[k][e] = sb[k][e] = 0.0f;
  int it = 0;
  for (int base = r0; base < r1; base += G, ++it) {
    const bool on = base + grp < r1;
    const int row = on ? base + grp : r1 - 1;  // every wave takes part in the barriers
    float xh[VPT][V], g[VPT][V];
    ln_bwd_load<T, LPR, VPT>(a, rv, row, xh, g);
    if (on) {
#pragma unroll
      for (int k = 0; k < VPT; ++k)
#pragma unroll
        for (int e = 0; e < V; ++e) {
          sb[k][e] += g[k][e];
          sg[k][e] = fmaf(g[k][e], xh[k][e], sg[k][e]);
        }
    }
    ln_bwd_row<T, LPR, VPT>(a, rv, row, on && row < r1 - a.RS, xh, g, lds[it & 1]);
  }
  if constexpr (G > 1) {
    auto tree = [&](float (&s)[VPT][V]) {
#pragma unroll
      for (int half = G / 2; half > 0; half >>= 1) {
        __syncthreads();
        if (grp >= half && grp < 2 * half) {
#pragma unroll
          for (int k = 0; k < VPT; ++k)
#pragma unroll
            for (int e = 0; e < V; ++e) red[((grp - half) * VPT + k) * LPR * V + e * LPR + rv.l] = s[k][e];
        }
        __syncthreads();
        if (grp < half) {
#pragma unroll
          for (int k = 0; k < VPT; ++k)
#pragma unroll
            for (int e = 0; e < V; ++e) s[k][e] += red[(grp * VPT + k) * LPR * V + e * LPR + rv.l];
        }
      }
    };
    tree(sg);
    tree(sb);
  }
  if (grp == 0) {
    float* out = a.partial(blockIdx.x);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      if (!rv.any(k)) continue;
      const int c = rv.col(k);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        out[c + e] = sg[k][e];
        out[a.N + c + e] = sb[k][e];
      }
    }
  }
}

// dgamma and dbeta from the P partial rows: 64 of the 2 N sums a workgroup,
// the 16 waves take every 16th partial, combined in LDS in a fixed order.
template <typename T>
__global__ __launch_bounds__(1024) void ln_bwd_finish_kernel(LnBwd<T> a) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float s = 0.0f;
  if (c < 2 * a.N) {
    int p = w;
    for (; p + 7 * 16 < a.P; p += 8 * 16) {  // eight loads in flight
      float q[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) q[u] = a.partial(p + u * 16)[c];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += q[u];
    }
    for (; p < a.P; p += 16) s += a.partial(p)[c];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w == 0 && c < 2 * a.N) {
    float t = red[0][lane];
#pragma unroll
    for (int k = 1; k < 16; ++k) t += red[k][lane];
    (c < a.N ? a.dgamma : a.dbeta)[c < a.N ? c : c - a.N] = t;
  }
}

// LNEP <f> eps; schema 0 (or anything else, or a short payload) => 1e-5
// (layernorm/launcher.cu:49-58).
float read_ln_eps(const void* attr) {
  const AttrBlob& a = blob(attr);
  if (!attr || a.schema_id != AICF_SCHEMA_LNEP || !payload_ok(a, 4)) return 1e-5f;
  return field<float>(a, 0);
}

bool vec1_len(const TensorDesc& t, DType d, int64_t n) {
  return dt(t) == d && t.rank == 1 && t.contiguous && t.shape[0] == n;
}

// layernorm/launcher.cu:399-429: inputs (X) or (X, G, B); outputs (Y, Mean, Rstd)
bool ln_fwd_check(const TensorDesc* in, int ni, const TensorDesc* out, int no, DType d) {
  if (!in || !out || !(ni == 1 || ni == 3) || no != 3) return false;
  const TensorDesc &X = in[0], &Y = out[0];
  if (dt(X) != d || dt(Y) != d || !is_contig_2d_rowmajor(X) || !is_contig_2d_rowmajor(Y)) return false;
  if (!same_shape(X, Y)) return false;
  const int64_t M = X.shape[0], N = X.shape[1];
  if (M > INT32_MAX || N > INT32_MAX || N < 1) return false;
  if (!vec1_len(out[1], DType::kF32, M) || !vec1_len(out[2], DType::kF32, M)) return false;
  if (ni == 3 && (!vec1_len(in[1], d, N) || !vec1_len(in[2], d, N))) return false;
  return true;
}

// layernorm/launcher.cu:538-573: (X, dY, Mean, Rstd) -> (dX) or
// (X, dY, G, Mean, Rstd) -> (dX, dG, dB)
bool ln_bwd_check(const TensorDesc* in, int ni, const TensorDesc* out, int no, DType d) {
  if (!in || !out) return false;
  const bool affine = ni == 5 && no == 3, noaff = ni == 4 && no == 1;
  if (!affine && !noaff) return false;
  const TensorDesc &X = in[0], &dY = in[1], &dX = out[0];
  for (const TensorDesc* t : {&X, &dY, &dX})
    if (dt(*t) != d || !is_contig_2d_rowmajor(*t)) return false;
  if (!same_shape(X, dY) || !same_shape(X, dX)) return false;
  const int64_t M = X.shape[0], N = X.shape[1];
  if (M > INT32_MAX || N > INT32_MAX || N < 1) return false;
  if (!vec1_len(in[affine ? 3 : 2], DType::kF32, M) || !vec1_len(in[affine ? 4 : 3], DType::kF32, M)) return false;
  if (affine && (!vec1_len(in[2], d, N) || !vec1_len(out[1], DType::kF32, N) || !vec1_len(out[2], DType::kF32, N)))
    return false;
  return true;
}

// Lanes and vectors a lane for a row of nv vectors: a wave up to 256 vectors
// (no barrier), then the fewest lanes with four vectors each.
#define LN_BY_WIDTH(CALL)        \
  if (nv <= 64) CALL(64, 1);     \
  else if (nv <= 128) CALL(64, 2);  \
  else if (nv <= 256) CALL(64, 4);  \
  else if (nv <= 512) CALL(128, 4); \
  else if (nv <= 1024) CALL(256, 4); \
  else if (nv <= 2048) CALL(512, 4); \
  else CALL(1024, 4)
constexpr int kLnMaxVecs = 4096;  // longer rows take the looping kernels

// Rows of nv vectors that one launch takes: the runtime counts a grid's lanes
// in 32 bits and starts too few workgroups, without an error, above that.
constexpr int64_t ln_rows_per_launch(int64_t nv) {
  int64_t lanes = 64;
  while (lanes < 1024 && nv > 4 * lanes) lanes *= 2;
  return ((int64_t)UINT32_MAX - 1024) / lanes;
}
// launch(first row, rows) for every part of M rows.  No rows: one launch, of an
// empty grid, which refuses the call.
template <typename F>
Status ln_row_parts(int64_t M, int64_t nv, F&& launch) {
  const int64_t most = ln_rows_per_launch(nv);
  int64_t r = 0;
  do {
    const Status st = launch(r, (int)(M - r < most ? M - r : most));
    if (st != Status::Ok) return st;
    r += most;
  } while (r < M);
  return Status::Ok;
}

template <typename T>
Status ln_fwd_run(const T* x0, const T* g, const T* b, T* y0, float* mean0, float* rstd0, int64_t all, int N,
                  float eps, hipStream_t s) {
  const int64_t nv = ((int64_t)N + kVec<T> - 1) / kVec<T>;
  return ln_row_parts(all, nv, [&](int64_t r, int M) {
    const T* x = x0 + r * N;
    T* y = y0 + r * N;
    float *mean = mean0 + r, *rstd = rstd0 + r;
#define LN_FWD(LPR, VPT)                                                                                   \
  ln_fwd_kernel<T, LPR, VPT><<<(unsigned)(((int64_t)M * LPR + ln_threads(LPR) - 1) / ln_threads(LPR)),    \
                               ln_threads(LPR), 0, s>>>(x, g, b, y, mean, rstd, M, N, eps)
    const unsigned by_wave = (unsigned)(((int64_t)M + 3) / 4);
    if (N <= 64) ln_fwd_narrow_kernel<T><<<by_wave, 256, 0, s>>>(x, g, b, y, mean, rstd, M, N, eps);
    else if (nv > kLnMaxVecs) ln_fwd_loop_kernel<T><<<by_wave, 256, 0, s>>>(x, g, b, y, mean, rstd, M, N, eps);
    else LN_BY_WIDTH(LN_FWD);
#undef LN_FWD
    return launch_status("layernorm_fwd");
  });
}

// Whether out[k] shares no byte with an input or another output.
bool output_apart(const TensorDesc* in, int ni, const TensorDesc* out, int no, int k) {
  for (int i = 0; i < ni; ++i)
    if (views_overlap(out[k], in[i])) return false;
  for (int i = 0; i < no; ++i)
    if (i != k && views_overlap(out[k], out[i])) return false;
  return true;
}

// What a backward call's outputs allow.  Apart: dx may hold partial sums, and
// its rows may be written before other rows of x and dy have been read.
// OnDx: dx is x's or dy's memory.  OnSums: dgamma or dbeta is memory that the
// call reads or dx (an input may be given up for them): dx is complete before
// they are written.
enum class LnOut { Apart, OnDx, OnSums };
LnOut ln_bwd_outputs(const TensorDesc* in, int ni, const TensorDesc* out, int no) {
  for (int k = 1; k < no; ++k)
    if (!output_apart(in, ni, out, no, k)) return LnOut::OnSums;
  return output_apart(in, ni, out, no, 0) ? LnOut::Apart : LnOut::OnDx;
}

template <typename T>
Status ln_bwd_run(LnBwd<T> a, LnOut where, hipStream_t s) {
  constexpr int V = kVec<T>;
  const int M = a.M, N = a.N;
  const int64_t nv = ((int64_t)N + V - 1) / V;
  const bool affine = a.dgamma != nullptr;
  auto sums_loop = [&] {
    ln_bwd_dgdb_loop_kernel<T><<<(unsigned)(((int64_t)N + 63) / 64), 256, 0, s>>>(a.x, a.dy, a.mean, a.rstd,
                                                                                a.dgamma, a.dbeta, M, N);
    return launch_status("layernorm_bwd_dgdb");
  };
  auto in_order = [&](auto first, auto second) {
    const Status st = first();
    return st == Status::Ok ? second() : st;
  };
  const unsigned col_blocks = (unsigned)((nv + kLnColLanes - 1) / kLnColLanes);
  auto rows = [&](const LnBwd<T>& a, int64_t n, unsigned extra, bool reserved) {
#define LN_BWD(LPR, VPT)                                                                                 \
  do {                                                                                                   \
    const unsigned rb = (unsigned)((n * LPR + ln_threads(LPR) - 1) / ln_threads(LPR));                   \
    ln_bwd_kernel<T, LPR, VPT><<<rb + extra, ln_threads(LPR), 0, s>>>(a, (int)rb, reserved);             \
  } while (0)
    LN_BY_WIDTH(LN_BWD);
#undef LN_BWD
    return launch_status("layernorm_bwd");
  };
  auto dx_all = [&] {
    return ln_row_parts(M, nv, [&](int64_t r, int n) {
      LnBwd<T> p = a;
      p.x += r * N;
      p.dy += r * N;
      p.dx += r * N;
      p.mean += r;
      p.rstd += r;
      p.M = n;
      if (N > 64 && nv <= kLnMaxVecs) return rows(p, n, 0, false);
      const unsigned by_wave = (unsigned)(((int64_t)n + 3) / 4);
      if (N <= 64)
        ln_bwd_dx_narrow_kernel<T><<<by_wave, 256, 0, s>>>(p.x, p.dy, p.gamma, p.mean, p.rstd, p.dx, n, N);
      else
        ln_bwd_dx_loop_kernel<T><<<by_wave, 256, 0, s>>>(p.x, p.dy, p.gamma, p.mean, p.rstd, p.dx, n, N);
      return launch_status("layernorm_bwd");
    });
  };
  if (!affine || M < 1) return dx_all();
  // dx, then the sums, 64 columns a workgroup (which has read all of them when
  // it writes): the sums may lie on gamma, and at N <= 64 on any input
  if (where == LnOut::OnSums) return in_order(dx_all, sums_loop);
  // the kernels below step 32-bit row indices to less than 1024 past M
  if (N < V || nv > kLnMaxVecs || M > INT32_MAX - 1024) return in_order(sums_loop, dx_all);
  // Large matrices: x and dy read once, P chunks of rows (one workgroup per
  // CU), partial sums in dx.  Below 16 MiB (x and dy together an eighth of the
  // 256 MB MALL) the second read of the one-launch form comes from the caches
  // and its two launches less count more, until its N / 2 V column workgroups
  // have too many rows each: f32 [2048, 632] 10.6 us against 13.9 fused,
  // [4096, 512] 22.7 against 13.1, [16384, 100] 50 against 18.  8 rows a chunk at
  // least: the last launch reads the RS reserved ones of each again, at 8 rows a
  // quarter of x and dy in fp32 and half or more in f16, where the fused form is
  // the faster one all the same (f16 [2048, 8192] 45 us against 68, [2049, 8200]
  // 61 against 67, [2560, 4096] 30 against 42).
  constexpr int64_t kFusedBytes = 16 << 20;
  constexpr int kChunks = 256, kFusedRows = 3584;
  if (where == LnOut::Apart && nv <= 2048 && M >= 8 * kChunks && ((int64_t)M * N * (int64_t)sizeof(T) >= kFusedBytes || M >= kFusedRows)) {
    a.P = kChunks;
    a.q = M / kChunks;
    a.r = M % kChunks;
    a.RS = sizeof(T) == 4 ? 2 : ((N & 1) == 0 && aligned(a.dx, 4)) ? 4 : 5;
    // 16 columns a lane: more would spill at 1024 lanes (so would 1024 lanes
    // of fp32 columns, nv > 2048)
    constexpr int W = 16 / V;
    if (nv <= 64 * W) ln_bwd_fused_kernel<T, 64, W><<<kChunks, 1024, 0, s>>>(a);
    else if (nv <= 128 * W) ln_bwd_fused_kernel<T, 128, W><<<kChunks, 1024, 0, s>>>(a);
    else if (nv <= 256 * W) ln_bwd_fused_kernel<T, 256, W><<<kChunks, 1024, 0, s>>>(a);
    else if (nv <= 512 * W) ln_bwd_fused_kernel<T, 512, W><<<kChunks, 1024, 0, s>>>(a);
    else if constexpr (sizeof(T) == 2) ln_bwd_fused_kernel<T, 1024, W><<<kChunks, 1024, 0, s>>>(a);
    Status st = launch_status("layernorm_bwd_fused");
    if (st != Status::Ok) return st;
    ln_bwd_finish_kernel<T><<<(unsigned)((2 * (int64_t)N + 63) / 64), 1024, 0, s>>>(a);
    st = launch_status("layernorm_bwd_finish");
    if (st != Status::Ok) return st;
    return rows(a, (int64_t)a.P * a.RS, 0, true);
  }
  if (where == LnOut::OnDx || nv > 2048) {  // two launches: the sums before dx, or its rows take wider workgroups
    auto columns = [&] {
      ln_bwd_columns_kernel<T><<<col_blocks, kLnColThreads, 0, s>>>(a);
      return launch_status("layernorm_bwd_columns");
    };
    return in_order(columns, dx_all);
  }
  return rows(a, M, col_blocks, false);
}

#define LN_VARIANTS(SFX, T, D)                                                                          \
  bool ln_fwd_##SFX##_sup(const TensorDesc* i, int ni, const TensorDesc* o, int no, const void*) {    \
    return ln_fwd_check(i, ni, o, no, D);                                                              \
  }                                                                                                    \
  Status ln_fwd_##SFX##_launch(const TensorDesc* i, int ni, TensorDesc* o, int no, const void* a,      \
                               void*, size_t, void* s) {                                               \
    if (!ln_fwd_check(i, ni, o, no, D)) return Status::InvalidArgument;                               \
    const T* g = ni == 3 ? (const T*)i[1].data : nullptr;                                              \
    const T* b = ni == 3 ? (const T*)i[2].data : nullptr;                                              \
    return ln_fwd_run<T>((const T*)i[0].data, g, b, (T*)o[0].data, (float*)o[1].data,                 \
                         (float*)o[2].data, (int)i[0].shape[0], (int)i[0].shape[1], read_ln_eps(a),   \
                         as_stream(s));                                                               \
  }                                                                                                    \
  bool ln_bwd_##SFX##_sup(const TensorDesc* i, int ni, const TensorDesc* o, int no, const void*) {    \
    return ln_bwd_check(i, ni, o, no, D);                                                              \
  }                                                                                                    \
  Status ln_bwd_##SFX##_launch(const TensorDesc* i, int ni, TensorDesc* o, int no, const void*,        \
                               void*, size_t, void* s) {                                               \
    if (!ln_bwd_check(i, ni, o, no, D)) return Status::InvalidArgument;                               \
    const bool aff = ni == 5;                                                                          \
    LnBwd<T> b{};                                                                                      \
    b.x = (const T*)i[0].data;                                                                         \
    b.dy = (const T*)i[1].data;                                                                        \
    b.gamma = aff ? (const T*)i[2].data : nullptr;                                                     \
    b.mean = (const float*)i[aff ? 3 : 2].data;                                                        \
    b.rstd = (const float*)i[aff ? 4 : 3].data;                                                        \
    b.dx = (T*)o[0].data;                                                                              \
    b.dgamma = aff ? (float*)o[1].data : nullptr;                                                      \
    b.dbeta = aff ? (float*)o[2].data : nullptr;                                                       \
    b.M = (int)i[0].shape[0];                                                                          \
    b.N = (int)i[0].shape[1];                                                                          \
    return ln_bwd_run<T>(b, ln_bwd_outputs(i, ni, o, no), as_stream(s));                               \
  }

LN_VARIANTS(f32, float, DType::kF32)
LN_VARIANTS(f16, uint16_t, DType::kF16)

// ===========================================================================
// BatchNorm (f16, NCHW)
// ===========================================================================
// Element (n, c, hw) of channel c sits at n*C*HW + c*HW + hw: the channel is N
// slabs of HW contiguous elements.  The kernels below walk it in vectors of V
// elements (V divides HW), HV = HW / V of them a slab.
struct BNShape {
  int N, C, HW, HV;
};

template <int V>
struct BNVec {
  typedef uint16_t type __attribute__((ext_vector_type(V), aligned(2)));
};
template <>
struct BNVec<1> {
  typedef uint16_t type;
};
template <int V>
__device__ __forceinline__ float bn_get(const typename BNVec<V>::type& v, int e) {
  if constexpr (V == 1) return f16_to_f32(v);
  else return f16_to_f32(v[e]);
}
template <int V>
__device__ __forceinline__ void bn_set(typename BNVec<V>::type& v, int e, float f) {
  if constexpr (V == 1) v = f32_to_f16(f);
  else v[e] = f32_to_f16(f);
}

// Makes the compiler take v for a new value: it then converts v's elements
// again where they are used next instead of keeping them as fp32 (twice the
// registers, which spill at 1024 lanes).
template <int V>
__device__ __forceinline__ void bn_hide(typename BNVec<V>::type& v) {
  if constexpr (V == 1) {
    asm("" : "+v"(v));
  } else {
    typedef uint32_t words __attribute__((ext_vector_type(V / 2)));
    words w = __builtin_bit_cast(words, v);
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
      uint32_t x = w[i];
      asm("" : "+v"(x));
      w[i] = x;
    }
    v = __builtin_bit_cast(typename BNVec<V>::type, w);
  }
}

// Vector k, k + step, k + 2 step, ... of a channel: one division at the
// start, then the slab and the place in it are advanced.
template <int V>
struct BNWalk {
  int n, r, dn, dr;
  int HV;
  int64_t base, slab;  // of channel c in slab 0; elements from a slab to the next
  __device__ __forceinline__ BNWalk(const BNShape& s, int c, unsigned k, int step) {
    HV = s.HV;
    n = (int)(k / (unsigned)HV);
    r = (int)(k - (unsigned)n * (unsigned)HV);
    dn = step / HV;
    dr = step - dn * HV;
    base = (int64_t)c * s.HW;
    slab = (int64_t)s.C * s.HW;
  }
  __device__ __forceinline__ int64_t at() const { return base + n * slab + (int64_t)r * V; }
  __device__ __forceinline__ void next() {
    n += dn;
    r += dr;
    if (r >= HV) {
      r -= HV;
      ++n;
    }
  }
};

// Sum over a workgroup of NW waves, every thread gets it (fixed order).
template <int NW>
__device__ __forceinline__ float bn_block_sum(float v, float* red) {
  v = wave_sum(v);
  if constexpr (NW == 1) return v;
  __syncthreads();  // red is reused across calls
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = red[0];
#pragma unroll
  for (int k = 1; k < NW; ++k) s += red[k];
  return s;
}

// Mean and centred square sum of the workgroup's `cnt` elements, held in
// registers (vectors i of the lane, `live` of them).
template <int V, int T, int VPT>
__device__ __forceinline__ void bn_stats(typename BNVec<V>::type (&v)[VPT], int live, float cnt, float* red,
                                        float& mu, float& m2) {
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
#pragma unroll
    for (int e = 0; e < V; ++e) s += i < live ? bn_get<V>(v[i], e) : 0.0f;
  mu = bn_block_sum<T / 64>(s, red) / cnt;
#pragma unroll
  for (int i = 0; i < VPT; ++i) bn_hide<V>(v[i]);
  float d = 0.0f;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float t = i < live ? bn_get<V>(v[i], e) - mu : 0.0f;
      d = fmaf(t, t, d);
    }
  m2 = bn_block_sum<T / 64>(d, red);
#pragma unroll
  for (int i = 0; i < VPT; ++i) bn_hide<V>(v[i]);
}

// How many of the vectors t, t + T, ... are below n.
template <int T>
__device__ __forceinline__ int bn_live(int n) {
  const int left = n - (int)threadIdx.x;
  return left > 0 ? (left + T - 1) / T : 0;
}

// Training forward, channel in registers: batch mean, centred variance,
// rstd = 1/sqrt(var + eps), then y = (x - mean) rstd gamma + beta (gamma/beta
// null => 1/0).  One workgroup a channel, x read once, y may be x.
template <int V, int T, int VPT>
__global__ __launch_bounds__(T) void bn_fwd_reg_kernel(const uint16_t* x,
                                                       const uint16_t* gamma,
                                                       const uint16_t* beta, uint16_t* y,
                                                       float* save_mean,
                                                       float* save_rstd, BNShape sh, float eps) {
  typedef typename BNVec<V>::type vec;
  __shared__ float red[T / 64];
  const int c = blockIdx.x, total = sh.N * sh.HV;
  const int live = bn_live<T>(total);
  vec v[VPT];
  {
    BNWalk<V> w(sh, c, threadIdx.x, T);
#pragma unroll
    for (int i = 0; i < VPT; ++i, w.next())
      if (i < live) v[i] = *reinterpret_cast<const vec*>(x + w.at());
  }
  const float cnt = (float)((int64_t)sh.N * sh.HW);
  float mu, m2;
  bn_stats<V, T, VPT>(v, live, cnt, red, mu, m2);
  const float rs = 1.0f / sqrtf(m2 / cnt + eps);
  const float g = gamma ? f16_to_f32(gamma[c]) : 1.0f, b = beta ? f16_to_f32(beta[c]) : 0.0f;
  BNWalk<V> w(sh, c, threadIdx.x, T);
#pragma unroll
  for (int i = 0; i < VPT; ++i, w.next())
    if (i < live) {
      vec o;
#pragma unroll
      for (int e = 0; e < V; ++e) bn_set<V>(o, e, fmaf((bn_get<V>(v[i], e) - mu) * rs, g, b));
      *reinterpret_cast<vec*>(y + w.at()) = o;
    }
  if (threadIdx.x == 0) {
    save_mean[c] = mu;
    save_rstd[c] = rs;
  }
}

// Backward (affine), channel in registers: dbeta = sum(dy), dgamma = sum(dy
// xhat), dx = (NHW dy - dbeta - xhat dgamma) gamma rstd / NHW.  dx may be x or dy.
template <int V, int T, int VPT>
__global__ __launch_bounds__(T) void bn_bwd_reg_kernel(const uint16_t* x, const uint16_t* dy,
                                                       const uint16_t* gamma,
                                                       const float* mean,
                                                       const float* rstd, uint16_t* dx,
                                                       float* dgamma, float* dbeta,
                                                       BNShape sh) {
  typedef typename BNVec<V>::type vec;
  __shared__ float red[T / 64];
  const int c = blockIdx.x, total = sh.N * sh.HV;
  const int live = bn_live<T>(total);
  const float mu = mean[c], rs = rstd[c];
  vec v[VPT], d[VPT];
  {
    BNWalk<V> w(sh, c, threadIdx.x, T);
#pragma unroll
    for (int i = 0; i < VPT; ++i, w.next())
      if (i < live) {
        v[i] = *reinterpret_cast<const vec*>(x + w.at());
        d[i] = *reinterpret_cast<const vec*>(dy + w.at());
      }
  }
  float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (i < live) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float t = bn_get<V>(d[i], e);
        s1 += t;
        s2 = fmaf(t, (bn_get<V>(v[i], e) - mu) * rs, s2);
      }
    }
  s1 = bn_block_sum<T / 64>(s1, red);
  s2 = bn_block_sum<T / 64>(s2, red);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    bn_hide<V>(v[i]);
    bn_hide<V>(d[i]);
  }
  const float fcnt = (float)((int64_t)sh.N * sh.HW), scale = f16_to_f32(gamma[c]) * rs / fcnt;
  BNWalk<V> w(sh, c, threadIdx.x, T);
#pragma unroll
  for (int i = 0; i < VPT; ++i, w.next())
    if (i < live) {
      vec o;
#pragma unroll
      for (int e = 0; e < V; ++e)
        bn_set<V>(o, e, (fcnt * bn_get<V>(d[i], e) - s1 - (bn_get<V>(v[i], e) - mu) * rs * s2) * scale);
      *reinterpret_cast<vec*>(dx + w.at()) = o;
    }
  if (threadIdx.x == 0) {
    dgamma[c] = s2;
    dbeta[c] = s1;
  }
}

// Large channels: chunk p of channel c is kBNChunk vectors, one workgroup
// (p, c) each, whose two partial values go to part[c P + p]: forward, the
// chunk's mean and centred square sum; backward, its sums of dy and dy xhat.
// [32, 64, 56, 56]: 5.2 + 2.8 + 7.0 us in the three kernels forward and 6.2 +
// 1.8 + 8.2 backward, against 342 and 366 with one workgroup a channel (64 of
// 256 CUs), 2-byte loads and a 64-bit division an element; launches are now half
// of it.
constexpr int kBNVpt = 4, kBNChunk = 256 * kBNVpt;

template <int V>
__global__ __launch_bounds__(256) void bn_fwd_part_kernel(const uint16_t* __restrict__ x, f32x2_t* __restrict__ part,
                                                          BNShape sh) {
  typedef typename BNVec<V>::type vec;
  __shared__ float red[4];
  const int c = blockIdx.y, k0 = blockIdx.x * kBNChunk;
  const int left = sh.N * sh.HV - k0, here = left < kBNChunk ? left : kBNChunk;
  const int live = bn_live<256>(here);
  vec v[kBNVpt];
  BNWalk<V> w(sh, c, (unsigned)k0 + threadIdx.x, 256);
#pragma unroll
  for (int i = 0; i < kBNVpt; ++i, w.next())
    if (i < live) v[i] = *reinterpret_cast<const vec*>(x + w.at());
  float mu, m2;
  bn_stats<V, 256, kBNVpt>(v, live, (float)(here * V), red, mu, m2);
  if (threadIdx.x == 0) part[(int64_t)c * gridDim.x + blockIdx.x] = f32x2_t{mu, m2};
}

// A wave a channel: the chunks' means and square sums merged (the mean of the
// means by their counts, then the square sums about it).
template <int V>
__global__ __launch_bounds__(256) void bn_fwd_finish_kernel(const f32x2_t* __restrict__ part,
                                                            float* __restrict__ save_mean,
                                                            float* __restrict__ save_rstd, BNShape sh, int P,
                                                            float eps) {
  const int lane = threadIdx.x & 63, c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= sh.C) return;  // whole wave
  const f32x2_t* q = part + (int64_t)c * P;
  const int total = sh.N * sh.HV;
  auto count = [&](int p) {
    const int left = total - p * kBNChunk;
    return (float)((left < kBNChunk ? left : kBNChunk) * V);
  };
  const float cnt = (float)((int64_t)sh.N * sh.HW);
  float s = 0.0f;
  for (int p = lane; p < P; p += 64) s += q[p][0] * count(p);
  const float mu = wave_sum(s) / cnt;
  float d = 0.0f;
  for (int p = lane; p < P; p += 64) {
    const float t = q[p][0] - mu;
    d += fmaf(count(p) * t, t, q[p][1]);
  }
  const float m2 = wave_sum(d);
  if (lane == 0) {
    save_mean[c] = mu;
    save_rstd[c] = 1.0f / sqrtf(m2 / cnt + eps);
  }
}

template <int V>
__global__ __launch_bounds__(256) void bn_bwd_part_kernel(const uint16_t* __restrict__ x,
                                                          const uint16_t* __restrict__ dy,
                                                          const float* __restrict__ mean,
                                                          const float* __restrict__ rstd,
                                                          f32x2_t* __restrict__ part, BNShape sh) {
  typedef typename BNVec<V>::type vec;
  __shared__ float red[4];
  const int c = blockIdx.y, k0 = blockIdx.x * kBNChunk;
  const int left = sh.N * sh.HV - k0, here = left < kBNChunk ? left : kBNChunk;
  const int live = bn_live<256>(here);
  const float mu = mean[c], rs = rstd[c];
  vec v[kBNVpt], d[kBNVpt];
  BNWalk<V> w(sh, c, (unsigned)k0 + threadIdx.x, 256);
#pragma unroll
  for (int i = 0; i < kBNVpt; ++i, w.next())
    if (i < live) {
      v[i] = *reinterpret_cast<const vec*>(x + w.at());
      d[i] = *reinterpret_cast<const vec*>(dy + w.at());
    }
  float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
  for (int i = 0; i < kBNVpt; ++i)
    if (i < live) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float t = bn_get<V>(d[i], e);
        s1 += t;
        s2 = fmaf(t, (bn_get<V>(v[i], e) - mu) * rs, s2);
      }
    }
  s1 = bn_block_sum<4>(s1, red);
  s2 = bn_block_sum<4>(s2, red);
  if (threadIdx.x == 0) part[(int64_t)c * gridDim.x + blockIdx.x] = f32x2_t{s1, s2};
}

__global__ __launch_bounds__(256) void bn_bwd_finish_kernel(const f32x2_t* __restrict__ part,
                                                            float* __restrict__ dgamma, float* __restrict__ dbeta,
                                                            int C, int P) {
  const int lane = threadIdx.x & 63, c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= C) return;  // whole wave
  const f32x2_t* q = part + (int64_t)c * P;
  float s1 = 0.0f, s2 = 0.0f;
  for (int p = lane; p < P; p += 64) {
    s1 += q[p][0];
    s2 += q[p][1];
  }
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  if (lane == 0) {
    dgamma[c] = s2;
    dbeta[c] = s1;
  }
}

// y = (x - mean) rstd gamma + beta, a vector a lane; blockIdx.y walks the
// batch.  VAR: `second` is the running variance, rstd = 1/sqrt(var + eps)
// (inference); else it is the saved rstd.
template <int V, bool VAR>
__global__ __launch_bounds__(256) void bn_fwd_apply_kernel(const uint16_t* x,
                                                           const uint16_t* gamma,
                                                           const uint16_t* beta,
                                                           const float* mean,
                                                           const float* second,
                                                           uint16_t* y, BNShape sh, float eps) {
  typedef typename BNVec<V>::type vec;
  const int64_t per = (int64_t)sh.C * sh.HV;  // vectors a batch entry
  for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < per; k += (int64_t)gridDim.x * 256) {
    const int c = per <= INT32_MAX ? (int)((unsigned)k / (unsigned)sh.HV) : (int)(k / sh.HV);
    const float mu = mean[c], rs = VAR ? 1.0f / sqrtf(second[c] + eps) : second[c];
    const float g = gamma ? f16_to_f32(gamma[c]) : 1.0f, b = beta ? f16_to_f32(beta[c]) : 0.0f;
    for (int n = blockIdx.y; n < sh.N; n += gridDim.y) {
      const int64_t at = (n * per + k) * V;
      const vec v = *reinterpret_cast<const vec*>(x + at);
      vec o;
#pragma unroll
      for (int e = 0; e < V; ++e) bn_set<V>(o, e, fmaf((bn_get<V>(v, e) - mu) * rs, g, b));
      *reinterpret_cast<vec*>(y + at) = o;
    }
  }
}

template <int V>
__global__ __launch_bounds__(256) void bn_bwd_apply_kernel(const uint16_t* x,
                                                           const uint16_t* dy,
                                                           const uint16_t* gamma,
                                                           const float* mean,
                                                           const float* rstd,
                                                           const float* dgamma,
                                                           const float* dbeta,
                                                           uint16_t* dx, BNShape sh) {
  typedef typename BNVec<V>::type vec;
  const int64_t per = (int64_t)sh.C * sh.HV;  // vectors a batch entry
  for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < per; k += (int64_t)gridDim.x * 256) {
    const int c = per <= INT32_MAX ? (int)((unsigned)k / (unsigned)sh.HV) : (int)(k / sh.HV);
    const float mu = mean[c], rs = rstd[c], s2 = dgamma[c], s1 = dbeta[c];
    const float fcnt = (float)((int64_t)sh.N * sh.HW), scale = f16_to_f32(gamma[c]) * rs / fcnt;
    for (int n = blockIdx.y; n < sh.N; n += gridDim.y) {
      const int64_t at = (n * per + k) * V;
      const vec v = *reinterpret_cast<const vec*>(x + at), d = *reinterpret_cast<const vec*>(dy + at);
      vec o;
#pragma unroll
      for (int e = 0; e < V; ++e)
        bn_set<V>(o, e, (fcnt * bn_get<V>(d, e) - s1 - (bn_get<V>(v, e) - mu) * rs * s2) * scale);
      *reinterpret_cast<vec*>(dx + at) = o;
    }
  }
}

// Channels too large for registers that cannot be split over workgroups (an
// output shares memory with an input): one workgroup a channel, x read from
// memory for each pass.
__device__ __forceinline__ int64_t bn_index(const BNShape& s, int c, int64_t k) {
  const int64_t n = k / s.HW, hw = k - n * s.HW;
  return (n * s.C + c) * (int64_t)s.HW + hw;
}
__global__ __launch_bounds__(256) void bn_fwd_loop_kernel(const uint16_t* x, const uint16_t* gamma,
                                                          const uint16_t* beta, uint16_t* y, float* save_mean,
                                                          float* save_rstd, BNShape sh, float eps) {
  __shared__ float red[4];
  const int c = blockIdx.x;
  const int64_t cnt = (int64_t)sh.N * sh.HW;
  float s = 0.0f;
  for (int64_t k = threadIdx.x; k < cnt; k += 256) s += f16_to_f32(x[bn_index(sh, c, k)]);
  const float mu = bn_block_sum<4>(s, red) / (float)cnt;
  float d = 0.0f;
  for (int64_t k = threadIdx.x; k < cnt; k += 256) {
    const float t = f16_to_f32(x[bn_index(sh, c, k)]) - mu;
    d = fmaf(t, t, d);
  }
  const float rs = 1.0f / sqrtf(bn_block_sum<4>(d, red) / (float)cnt + eps);
  const float g = gamma ? f16_to_f32(gamma[c]) : 1.0f, b = beta ? f16_to_f32(beta[c]) : 0.0f;
  for (int64_t k = threadIdx.x; k < cnt; k += 256) {
    const int64_t i = bn_index(sh, c, k);
    y[i] = f32_to_f16(fmaf((f16_to_f32(x[i]) - mu) * rs, g, b));
  }
  if (threadIdx.x == 0) {
    save_mean[c] = mu;
    save_rstd[c] = rs;
  }
}
__global__ __launch_bounds__(256) void bn_bwd_loop_kernel(const uint16_t* x, const uint16_t* dy,
                                                          const uint16_t* gamma, const float* mean,
                                                          const float* rstd, uint16_t* dx, float* dgamma,
                                                          float* dbeta, BNShape sh) {
  __shared__ float red[4];
  const int c = blockIdx.x;
  const int64_t cnt = (int64_t)sh.N * sh.HW;
  const float mu = mean[c], rs = rstd[c];
  float s1 = 0.0f, s2 = 0.0f;
  for (int64_t k = threadIdx.x; k < cnt; k += 256) {
    const int64_t i = bn_index(sh, c, k);
    const float d = f16_to_f32(dy[i]);
    s1 += d;
    s2 = fmaf(d, (f16_to_f32(x[i]) - mu) * rs, s2);
  }
  s1 = bn_block_sum<4>(s1, red);
  s2 = bn_block_sum<4>(s2, red);
  const float fcnt = (float)cnt, scale = f16_to_f32(gamma[c]) * rs / fcnt;
  for (int64_t k = threadIdx.x; k < cnt; k += 256) {
    const int64_t i = bn_index(sh, c, k);
    const float xh = (f16_to_f32(x[i]) - mu) * rs;
    dx[i] = f32_to_f16((fcnt * f16_to_f32(dy[i]) - s1 - xh * s2) * scale);
  }
  if (threadIdx.x == 0) {
    dgamma[c] = s2;
    dbeta[c] = s1;
  }
}

// Whether a channel may be split over workgroups and kernels: the large output
// holds partial sums while the inputs are read, and the per-channel outputs
// are written by one kernel and read by the next, so none of them shares a
// byte with an input or another output.  (One workgroup a channel reads all
// that it needs of its channel before it writes.)
bool bn_outputs_apart(const TensorDesc* in, int ni, const TensorDesc* out, int no) {
  for (int k = 0; k < no; ++k)
    if (!output_apart(in, ni, out, no, k)) return false;
  return true;
}

// Launch shape of a register-resident channel by its vectors: (threads,
// vectors a lane), up to 8192 vectors.
#define BN_REG_BY_SIZE(V, total, CALL)                  \
  if constexpr (V == 1) {                               \
    if (total <= 64 * 8) { CALL(1, 64, 8); }            \
    else if (total <= 256 * 16) { CALL(1, 256, 16); }   \
    else { CALL(1, 1024, 8); }                         \
  } else {                                              \
    if (total <= 64 * 4) { CALL(V, 64, 4); }            \
    else if (total <= 256 * 4) { CALL(V, 256, 4); }     \
    else if (total <= 512 * 8) { CALL(V, 512, 8); }     \
    else { CALL(V, 1024, 8); }                          \
  }
// The runtime counts a grid's lanes in 32 bits and starts too few workgroups,
// without an error, above that: no more channels of over 256 lanes than fit.
bool bn_in_registers(int64_t total, int64_t C) { return total <= 1024 || (total <= 1024 * 8 && C < 1 << 22); }

template <int V>
dim3 bn_apply_grid(const BNShape& sh) {
  return dim3(grid_1d((int64_t)sh.C * sh.HV, 256, 1 << 22), (unsigned)(sh.N < 65535 ? sh.N : 65535));
}

template <int V>
Status bn_fwd_train(const uint16_t* x, const uint16_t* g, const uint16_t* b, uint16_t* y, float* sm, float* sr,
                    BNShape sh, float eps, bool apart, hipStream_t s) {
  sh.HV = sh.HW / V;
  const int64_t total = (int64_t)sh.N * sh.HV;
  if (bn_in_registers(total, sh.C)) {
#define BN_FWD(VV, T, VPT) bn_fwd_reg_kernel<VV, T, VPT><<<(unsigned)sh.C, T, 0, s>>>(x, g, b, y, sm, sr, sh, eps)
    BN_REG_BY_SIZE(V, total, BN_FWD)
#undef BN_FWD
    return launch_status("batchnorm_fwd");
  }
  if (!apart || sh.C > 65535 || (int64_t)sh.C * sh.HW > INT32_MAX) {
    bn_fwd_loop_kernel<<<(unsigned)sh.C, 256, 0, s>>>(x, g, b, y, sm, sr, sh, eps);
    return launch_status("batchnorm_fwd");
  }
  const int P = (int)((total + kBNChunk - 1) / kBNChunk);
  f32x2_t* part = reinterpret_cast<f32x2_t*>(((uintptr_t)y + 7) & ~(uintptr_t)7);
  bn_fwd_part_kernel<V><<<dim3((unsigned)P, (unsigned)sh.C), 256, 0, s>>>(x, part, sh);
  Status st = launch_status("batchnorm_fwd_part");
  if (st != Status::Ok) return st;
  bn_fwd_finish_kernel<V><<<(unsigned)((sh.C + 3) / 4), 256, 0, s>>>(part, sm, sr, sh, P, eps);
  st = launch_status("batchnorm_fwd_finish");
  if (st != Status::Ok) return st;
  bn_fwd_apply_kernel<V, false><<<bn_apply_grid<V>(sh), 256, 0, s>>>(x, g, b, sm, sr, y, sh, eps);
  return launch_status("batchnorm_fwd");
}

template <int V>
Status bn_fwd_infer(const uint16_t* x, const uint16_t* g, const uint16_t* b, const float* rm, const float* rv,
                    uint16_t* y, BNShape sh, float eps, hipStream_t s) {
  sh.HV = sh.HW / V;
  bn_fwd_apply_kernel<V, true><<<bn_apply_grid<V>(sh), 256, 0, s>>>(x, g, b, rm, rv, y, sh, eps);
  return launch_status("batchnorm_fwd");
}

template <int V>
Status bn_bwd_run(const uint16_t* x, const uint16_t* dy, const uint16_t* g, const float* sm, const float* sr,
                  uint16_t* dx, float* dg, float* db, BNShape sh, bool apart, hipStream_t s) {
  sh.HV = sh.HW / V;
  const int64_t total = (int64_t)sh.N * sh.HV;
  if (bn_in_registers(total, sh.C)) {
#define BN_BWD(VV, T, VPT) \
  bn_bwd_reg_kernel<VV, T, VPT><<<(unsigned)sh.C, T, 0, s>>>(x, dy, g, sm, sr, dx, dg, db, sh)
    BN_REG_BY_SIZE(V, total, BN_BWD)
#undef BN_BWD
    return launch_status("batchnorm_bwd");
  }
  if (!apart || sh.C > 65535 || (int64_t)sh.C * sh.HW > INT32_MAX) {
    bn_bwd_loop_kernel<<<(unsigned)sh.C, 256, 0, s>>>(x, dy, g, sm, sr, dx, dg, db, sh);
    return launch_status("batchnorm_bwd");
  }
  const int P = (int)((total + kBNChunk - 1) / kBNChunk);
  f32x2_t* part = reinterpret_cast<f32x2_t*>(((uintptr_t)dx + 7) & ~(uintptr_t)7);
  bn_bwd_part_kernel<V><<<dim3((unsigned)P, (unsigned)sh.C), 256, 0, s>>>(x, dy, sm, sr, part, sh);
  Status st = launch_status("batchnorm_bwd_part");
  if (st != Status::Ok) return st;
  bn_bwd_finish_kernel<<<(unsigned)((sh.C + 3) / 4), 256, 0, s>>>(part, dg, db, sh.C, P);
  st = launch_status("batchnorm_bwd_finish");
  if (st != Status::Ok) return st;
  bn_bwd_apply_kernel<V><<<bn_apply_grid<V>(sh), 256, 0, s>>>(x, dy, g, sm, sr, dg, db, dx, sh);
  return launch_status("batchnorm_bwd");
}

struct BNAttr {
  float eps = 1e-5f;
  bool use_running_stats = true;
};
// batchnorm/launcher.cu:69-84: BNEP <fI> with >= 8 bytes, else defaults.
BNAttr read_bn_attr(const void* attr) {
  BNAttr r;
  const AttrBlob& a = blob(attr);
  if (!attr || a.schema_id != AICF_SCHEMA_BNEP || !payload_ok(a, 8)) return r;
  r.eps = field<float>(a, 0);
  r.use_running_stats = (field<uint32_t>(a, 4) & 1u) != 0;
  return r;
}

bool nchw_f16(const TensorDesc& t) {
  if (dt(t) != DType::kF16 || t.rank != 4) return false;
  for (int i = 0; i < 4; ++i)
    if (t.stride[i] <= 0 || t.shape[i] <= 0) return false;
  return t.stride[3] == 1 && t.stride[2] == t.shape[3] && t.stride[1] == t.shape[2] * t.shape[3] &&
         t.stride[0] == t.shape[1] * t.shape[2] * t.shape[3];
}
bool vec_c(const TensorDesc& t, DType d, int64_t C) { return dt(t) == d && t.rank == 1 && t.shape[0] == C; }

// batchnorm/launcher.cu:295-345: inference (X,G,B,RM,RV)->(Y) or (X,RM,RV)->(Y);
// training (X,G,B)->(Y,SM,SR) or (X)->(Y,SM,SR).
bool bn_fwd_sup(const TensorDesc* in, int ni, const TensorDesc* out, int no, const void*) {
  if (!in || !out) return false;
  const bool inf_aff = ni == 5 && no == 1, inf_no = ni == 3 && no == 1;
  const bool tr_aff = ni == 3 && no == 3, tr_no = ni == 1 && no == 3;
  if (!(inf_aff || inf_no || tr_aff || tr_no)) return false;
  const TensorDesc &X = in[0], &Y = out[0];
  if (!nchw_f16(X) || !nchw_f16(Y) || !same_shape(X, Y)) return false;
  const int64_t C = X.shape[1];
  if (X.shape[0] * X.shape[2] * X.shape[3] > INT32_MAX) return false;
  if ((inf_aff || tr_aff) && (!vec_c(in[1], DType::kF16, C) || !vec_c(in[2], DType::kF16, C))) return false;
  if (inf_aff || inf_no) return vec_c(in[inf_aff ? 3 : 1], DType::kF32, C) && vec_c(in[inf_aff ? 4 : 2], DType::kF32, C);
  return vec_c(out[1], DType::kF32, C) && vec_c(out[2], DType::kF32, C);
}

Status bn_fwd_launch(const TensorDesc* in, int ni, TensorDesc* out, int no, const void* attr, void*, size_t,
                     void* stream) {
  if (!bn_fwd_sup(in, ni, out, no, attr)) return Status::InvalidArgument;
  const BNAttr A = read_bn_attr(attr);
  const bool training = no == 3;
  if (training && A.use_running_stats) return Status::InvalidArgument;  // launcher.cu:364-366
  const TensorDesc& X = in[0];
  const BNShape sh{(int)X.shape[0], (int)X.shape[1], (int)(X.shape[2] * X.shape[3]), 0};
  hipStream_t s = as_stream(stream);
  const uint16_t* x = (const uint16_t*)X.data;
  uint16_t* y = (uint16_t*)out[0].data;
  if (training) {
    const uint16_t* g = ni == 3 ? (const uint16_t*)in[1].data : nullptr;
    const uint16_t* b = ni == 3 ? (const uint16_t*)in[2].data : nullptr;
    float *sm = (float*)out[1].data, *sr = (float*)out[2].data;
    const bool apart = bn_outputs_apart(in, ni, out, no);
    if (sh.HW % 8 == 0) return bn_fwd_train<8>(x, g, b, y, sm, sr, sh, A.eps, apart, s);
    if (sh.HW % 4 == 0) return bn_fwd_train<4>(x, g, b, y, sm, sr, sh, A.eps, apart, s);
    return bn_fwd_train<1>(x, g, b, y, sm, sr, sh, A.eps, apart, s);
  }
  const bool aff = ni == 5;
  const uint16_t* g = aff ? (const uint16_t*)in[1].data : nullptr;
  const uint16_t* b = aff ? (const uint16_t*)in[2].data : nullptr;
  const float *rm = (const float*)in[aff ? 3 : 1].data, *rv = (const float*)in[aff ? 4 : 2].data;
  if (sh.HW % 8 == 0) return bn_fwd_infer<8>(x, g, b, rm, rv, y, sh, A.eps, s);
  if (sh.HW % 4 == 0) return bn_fwd_infer<4>(x, g, b, rm, rv, y, sh, A.eps, s);
  return bn_fwd_infer<1>(x, g, b, rm, rv, y, sh, A.eps, s);
}

// batchnorm/launcher.cu:483-526: (X, dY, G, SM, SR) -> (dX, dG, dB); the
// non-affine form (X, dY, SM, SR) -> (dX) is accepted by supported() and
// answered with NotImplemented at launch, as in the reference.
bool bn_bwd_sup(const TensorDesc* in, int ni, const TensorDesc* out, int no, const void*) {
  if (!in || !out) return false;
  const bool affine = ni == 5 && no == 3, noaff = ni == 4 && no == 1;
  if (!affine && !noaff) return false;
  const TensorDesc &X = in[0], &dY = in[1], &dX = out[0];
  if (!nchw_f16(X) || !nchw_f16(dY) || !nchw_f16(dX) || !same_shape(X, dY) || !same_shape(X, dX)) return false;
  const int64_t C = X.shape[1];
  if (X.shape[0] * X.shape[2] * X.shape[3] > INT32_MAX) return false;
  if (!vec_c(in[affine ? 3 : 2], DType::kF32, C) || !vec_c(in[affine ? 4 : 3], DType::kF32, C)) return false;
  if (affine && (!vec_c(in[2], DType::kF16, C) || !vec_c(out[1], DType::kF32, C) || !vec_c(out[2], DType::kF32, C)))
    return false;
  return true;
}

Status bn_bwd_launch(const TensorDesc* in, int ni, TensorDesc* out, int no, const void* attr, void*, size_t,
                     void* stream) {
  if (!bn_bwd_sup(in, ni, out, no, attr)) return Status::InvalidArgument;
  if (ni != 5) return Status::NotImplemented;
  const TensorDesc& X = in[0];
  const BNShape sh{(int)X.shape[0], (int)X.shape[1], (int)(X.shape[2] * X.shape[3]), 0};
  const uint16_t *x = (const uint16_t*)X.data, *dy = (const uint16_t*)in[1].data, *g = (const uint16_t*)in[2].data;
  const float *sm = (const float*)in[3].data, *sr = (const float*)in[4].data;
  uint16_t* dx = (uint16_t*)out[0].data;
  float *dg = (float*)out[1].data, *db = (float*)out[2].data;
  const bool apart = bn_outputs_apart(in, ni, out, no);
  hipStream_t s = as_stream(stream);
  if (sh.HW % 8 == 0) return bn_bwd_run<8>(x, dy, g, sm, sr, dx, dg, db, sh, apart, s);
  if (sh.HW % 4 == 0) return bn_bwd_run<4>(x, dy, g, sm, sr, dx, dg, db, sh, apart, s);
  return bn_bwd_run<1>(x, dy, g, sm, sr, dx, dg, db, sh, apart, s);
}

}  // namespace

KernelVariant make_layernorm_fwd_f32_variant() {
  return make("layernorm_fwd_f32_contig2d", ln_fwd_f32_launch, ln_fwd_f32_sup, AICF_SCHEMA_LNEP);
}
KernelVariant make_layernorm_fwd_f16_variant() {
  return make("layernorm_fwd_f16_contig2d", ln_fwd_f16_launch, ln_fwd_f16_sup, AICF_SCHEMA_LNEP);
}
KernelVariant make_layernorm_bwd_f32_variant() {
  return make("layernorm_bwd_f32_contig2d", ln_bwd_f32_launch, ln_bwd_f32_sup);
}
KernelVariant make_layernorm_bwd_f16_variant() {
  return make("layernorm_bwd_f16_contig2d", ln_bwd_f16_launch, ln_bwd_f16_sup);
}
KernelVariant make_batchnorm_fwd_f16_variant() {
  return make("batchnorm_fwd_f16_nchw", bn_fwd_launch, bn_fwd_sup, AICF_SCHEMA_BNEP);
}
KernelVariant make_batchnorm_bwd_f16_variant() {
  return make("batchnorm_bwd_f16_nchw_affine", bn_bwd_launch, bn_bwd_sup);
}

}  // namespace aicf::hip
