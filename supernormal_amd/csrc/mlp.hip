// The SDF MLP of models/fields.py:85-99 (input_concat: h0 = [x, enc]; NH
// hidden layers of width H with Softplus(beta, threshold 20); linear output of
// width 1) in fp32 on the fp32 matrix cores (v_mfma_f32_16x16x4f32), the
// activations in registers from layer to layer.
//
// Layout.  Every layer is computed transposed, Z^T = W * H^T: units are the
// MFMA rows and 16 points of a wavefront its columns.  With lane l, r = l % 16,
// q = l / 16 one MFMA takes A[r][q], B[q][r] and returns D[4q + e][r], so a lane
// ends a layer with point r's units 16 mb + 4q + e.  A dot product does not
// depend on the order of K as long as A and B agree; the K axis of the next
// layer is taken as step (mb, e), slot q -> unit 16 mb + 4q + e, which makes
// the lane's own value (mb, e) its B operand, and the four weights of steps
// (mb, 0..3) four consecutive floats of a weight row: one 16-byte LDS read per
// four MFMAs (rows padded by 4 floats: conflict-free), no activation through
// LDS.  The transposed products (W^T g of the backward) read the same weights
// column-wise, one 4-byte read per MFMA.  h0 is held as [enc | x | 0 ...] in
// KB blocks of 16 dims, so that a lane's four dims of a block are one 16-byte
// load of the encoding.
//
// Weight gradients need the points on the K axis: each step's gradient and
// activation blocks go through two fp32 LDS tiles (64 rows x 64 points of a
// workgroup's step) and back as 16-byte operands; the blocks are split over
// the wavefronts.  Per-workgroup partial rows are summed in a fixed order by
// mlp_reduce_rows, so results do not depend on scheduling (no float atomics).
//
// Bound: the fp32 matrix rate (32 cycles per MFMA and SIMD; 100 MFMAs per 16
// points forward, ~330 backward at 35 -> 64 -> 64 -> 1) and the softplus VALU
// work beside it.  Operands through LDS tiles with a wavefront per SIMD (the
// weights and every activation in LDS) had measured 387 us forward and 560 us
// backward over 299 593 points; 77 and 186 us with the activations in
// registers.
//
// Packed parameter layout (fp32, row-major; the gradient uses the same):
//   W0[H][d_in] b0[H] { W1[H][H] b1[H] } wo[H] bo
#include "sn_common.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace sn {

constexpr int kWaves = 4;
constexpr float kSpThr = 20.f;

// The lane's row and quarter, opaque to the compiler at each use: LDS
// addresses derive from them and are formed where used; as loop invariants
// they had been hoisted and held in ~80 registers.
struct Lane {
  int r, q;
};
__device__ __forceinline__ Lane lane_here() {
  Lane v{(int)threadIdx.x & 15, ((int)threadIdx.x & 63) >> 4};
  asm volatile("" : "+v"(v.r), "+v"(v.q));
  return v;
}

__device__ __forceinline__ floatx4 mma(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Softplus(beta) with torch's threshold (z above it): value h, derivative
// d = sigma(beta z) and its complement c = 1 - d (s'' = beta d c; 0 above the
// threshold, where torch's derivative is the constant 1).  Branch-free, from
// t = e^(-|beta z|) in (0, 1]: h = max(z, 0) + log1p(t) / beta (the large part
// exact; log(1 + e^(beta z)) / beta from the hardware logarithm had a mean
// error of -4e-8 in the sdf), d and c are 1 / (1 + t) and t / (1 + t).  On the
// hardware exp2 / log2 / reciprocal, completed to about the accuracy of the
// library functions: the low part of beta z log2(e) is multiplied back, log1p
// takes the rounding of 1 + t as a correction, the reciprocal one Newton step.
// A NaN z gives a NaN value.
struct Sp {
  float h, d, c;
};
template <bool kSecond = false>
__device__ __forceinline__ Sp softplus(float z, float beta, float inv_beta) {
  constexpr float kLog2e = 1.44269502f, kLog2eLo = 1.92596303e-8f, kLn2 = 0.693147182f;
  const float bz = z * beta, a = -fabsf(bz);
  const float p = a * kLog2e;
  const float lo = fmaf(a, kLog2eLo, fmaf(a, kLog2e, -p)) * kLn2;
  const float t0 = __builtin_amdgcn_exp2f(p);
  const float t = fmaf(t0, lo, t0);
  const float u = 1.f + t;
  const float r0 = __builtin_amdgcn_rcpf(u);
  const float r = fmaf(fmaf(-u, r0, 1.f), r0, r0);
  const float tr = t * r;
  const bool lin = bz > kSpThr, pos = bz >= 0.f;
  Sp s;
  const float l = fmaf(t - (u - 1.f), r, __builtin_amdgcn_logf(u) * kLn2) * inv_beta;
  s.h = lin ? z : (pos ? z : 0.f) + l;
  s.d = lin ? 1.f : (pos ? r : tr);
  s.c = lin ? 0.f : (pos ? tr : r);
  // selected here: sunk to their uses, the selections' masks are held instead
  asm volatile("" : "+v"(s.h), "+v"(s.d));
  if (kSecond) asm volatile("" : "+v"(s.c));
  return s;
}

template <int H, int NH, int KB>
struct Mlp {
  static constexpr int MB = H / 16;
  static constexpr int D0 = 16 * KB;  // padded input dims
  static constexpr int LD0 = D0 + 4, LD1 = H + 4;
  // LDS (floats): weights, vectors b0 b1 wo bo, then the two block tiles
  static constexpr int oW1 = H * LD0;
  static constexpr int oVec = oW1 + (NH == 2 ? H * LD1 : 0);
  static constexpr int kFwd = oVec + 3 * H + 4;
  static constexpr int kRowsB = H > D0 ? H : D0;
  static constexpr int kTileP = 16 * kWaves + 4;
  static constexpr int oTA = kFwd, oTB = oTA + H * kTileP;
  static constexpr int kBwd = oTB + kRowsB * kTileP;
  // weight-gradient blocks: wavefront w owns column block w % MB of dW1 and
  // row block w % MB of dW0, and every (kWaves / MB)-th of the other index
  static constexpr int S = kWaves / MB;
  static constexpr int T1 = NH == 2 ? MB / S : 1, T0 = (KB + S - 1) / S;
  // packed parameter offsets
  __host__ __device__ static int n_params(int d) {
    return H * d + H + (NH == 2 ? H * H + H : 0) + H + 1;
  }
  __host__ __device__ static int gB0(int d) { return H * d; }
  __host__ __device__ static int gW1(int d) { return H * d + H; }
  __host__ __device__ static int gB1(int d) { return H * d + H + H * H; }
  __host__ __device__ static int gWo(int d) { return H * d + H + (NH == 2 ? H * H + H : 0); }
  __host__ __device__ static int gBo(int d) { return gWo(d) + H; }
};

// packed W0 column of input dim c ([enc | x | pad]); -1 for padding
__device__ __forceinline__ int in_col(int c, int E) {
  return c < E ? 3 + c : (c < E + 3 ? c - E : -1);
}

template <int H, int NH, int KB>
__device__ void load_weights(float* sw, const float* __restrict__ mlp, int E) {
  using M = Mlp<H, NH, KB>;
  const int d = 3 + E;
  for (int t = threadIdx.x; t < H * M::LD0; t += blockDim.x) {
    const int o = t / M::LD0, c = t % M::LD0;
    const int col = c < M::D0 ? in_col(c, E) : -1;
    sw[t] = col >= 0 ? mlp[o * d + col] : 0.f;
  }
  if (NH == 2)
    for (int t = threadIdx.x; t < H * M::LD1; t += blockDim.x) {
      const int o = t / M::LD1, c = t % M::LD1;
      sw[M::oW1 + t] = c < H ? mlp[M::gW1(d) + o * H + c] : 0.f;
    }
  float* vec = sw + M::oVec;
  for (int t = threadIdx.x; t < H; t += blockDim.x) {
    vec[t] = mlp[M::gB0(d) + t];
    vec[H + t] = NH == 2 ? mlp[M::gB1(d) + t] : 0.f;
    vec[2 * H + t] = mlp[M::gWo(d) + t];
  }
  if (threadIdx.x == 0) vec[3 * H] = mlp[M::gBo(d)];
}

// The 4 input dims 16 kb + 4q .. +3 of point p, zero past n and past E + 3.
// With vec4 (E % 4 == 0, 16-byte rows) they are encoding dims (one load), the
// position, or padding; otherwise one guarded load per dim.  vec4 = 2: the
// encoding by levels ([E / 2][n_cap][2], see hash_fwd_levels_kernel).
__device__ __forceinline__ void load_in(const float* __restrict__ x, const float* __restrict__ enc,
                                        int E, int vec4, int64_t n_cap, int64_t p, bool ok, int c4,
                                        float (&v)[4]) {
  if (vec4) {
    float4 a = {0.f, 0.f, 0.f, 0.f};
    if (ok && c4 < E) {
      if (vec4 == 2) {
        const float2* e2 = reinterpret_cast<const float2*>(enc) + (int64_t)(c4 >> 1) * n_cap + p;
        const float2 lo = e2[0], hi = e2[n_cap];
        a = float4{lo.x, lo.y, hi.x, hi.y};
      } else {
        a = *reinterpret_cast<const float4*>(enc + p * E + c4);
      }
    } else if (ok && c4 == E) a = float4{x[p * 3], x[p * 3 + 1], x[p * 3 + 2], 0.f};
    v[0] = a.x;
    v[1] = a.y;
    v[2] = a.z;
    v[3] = a.w;
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = c4 + j;
    const float* src = c < E ? enc + p * E + c : x + p * 3 + (c - E);
    v[j] = 0.f;
    if (ok && c < E + 3) v[j] = *src;
  }
}

// z[mb] += W (rows 16 mb + r) * b over NB blocks of 16 K dims.  (The scheduling
// barriers keep the operand reads of one block from being hoisted over the
// blocks before it: without them the backward kernels spilled up to 190
// registers; the other wavefronts of the SIMD cover the reads.)
template <int MB, int NB>
__device__ __forceinline__ void gemm(const float* __restrict__ sw, int ld, const float (&b)[NB][4],
                                     floatx4 (&z)[MB]) {
  const auto [r, q] = lane_here();
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) {
    floatx4 a[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      a[mb] = *reinterpret_cast<const floatx4*>(sw + (16 * mb + r) * ld + 16 * kb + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) z[mb] = mma(a[mb][e], b[kb][e], z[mb]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// z = W^T g (columns 16 c0 .. of W): NO blocks of 16 output dims.
template <int NO, int MB>
__device__ __forceinline__ void gemm_t(const float* __restrict__ sw, int ld, const float (&g)[MB][4],
                                       floatx4 (&z)[NO]) {
  const auto [r, q] = lane_here();
#pragma unroll
  for (int i = 0; i < NO; ++i) z[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int mo = 0; mo < MB; ++mo) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < NO; ++i)
        z[i] = mma(sw[(16 * mo + 4 * q + e) * ld + 16 * i + r], g[mo][e], z[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Block starting values: a bias vector's rows (or zero).
template <int MB>
__device__ __forceinline__ void init_bias(const float* bias, floatx4 (&z)[MB]) {
  const int q = lane_here().q;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) z[mb] = *reinterpret_cast<const floatx4*>(bias + 16 * mb + 4 * q);
}
template <int MB>
__device__ __forceinline__ void init_zero(floatx4 (&z)[MB]) {
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) z[mb] = floatx4{0.f, 0.f, 0.f, 0.f};
}

__device__ __forceinline__ float sum_q(float v) {  // over the 4 lanes of a point (same r)
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}
__device__ __forceinline__ float sum_r(float v) {  // over the 16 points of a q group
  v += __shfl_xor(v, 1, 64);
  v += __shfl_xor(v, 2, 64);
  v += __shfl_xor(v, 4, 64);
  v += __shfl_xor(v, 8, 64);
  return v;
}

// ----------------------------------------------------------------------------
// Forward: sdf [n]; kGrad: also dsdf/dh0 [n, d] (backprop of 1).
// ----------------------------------------------------------------------------
template <int H, int NH, int KB, bool kGrad>
__global__ void __launch_bounds__(64 * kWaves, 4)
mlp_fwd_kernel(const float* __restrict__ x, const float* __restrict__ enc, int E, int vec4,
               int64_t n_cap, const int32_t* __restrict__ n_dev, const float* __restrict__ mlp,
               float beta, float* __restrict__ sdf_out, float* __restrict__ dh0) {
  using M = Mlp<H, NH, KB>;
  constexpr int MB = M::MB;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  load_weights<H, NH, KB>(smem, mlp, E);
  const float* sW1 = smem + M::oW1;
  const float* vec = smem + M::oVec;
  const float inv_beta = 1.f / beta;
  const int64_t n = dev_count(n_cap, n_dev);
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  const int d = 3 + E;
  __syncthreads();
  const int64_t n_groups = ceil_div(n, 16), waves = (int64_t)gridDim.x * kWaves;
  for (int64_t g = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6); g < n_groups; g += waves) {
    // weights re-read from LDS every group rather than held in registers
    asm volatile("" ::: "memory");
    const int64_t p = g * 16 + r;
    const bool ok = p < n;
    // the lane's quarter index and the encoding's shape, opaque in every step:
    // the boundary tests of the loads and stores derive from them and are then
    // evaluated where used instead of hoisted as dozens of execution masks
    int qs = q, Es = E, v4s = vec4;
    asm volatile("" : "+v"(qs), "+s"(Es), "+s"(v4s));
    float h0[KB][4];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) load_in(x, enc, Es, v4s, n_cap, p, ok, 16 * kb + 4 * qs, h0[kb]);
    floatx4 z[MB];
    init_bias<MB>(vec, z);
    gemm<MB, KB>(smem, M::LD0, h0, z);
    float d1[MB][4];
    if (NH == 2) {
      float h1[MB][4];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Sp s = softplus(z[mb][e], beta, inv_beta);
          h1[mb][e] = s.h;
          d1[mb][e] = s.d;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      init_bias<MB>(vec + H, z);
      gemm<MB, MB>(sW1, M::LD1, h1, z);
    }
    float f = 0.f, gz[MB][4];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const floatx4 wo = *reinterpret_cast<const floatx4*>(vec + 2 * H + 16 * mb + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const Sp s = softplus(z[mb][e], beta, inv_beta);
        f += wo[e] * s.h;
        gz[mb][e] = wo[e] * s.d;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    f = sum_q(f) + vec[3 * H];
    if (q == 0 && ok) sdf_out[p] = f;
    if constexpr (kGrad) {
      if (NH == 2) {
        gemm_t<MB, MB>(sW1, M::LD1, gz, z);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int e = 0; e < 4; ++e) gz[mb][e] = z[mb][e] * d1[mb][e];
      }
      floatx4 gi[KB];
      gemm_t<KB, MB>(smem, M::LD0, gz, gi);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = in_col(16 * kb + 4 * qs + e, Es);
          if (ok && col >= 0) dh0[p * d + col] = gi[kb][e];
        }
    }
  }
}

// ----------------------------------------------------------------------------
// Weight-gradient helpers.  A workgroup steps over 64 points (16 per
// wavefront): block tiles hold rows of 64 points (pitch 68 floats: a
// wavefront's writes and its 16-byte operand reads are conflict-free).
// ----------------------------------------------------------------------------
template <int TP, int NB>
__device__ __forceinline__ void tile_store(float* t, const float (&v)[NB][4]) {
  const auto [r, q] = lane_here();
  const int col = 16 * (threadIdx.x >> 6) + r;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) t[(16 * b + 4 * q + e) * TP + col] = v[b][e];
}

// acc[t] += A[row block ia(t)] * B[row block ib(t)]^T over the step's points,
// one of the two row blocks the same for every t.
template <int TP, int T, bool kAFixed>
__device__ __forceinline__ void tile_mma(const float* tA, const float* tB, int fixed, int first,
                                         int stride, int n_blocks, floatx4 (&acc)[T]) {
  const auto [r, q] = lane_here();
  const float* tF = kAFixed ? tA : tB;
  const float* tV = kAFixed ? tB : tA;
#pragma unroll
  for (int k = 0; k < kWaves; ++k) {
    const floatx4 f = *reinterpret_cast<const floatx4*>(tF + (16 * fixed + r) * TP + 16 * k + 4 * q);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int b = first + stride * t;  // uniform
      if (b >= n_blocks) continue;
      const floatx4 v = *reinterpret_cast<const floatx4*>(tV + (16 * b + r) * TP + 16 * k + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[t] = kAFixed ? mma(f[e], v[e], acc[t]) : mma(v[e], f[e], acc[t]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The workgroup's partial row of the weight gradient (packed layout): weight
// blocks from the wavefronts that own them, vector sums combined over the
// wavefronts in a fixed order through LDS (red: >= kWaves (3H + 1) floats no
// longer in use).  Called by every lane of the workgroup.
template <int H, int NH, int KB>
__device__ __forceinline__ void write_partial(float* __restrict__ out, int E, int wid, float* red,
                                              const floatx4 (&acc1)[Mlp<H, NH, KB>::T1],
                                              const floatx4 (&acc0)[Mlp<H, NH, KB>::T0],
                                              const float (&db0)[H / 16][4],
                                              const float (&db1)[H / 16][4],
                                              const float (&dwo)[H / 16][4], float dbo) {
  using M = Mlp<H, NH, KB>;
  constexpr int MB = M::MB;
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4, d = 3 + E;
#pragma unroll
  for (int t = 0; t < M::T0; ++t) {
    const int md = wid / MB + M::S * t, ob = wid % MB;
    if (md >= KB) continue;
    const int col = in_col(16 * md + r, E);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col >= 0) out[(16 * ob + 4 * q + e) * d + col] = acc0[t][e];
  }
  if (NH == 2) {
#pragma unroll
    for (int t = 0; t < M::T1; ++t) {
      const int ob = wid / MB + M::S * t, ib = wid % MB;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        out[M::gW1(d) + (16 * ob + 4 * q + e) * H + 16 * ib + r] = acc1[t][e];
    }
  }
  float* mine = red + wid * (3 * H + 1);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int u = 16 * mb + 4 * q + e;
      const float s0 = sum_r(db0[mb][e]), s1 = sum_r(db1[mb][e]), so = sum_r(dwo[mb][e]);
      if (r == 0) {
        mine[u] = s0;
        mine[H + u] = s1;
        mine[2 * H + u] = so;
      }
    }
  const float sbo = sum_q(sum_r(dbo));
  if (l == 0) mine[3 * H] = sbo;
  __syncthreads();
  for (int t = threadIdx.x; t < 3 * H + 1; t += blockDim.x) {
    float v = 0.f;
    for (int w = 0; w < kWaves; ++w) v += red[w * (3 * H + 1) + t];
    if (t < H) out[M::gB0(d) + t] = v;
    else if (t < 2 * H) { if (NH == 2) out[M::gB1(d) + t - H] = v; }
    else if (t < 3 * H) out[M::gWo(d) + t - 2 * H] = v;
    else out[M::gBo(d)] = v;
  }
}

// Stores 4 input dims c4..c4+3 of point p: encoding columns to g_enc, position
// columns to g_x (either may be null).
__device__ __forceinline__ void store_in(float* __restrict__ g_enc, float* __restrict__ g_x, int E,
                                         int vec4, int64_t p, bool ok, int c4, floatx4 v) {
  if (!ok) return;
  if (vec4) {
    if (c4 < E) {
      if (g_enc) *reinterpret_cast<float4*>(g_enc + p * E + c4) = float4{v[0], v[1], v[2], v[3]};
    } else if (c4 == E && g_x) {
      g_x[p * 3] = v[0];
      g_x[p * 3 + 1] = v[1];
      g_x[p * 3 + 2] = v[2];
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = c4 + e;
    if (c < E) {
      if (g_enc) g_enc[p * E + c] = v[e];
    } else if (c < E + 3 && g_x) {
      g_x[p * 3 + (c - E)] = v[e];
    }
  }
}

// ----------------------------------------------------------------------------
// Backward (sdf only): given dL/dsdf, one weight-gradient partial row per
// workgroup and dL/denc [n, E] (+ dL/dx [n,3] if requested).
// ----------------------------------------------------------------------------
template <int H, int NH, int KB>
__global__ void __launch_bounds__(64 * kWaves, 2)
mlp_bwd_kernel(const float* __restrict__ x, const float* __restrict__ enc, int E, int vec4,
               int64_t n_cap, const int32_t* __restrict__ n_dev, const float* __restrict__ mlp,
               float beta, const float* __restrict__ g_sdf, float* __restrict__ g_enc,
               float* __restrict__ g_x, float* __restrict__ partials) {
  using M = Mlp<H, NH, KB>;
  constexpr int MB = M::MB, TP = M::kTileP;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  load_weights<H, NH, KB>(smem, mlp, E);
  const float* sW1 = smem + M::oW1;
  const float* vec = smem + M::oVec;
  float* tA = smem + M::oTA;
  float* tB = smem + M::oTB;
  const float inv_beta = 1.f / beta;
  const int64_t n = dev_count(n_cap, n_dev);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  const int fixed = wid % MB, first = wid / MB;
  floatx4 acc1[M::T1], acc0[M::T0];
  init_zero<M::T1>(acc1);
  init_zero<M::T0>(acc0);
  float db0[MB][4], db1[MB][4], dwo[MB][4], dbo = 0.f;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int e = 0; e < 4; ++e) db0[mb][e] = db1[mb][e] = dwo[mb][e] = 0.f;
  __syncthreads();
  const int64_t n_steps = ceil_div(n, (int64_t)16 * kWaves);
  for (int64_t step = blockIdx.x; step < n_steps; step += gridDim.x) {
    const int64_t p = (step * kWaves + wid) * 16 + r;
    const bool ok = p < n;
    int qs = q, Es = E, v4s = vec4;  // opaque: see mlp_fwd_kernel
    asm volatile("" : "+v"(qs), "+s"(Es), "+s"(v4s));
    float h0[KB][4];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) load_in(x, enc, Es, v4s, n_cap, p, ok, 16 * kb + 4 * qs, h0[kb]);
    const float gs = ok ? g_sdf[p] : 0.f;
    if (q == 0) dbo += gs;
    floatx4 z[MB];
    init_bias<MB>(vec, z);
    gemm<MB, KB>(smem, M::LD0, h0, z);
    float h1[MB][4], d1[MB][4], gz[MB][4];
    if (NH == 2) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Sp s = softplus(z[mb][e], beta, inv_beta);
          h1[mb][e] = s.h;
          d1[mb][e] = s.d;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      init_bias<MB>(vec + H, z);
      gemm<MB, MB>(sW1, M::LD1, h1, z);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const floatx4 wo = *reinterpret_cast<const floatx4*>(vec + 2 * H + 16 * mb + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const Sp s = softplus(z[mb][e], beta, inv_beta);
        dwo[mb][e] += gs * s.h;
        gz[mb][e] = gs * wo[e] * s.d;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (NH == 2) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int e = 0; e < 4; ++e) db1[mb][e] += gz[mb][e];
      tile_store<TP, MB>(tA, gz);
      tile_store<TP, MB>(tB, h1);
      __syncthreads();
      tile_mma<TP, M::T1, false>(tA, tB, fixed, first, M::S, MB, acc1);
      gemm_t<MB, MB>(sW1, M::LD1, gz, z);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int e = 0; e < 4; ++e) gz[mb][e] = z[mb][e] * d1[mb][e];
      __syncthreads();  // every wavefront is done reading the tiles
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int e = 0; e < 4; ++e) db0[mb][e] += gz[mb][e];
    tile_store<TP, MB>(tA, gz);
    tile_store<TP, KB>(tB, h0);
    __syncthreads();
    tile_mma<TP, M::T0, true>(tA, tB, fixed, first, M::S, KB, acc0);
    if (g_enc || g_x) {
      floatx4 gi[KB];
      gemm_t<KB, MB>(smem, M::LD0, gz, gi);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        store_in(g_enc, g_x, Es, v4s, p, ok, 16 * kb + 4 * qs, gi[kb]);
    }
    __syncthreads();  // tiles are rewritten by the next step
  }
  write_partial<H, NH, KB>(partials + (int64_t)blockIdx.x * M::n_params(3 + E), E, wid, tA, acc1,
                           acc0, db0, db1, dwo, dbo);
}

// ----------------------------------------------------------------------------
// Backward of J = sum_p a_p sdf(x_p) + v_p . grad_x sdf(x_p) (the analytic
// gradient trained through its value, fields.py:107-119 with create_graph):
// forward-over-reverse.  Tangents along v: hd0 = [encd, v] where encd is the
// directional derivative of enc along v (from the hash-grid kernel).  Outputs
// the weight-gradient partials, gb_h0 = dJ/dh0 and gt_h0 = dJ/dhd0: rows of
// out_ld floats in the packed column order, without the first out_c0 columns.
// The weight gradient gb (x) h + gt (x) hd goes through the two tiles in turn,
// so that two workgroups fit a CU.
// ----------------------------------------------------------------------------
template <int H, int NH, int KB>
__global__ void __launch_bounds__(64 * kWaves, 2)
mlp_bwd_ad_kernel(const float* __restrict__ x, const float* __restrict__ enc,
                  const float* __restrict__ v, const float* __restrict__ encd, int E, int vec4,
                  int64_t n_cap, const int32_t* __restrict__ n_dev, const float* __restrict__ mlp,
                  float beta, const float* __restrict__ a_sdf, float* __restrict__ gb_h0,
                  float* __restrict__ gt_h0, float* __restrict__ partials, int out_ld,
                  int out_c0) {
  using M = Mlp<H, NH, KB>;
  constexpr int MB = M::MB, TP = M::kTileP;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  load_weights<H, NH, KB>(smem, mlp, E);
  const float* sW1 = smem + M::oW1;
  const float* vec = smem + M::oVec;
  float* tA = smem + M::oTA;
  float* tB = smem + M::oTB;
  const float inv_beta = 1.f / beta;
  const int64_t n = dev_count(n_cap, n_dev);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  const int fixed = wid % MB, first = wid / MB;
  floatx4 acc1[M::T1], acc0[M::T0];
  init_zero<M::T1>(acc1);
  init_zero<M::T0>(acc0);
  float db0[MB][4], db1[MB][4], dwo[MB][4], dbo = 0.f;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int e = 0; e < 4; ++e) db0[mb][e] = db1[mb][e] = dwo[mb][e] = 0.f;
  __syncthreads();
  const int64_t n_steps = ceil_div(n, (int64_t)16 * kWaves);
  for (int64_t step = blockIdx.x; step < n_steps; step += gridDim.x) {
    const int64_t p = (step * kWaves + wid) * 16 + r;
    const bool ok = p < n;
    int qs = q, Es = E, v4s = vec4;  // opaque: see mlp_fwd_kernel
    asm volatile("" : "+v"(qs), "+s"(Es), "+s"(v4s));
    const float as = ok ? a_sdf[p] : 0.f;
    if (q == 0) dbo += as;
    floatx4 z[MB], zd[MB];
    {
      float h0[KB][4];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) load_in(x, enc, Es, v4s, n_cap, p, ok, 16 * kb + 4 * qs, h0[kb]);
      init_bias<MB>(vec, z);
      gemm<MB, KB>(smem, M::LD0, h0, z);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) load_in(v, encd, Es, v4s, n_cap, p, ok, 16 * kb + 4 * qs, h0[kb]);
      init_zero<MB>(zd);
      gemm<MB, KB>(smem, M::LD0, h0, zd);
    }
    // derivatives and tangent of layer 0 (NH == 2), cotangents of the value
    // (gb) and of the tangent (gt) of the current layer's pre-activation
    float d1[MB][4], w1[MB][4], gb[MB][4], gt[MB][4];  // w1 = zd0 s''(z0)
    float h1[MB][4], hd1[MB][4];
    if (NH == 2) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Sp s = softplus<true>(z[mb][e], beta, inv_beta);
          h1[mb][e] = s.h;
          d1[mb][e] = s.d;
          w1[mb][e] = zd[mb][e] * (beta * s.d * s.c);
          hd1[mb][e] = s.d * zd[mb][e];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      init_bias<MB>(vec + H, z);
      gemm<MB, MB>(sW1, M::LD1, h1, z);
      init_zero<MB>(zd);
      gemm<MB, MB>(sW1, M::LD1, hd1, zd);
      tile_store<TP, MB>(tB, h1);
    }
    // output: J = a*(wo.hL + bo) + wo.hdL;  gb_zL = a wo s' + wo zdL s'';  gt_zL = wo s'
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const floatx4 wo = *reinterpret_cast<const floatx4*>(vec + 2 * H + 16 * mb + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const Sp s = softplus<true>(z[mb][e], beta, inv_beta);
        dwo[mb][e] += as * s.h + s.d * zd[mb][e];
        gb[mb][e] = as * wo[e] * s.d + wo[e] * zd[mb][e] * (beta * s.d * s.c);
        gt[mb][e] = wo[e] * s.d;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (NH == 2) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int e = 0; e < 4; ++e) db1[mb][e] += gb[mb][e];
      tile_store<TP, MB>(tA, gb);
      __syncthreads();
      tile_mma<TP, M::T1, false>(tA, tB, fixed, first, M::S, MB, acc1);
      __syncthreads();  // every wavefront is done reading the tiles
      tile_store<TP, MB>(tA, gt);
      tile_store<TP, MB>(tB, hd1);
      gemm_t<MB, MB>(sW1, M::LD1, gb, z);
      gemm_t<MB, MB>(sW1, M::LD1, gt, zd);
      __syncthreads();
      tile_mma<TP, M::T1, false>(tA, tB, fixed, first, M::S, MB, acc1);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          gb[mb][e] = z[mb][e] * d1[mb][e] + zd[mb][e] * w1[mb][e];
          gt[mb][e] = zd[mb][e] * d1[mb][e];
        }
      __syncthreads();
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int e = 0; e < 4; ++e) db0[mb][e] += gb[mb][e];
    // layer 0's weights: gb (x) h0, then gt (x) hd0 (the inputs read again)
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      float h0[KB][4];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        load_in(pass ? v : x, pass ? encd : enc, Es, v4s, n_cap, p, ok, 16 * kb + 4 * qs, h0[kb]);
      tile_store<TP, MB>(tA, pass ? gt : gb);
      tile_store<TP, KB>(tB, h0);
      __syncthreads();
      tile_mma<TP, M::T0, true>(tA, tB, fixed, first, M::S, KB, acc0);
      float* out = pass ? gt_h0 : gb_h0;
      if (out) {
        floatx4 gi[KB];
        gemm_t<KB, MB>(smem, M::LD0, pass ? gt : gb, gi);
        if (out_c0 == 3) {
          // the encoding's columns alone
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
            store_in(out, nullptr, Es, v4s, p, ok, 16 * kb + 4 * qs, gi[kb]);
        } else {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int col = in_col(16 * kb + 4 * qs + e, Es);
              if (ok && col >= 0) out[p * out_ld + col] = gi[kb][e];
            }
        }
      }
      __syncthreads();  // tiles are rewritten by the next pass
    }
  }
  write_partial<H, NH, KB>(partials + (int64_t)blockIdx.x * M::n_params(3 + E), E, wid, tA, acc1,
                           acc0, db0, db1, dwo, dbo);
}

// Column sums of the partial rows in a fixed order: a workgroup owns 64
// columns; its 16 row groups each sum every 16th row, then the 16 group sums
// are added in order.  Independent of the launch, so results are reproducible.
constexpr int kRedCols = 64, kRedGroups = 16;

__global__ void __launch_bounds__(kRedCols * kRedGroups)
reduce_rows_kernel(const float* __restrict__ partials, int64_t rows, int cols, float* __restrict__ out,
                   int accumulate) {
  // (in 64 bits: a bias or norm gradient may be a sum that all but cancels)
  __shared__ double part[kRedGroups][kRedCols];
  const int cl = threadIdx.x % kRedCols, g = threadIdx.x / kRedCols;
  const int c = blockIdx.x * kRedCols + cl;
  double s = 0.;
  if (c < cols) {
#pragma unroll 8
    for (int64_t r = g; r < rows; r += kRedGroups) s += partials[r * cols + c];
  }
  part[g][cl] = s;
  __syncthreads();
  if (g == 0 && c < cols) {
    double t = 0.;
#pragma unroll
    for (int k = 0; k < kRedGroups; ++k) t += part[k][cl];
    out[c] = accumulate ? out[c] + (float)t : (float)t;
  }
}

int mlp_reduce_rows(const float* part, int64_t rows, int cols, float* out, int accumulate,
                    hipStream_t s) {
  reduce_rows_kernel<<<(unsigned)ceil_div(cols, kRedCols), kRedCols * kRedGroups, 0, s>>>(
      part, rows, cols, out, accumulate);
  return check_launch("mlp_reduce_rows");
}

// ---------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------
// workgroups: 4 of the forward and 2 of the backward fit a CU (LDS)
constexpr int kFwdBlocksMax = 256 * 4;
constexpr int kBwdBlocksMax = 256 * 2;

struct MlpCfg {
  int H, NH, KB, d;
};

static int mlp_cfg(const char* who, int E, int H, int NH, MlpCfg* c) {
  SN_REQUIRE(H == 32 || H == 64, "%s: d_hidden must be 32 or 64 (got %d)", who, H);
  SN_REQUIRE(NH == 1 || NH == 2, "%s: n_layers must be 1 or 2 (got %d)", who, NH);
  SN_REQUIRE(E >= 0 && 3 + E <= 64, "%s: input width 3+%d must be <= 64", who, E);
  c->H = H;
  c->NH = NH;
  c->d = 3 + E;
  c->KB = c->d <= 32 ? 2 : (c->d <= 48 ? 3 : 4);
  return SN_OK;
}

#define SN_MLP_DISPATCH(c, ...)                                                        \
  do {                                                                                 \
    if (c.H == 32 && c.NH == 1 && c.KB == 2) { constexpr int kH = 32, kNH = 1, kKB = 2; __VA_ARGS__; } \
    else if (c.H == 32 && c.NH == 1 && c.KB == 3) { constexpr int kH = 32, kNH = 1, kKB = 3; __VA_ARGS__; } \
    else if (c.H == 32 && c.NH == 1) { constexpr int kH = 32, kNH = 1, kKB = 4; __VA_ARGS__; } \
    else if (c.H == 32 && c.KB == 2) { constexpr int kH = 32, kNH = 2, kKB = 2; __VA_ARGS__; } \
    else if (c.H == 32 && c.KB == 3) { constexpr int kH = 32, kNH = 2, kKB = 3; __VA_ARGS__; } \
    else if (c.H == 32) { constexpr int kH = 32, kNH = 2, kKB = 4; __VA_ARGS__; }      \
    else if (c.NH == 1 && c.KB == 2) { constexpr int kH = 64, kNH = 1, kKB = 2; __VA_ARGS__; } \
    else if (c.NH == 1 && c.KB == 3) { constexpr int kH = 64, kNH = 1, kKB = 3; __VA_ARGS__; } \
    else if (c.NH == 1) { constexpr int kH = 64, kNH = 1, kKB = 4; __VA_ARGS__; }      \
    else if (c.KB == 2) { constexpr int kH = 64, kNH = 2, kKB = 2; __VA_ARGS__; }      \
    else if (c.KB == 3) { constexpr int kH = 64, kNH = 2, kKB = 3; __VA_ARGS__; }      \
    else { constexpr int kH = 64, kNH = 2, kKB = 4; __VA_ARGS__; }                     \
  } while (0)

// Blocks use more than the default 64 KB of dynamic LDS (gfx950 has 160 KB).
template <typename Kern>
static void allow_smem(Kern k, size_t bytes) {
  // once per kernel (kernels of one signature share this instantiation, so
  // the cache is keyed by the kernel); a refusal surfaces as a launch error
  static const void* done[64];
  static size_t done_bytes[64];
  static int n_done = 0;
  const void* f = reinterpret_cast<const void*>(k);
  for (int i = 0; i < n_done; ++i)
    if (done[i] == f && done_bytes[i] >= bytes) return;
  (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (n_done < 64) {
    done[n_done] = f;
    done_bytes[n_done++] = bytes;
  }
}

static unsigned grid_blocks(int64_t n_cap, int max_blocks) {
  const int64_t b = ceil_div(n_cap > 0 ? n_cap : 1, (int64_t)16 * kWaves);
  return (unsigned)(b < max_blocks ? b : max_blocks);
}

// float4 access to rows of E floats
static int vec4_ok(const float* p, int E) {
  return (E % 4 == 0) && ((uintptr_t)p % 16 == 0) ? 1 : 0;
}

}  // namespace sn

using namespace sn;

extern "C" {

int sn_mlp_n_params(int32_t d_in, int32_t d_hidden, int32_t n_layers) {
  if (d_in <= 0 || d_hidden <= 0 || n_layers < 1 || n_layers > 2) return -1;
  return d_hidden * d_in + d_hidden + (n_layers == 2 ? d_hidden * d_hidden + d_hidden : 0) +
         d_hidden + 1;
}

size_t sn_mlp_bwd_workspace_bytes(int64_t n_cap, int32_t enc_dims, int32_t d_hidden,
                                  int32_t n_layers, int32_t analytic) {
  int np = sn_mlp_n_params(3 + enc_dims, d_hidden, n_layers);
  if (np < 0) return 0;
  (void)analytic;
  return (size_t)grid_blocks(n_cap, kBwdBlocksMax) * np * sizeof(float);
}

}  // extern "C"

template <bool kLevels>
static int mlp_fwd_impl(const float* x, const float* enc, int32_t enc_dims, int64_t n_cap,
                        const int32_t* n_dev, const float* mlp, int32_t d_hidden, int32_t n_layers,
                        float beta, float* sdf, float* dsdf_dh0, void* stream) {
  clear_error();
  MlpCfg c;
  int rc = mlp_cfg("sn_mlp_fwd", enc_dims, d_hidden, n_layers, &c);
  if (rc) return rc;
  SN_REQUIRE(n_cap >= 0, "sn_mlp_fwd: n < 0");
  if (n_cap == 0) return SN_OK;
  SN_REQUIRE(x && mlp && sdf && (enc || enc_dims == 0), "sn_mlp_fwd: null pointer");
  hipStream_t s = as_stream(stream);
  const unsigned grid = grid_blocks(n_cap, kFwdBlocksMax);
  int v4 = vec4_ok(enc, enc_dims);
  if (kLevels) {
    SN_REQUIRE(v4, "sn_mlp_fwd: a levels encoding has E % 4 == 0 and is 16-byte aligned");
    v4 = 2;
  }
  SN_MLP_DISPATCH(c, {
    constexpr size_t sm = sizeof(float) * Mlp<kH, kNH, kKB>::kFwd;
    if (dsdf_dh0)
      mlp_fwd_kernel<kH, kNH, kKB, true><<<grid, 64 * kWaves, sm, s>>>(
          x, enc, enc_dims, v4, n_cap, n_dev, mlp, beta, sdf, dsdf_dh0);
    else
      mlp_fwd_kernel<kH, kNH, kKB, false><<<grid, 64 * kWaves, sm, s>>>(
          x, enc, enc_dims, v4, n_cap, n_dev, mlp, beta, sdf, nullptr);
  });
  return check_launch("sn_mlp_fwd");
}

extern "C" {

int sn_mlp_fwd(const float* x, const float* enc, int32_t enc_dims, int64_t n_cap,
               const int32_t* n_dev, const float* mlp, int32_t d_hidden, int32_t n_layers,
               float beta, float* sdf, float* dsdf_dh0, void* stream) {
  return mlp_fwd_impl<false>(
      x, enc, enc_dims, n_cap, n_dev, mlp, d_hidden, n_layers, beta, sdf, dsdf_dh0, stream);
}

int sn_mlp_fwd_levels(const float* x, const float* enc, int32_t enc_dims, int64_t n_cap,
                      const int32_t* n_dev, const float* mlp, int32_t d_hidden, int32_t n_layers,
                      float beta, float* sdf, float* dsdf_dh0, void* stream) {
  return mlp_fwd_impl<true>(
      x, enc, enc_dims, n_cap, n_dev, mlp, d_hidden, n_layers, beta, sdf, dsdf_dh0, stream);
}

}  // extern "C"

template <bool kLevels>
static int mlp_bwd_impl(const float* x, const float* enc, int32_t enc_dims, int64_t n_cap,
                        const int32_t* n_dev, const float* mlp, int32_t d_hidden, int32_t n_layers,
                        float beta, const float* g_sdf, float* g_enc, float* g_x, float* g_mlp,
                        int32_t accumulate, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  MlpCfg c;
  int rc = mlp_cfg("sn_mlp_bwd", enc_dims, d_hidden, n_layers, &c);
  if (rc) return rc;
  SN_REQUIRE(n_cap >= 0, "sn_mlp_bwd: n < 0");
  SN_REQUIRE(mlp && g_mlp, "sn_mlp_bwd: null pointer");
  const size_t need = sn_mlp_bwd_workspace_bytes(n_cap, enc_dims, d_hidden, n_layers, 0);
  if (workspace_bytes < need) {
    set_error("sn_mlp_bwd: workspace %zu < %zu bytes", workspace_bytes, need);
    return SN_ESPACE;
  }
  hipStream_t s = as_stream(stream);
  const int np = sn_mlp_n_params(c.d, d_hidden, n_layers);
  const unsigned grid = grid_blocks(n_cap, kBwdBlocksMax);
  float* part = reinterpret_cast<float*>(workspace);
  int v4 = vec4_ok(enc, enc_dims) && vec4_ok(g_enc, enc_dims);
  if (kLevels) {
    SN_REQUIRE(v4, "sn_mlp_bwd: a levels encoding has E % 4 == 0 and is 16-byte aligned");
    v4 = 2;
  }
  SN_MLP_DISPATCH(c, {
    constexpr size_t sm = sizeof(float) * Mlp<kH, kNH, kKB>::kBwd;
    allow_smem(mlp_bwd_kernel<kH, kNH, kKB>, sm);
    mlp_bwd_kernel<kH, kNH, kKB><<<grid, 64 * kWaves, sm, s>>>(
        x, enc, enc_dims, v4, n_cap, n_dev, mlp, beta, g_sdf, g_enc, g_x, part);
  });
  if ((rc = mlp_reduce_rows(part, (int64_t)grid, np, g_mlp, accumulate, s))) return rc;
  return check_launch("sn_mlp_bwd");
}

extern "C" {

int sn_mlp_bwd(const float* x, const float* enc, int32_t enc_dims, int64_t n_cap,
               const int32_t* n_dev, const float* mlp, int32_t d_hidden, int32_t n_layers,
               float beta, const float* g_sdf, float* g_enc, float* g_x, float* g_mlp,
               int32_t accumulate, void* workspace, size_t workspace_bytes, void* stream) {
  return mlp_bwd_impl<false>(
      x, enc, enc_dims, n_cap, n_dev, mlp, d_hidden, n_layers, beta, g_sdf, g_enc, g_x, g_mlp,
      accumulate, workspace, workspace_bytes, stream);
}

int sn_mlp_bwd_levels(const float* x, const float* enc, int32_t enc_dims, int64_t n_cap,
                      const int32_t* n_dev, const float* mlp, int32_t d_hidden, int32_t n_layers,
                      float beta, const float* g_sdf, float* g_enc, float* g_x, float* g_mlp,
                      int32_t accumulate, void* workspace, size_t workspace_bytes, void* stream) {
  return mlp_bwd_impl<true>(
      x, enc, enc_dims, n_cap, n_dev, mlp, d_hidden, n_layers, beta, g_sdf, g_enc, g_x, g_mlp,
      accumulate, workspace, workspace_bytes, stream);
}

static int mlp_bwd_ad(const float* x, const float* enc, const float* v, const float* enc_dot,
                      int32_t enc_dims, int64_t n_cap, const int32_t* n_dev, const float* mlp,
                      int32_t d_hidden, int32_t n_layers, float beta, const float* g_sdf,
                      float* g_h0, float* g_h0_dot, float* g_mlp, int32_t accumulate,
                      void* workspace, size_t workspace_bytes, void* stream, int out_ld,
                      int out_c0) {
  MlpCfg c;
  int rc = mlp_cfg("sn_mlp_bwd_ad", enc_dims, d_hidden, n_layers, &c);
  if (rc) return rc;
  SN_REQUIRE(n_cap >= 0, "sn_mlp_bwd_ad: n < 0");
  SN_REQUIRE(mlp && g_mlp && v && (enc_dot || enc_dims == 0), "sn_mlp_bwd_ad: null pointer");
  const size_t need = sn_mlp_bwd_workspace_bytes(n_cap, enc_dims, d_hidden, n_layers, 1);
  if (workspace_bytes < need) {
    set_error("sn_mlp_bwd_ad: workspace %zu < %zu bytes", workspace_bytes, need);
    return SN_ESPACE;
  }
  hipStream_t s = as_stream(stream);
  const int np = sn_mlp_n_params(c.d, d_hidden, n_layers);
  const unsigned grid = grid_blocks(n_cap, kBwdBlocksMax);
  float* part = reinterpret_cast<float*>(workspace);
  const int v4 = vec4_ok(enc, enc_dims) && vec4_ok(enc_dot, enc_dims) &&
                 (out_c0 != 3 || (vec4_ok(g_h0, enc_dims) && vec4_ok(g_h0_dot, enc_dims)));
  SN_MLP_DISPATCH(c, {
    constexpr size_t sm = sizeof(float) * Mlp<kH, kNH, kKB>::kBwd;
    allow_smem(mlp_bwd_ad_kernel<kH, kNH, kKB>, sm);
    mlp_bwd_ad_kernel<kH, kNH, kKB><<<grid, 64 * kWaves, sm, s>>>(
        x, enc, v, enc_dot, enc_dims, v4, n_cap, n_dev, mlp, beta, g_sdf, g_h0, g_h0_dot, part,
        out_ld, out_c0);
  });
  if ((rc = mlp_reduce_rows(part, (int64_t)grid, np, g_mlp, accumulate, s))) return rc;
  return check_launch("sn_mlp_bwd_ad");
}

int sn_mlp_bwd_ad(const float* x, const float* enc, const float* v, const float* enc_dot,
                  int32_t enc_dims, int64_t n_cap, const int32_t* n_dev, const float* mlp,
                  int32_t d_hidden, int32_t n_layers, float beta, const float* g_sdf,
                  float* g_h0, float* g_h0_dot, float* g_mlp, int32_t accumulate,
                  void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  return mlp_bwd_ad(x, enc, v, enc_dot, enc_dims, n_cap, n_dev, mlp, d_hidden, n_layers, beta,
                    g_sdf, g_h0, g_h0_dot, g_mlp, accumulate, workspace, workspace_bytes, stream,
                    3 + enc_dims, 0);
}

int sn_mlp_bwd_ad_enc(const float* x, const float* enc, const float* v, const float* enc_dot,
                      int32_t enc_dims, int64_t n_cap, const int32_t* n_dev, const float* mlp,
                      int32_t d_hidden, int32_t n_layers, float beta, const float* g_sdf,
                      float* g_enc, float* g_enc_dot, float* g_mlp, int32_t accumulate,
                      void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  return mlp_bwd_ad(x, enc, v, enc_dot, enc_dims, n_cap, n_dev, mlp, d_hidden, n_layers, beta,
                    g_sdf, g_enc, g_enc_dot, g_mlp, accumulate, workspace, workspace_bytes,
                    stream, enc_dims, 3);
}

}  // extern "C"
