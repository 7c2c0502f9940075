// Patch-based render weights / transmittance, per-ray visibility and the
// scatter-add used by accumulate_along_rays_patch_based.
//
// The recurrence along a patch's samples is sequential per ray, in the same
// order as the reference loop (csrc/render_weight.cu:108-116), so forward
// results are bit-identical to that loop.  Built with -ffp-contract=off.
//
// That recurrence is a few cycles a sample; what it waits for is memory.  A
// patch's samples are one contiguous block, so a wavefront takes a patch,
// brings kChunk values at a time into LDS with whole lines in flight, runs the
// rays' recurrences there on its first P lanes and writes the block back.
// Patches of more than 64 rays: one lane per (patch, ray), kAhead samples'
// loads issued together.  2048 patches of 9 rays, 64 samples each on average:
// forward 182 us with a lane per ray and a load per step, 74 with kAhead loads,
// 32 from LDS; backward 315, 175, 99 (the longest patch, 884 samples, is all of it).
#include "sn_common.h"

namespace sn {

constexpr int kAhead = 16;
constexpr int kChunk = 1024;

// A chunk of a patch's values, in registers (zero past m; an absent gradient is
// zeros: a branch on it between loads keeps them from being issued together)
// and from there in LDS.
struct Chunk {
  float v[kChunk / 64];
  __device__ __forceinline__ void load(const float* __restrict__ src, int m) {
#pragma unroll
    for (int u = 0; u < kChunk / 64; ++u) {
      const int i = u * 64 + threadIdx.x;
      v[u] = i < m ? src[i] : 0.f;
    }
  }
  __device__ __forceinline__ void put(float* dst) const {
#pragma unroll
    for (int u = 0; u < kChunk / 64; ++u) dst[u * 64 + threadIdx.x] = v[u];
  }
};

// Orders a lone wavefront's LDS accesses (a workgroup barrier would also wait
// for the chunk's stores to memory).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// alphas in sa -> transmittances in sT, lanes 0 .. P - 1 a ray each
__device__ __forceinline__ void trans_chain(const float* sa, float* sT, int rows, int P,
                                            float& T) {
#pragma unroll 8
  for (int j = 0; j < rows; ++j) {
    const float a = sa[j * P + threadIdx.x];
    sT[j * P + threadIdx.x] = T;
    T *= (1.f - a);
  }
}

__global__ void __launch_bounds__(64)
patch_weight_fwd_lds_kernel(const int32_t* __restrict__ packed_info, int32_t P, int64_t n_samples,
                            const float* __restrict__ alphas, float* __restrict__ weights,
                            float* __restrict__ trans) {
  __shared__ float sa[kChunk], sT[kChunk];
  const int32_t base = packed_info[2 * blockIdx.x], steps = packed_info[2 * blockIdx.x + 1];
  if (steps <= 0 || base < 0 || (int64_t)base + steps > n_samples) return;  // uniform
  const int32_t R = kChunk / P;
  const int64_t off0 = (int64_t)base * P;
  float T = 1.f;
  Chunk a;
  a.load(alphas + off0, min(R, steps) * P);
  for (int32_t c0 = 0; c0 < steps; c0 += R) {
    const int32_t rows = min(R, steps - c0), m = rows * P;
    const int64_t off = off0 + (int64_t)c0 * P;
    a.put(sa);
    wave_sync();
    if (c0 + R < steps)  // the next chunk, while this one's recurrence runs
      a.load(alphas + off + (int64_t)R * P, min(R, steps - c0 - R) * P);
    if ((int)threadIdx.x < P) trans_chain(sa, sT, rows, P, T);
    wave_sync();
    if (trans)
      for (int i = threadIdx.x; i < m; i += 64) trans[off + i] = sT[i];
    if (weights)
      for (int i = threadIdx.x; i < m; i += 64) weights[off + i] = sa[i] * sT[i];
    wave_sync();
  }
}

// As patch_weight_bwd_kernel: T goes to grad_alphas first (the last chunk's
// stays in LDS), then the chunks in reverse.
__global__ void __launch_bounds__(64)
patch_weight_bwd_lds_kernel(const int32_t* __restrict__ packed_info, int32_t P, int64_t n_samples,
                            const float* __restrict__ alphas, const float* __restrict__ gw,
                            const float* __restrict__ gT, float* __restrict__ ga) {
  __shared__ float sa[kChunk], sT[kChunk], sw[kChunk], st[kChunk];
  const int32_t base = packed_info[2 * blockIdx.x], steps = packed_info[2 * blockIdx.x + 1];
  if (steps <= 0 || base < 0 || (int64_t)base + steps > n_samples) return;  // uniform
  const int32_t R = kChunk / P, last = (steps - 1) / R * R;
  const int64_t off0 = (int64_t)base * P;
  float T = 1.f;
  Chunk a, t, w, z;
  a.load(alphas + off0, min(R, steps) * P);
  auto gradients = [&](int64_t off, int m) {
    w.load(gw ? gw + off : alphas, gw ? m : 0);
    z.load(gT ? gT + off : alphas, gT ? m : 0);
  };
  for (int32_t c0 = 0; c0 < steps; c0 += R) {
    const int32_t rows = min(R, steps - c0), m = rows * P;
    const int64_t off = off0 + (int64_t)c0 * P;
    a.put(sa);
    wave_sync();
    if (c0 < last)
      a.load(alphas + off + (int64_t)R * P, min(R, steps - c0 - R) * P);
    else
      gradients(off, m);
    if ((int)threadIdx.x < P) trans_chain(sa, sT, rows, P, T);
    wave_sync();
    if (c0 < last)
      for (int i = threadIdx.x; i < m; i += 64) ga[off + i] = sT[i];
    wave_sync();
  }
  __syncthreads();  // the parked T is read back below
  float Q = 0.f;
  for (int32_t c0 = last; c0 >= 0; c0 -= R) {
    const int32_t rows = min(R, steps - c0), m = rows * P;
    const int64_t off = off0 + (int64_t)c0 * P, before = off - (int64_t)R * P;
    w.put(sw);
    z.put(st);
    if (c0 < last) {
      a.put(sa);
      t.put(sT);
    }
    wave_sync();
    if (c0 > 0) {  // the chunk before, while this one's recurrence runs
      a.load(alphas + before, R * P);
      t.load(ga + before, R * P);
      gradients(before, R * P);
    }
    if ((int)threadIdx.x < P) {
      // 8 steps' operands before the first result is stored (in place)
      for (int j0 = rows - 1; j0 >= 0; j0 -= 8) {
        float av[8], wv[8], tv[8], Tv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = max(j0 - u, 0) * P + threadIdx.x;
          av[u] = sa[i];
          Tv[u] = sT[i];
          wv[u] = sw[i];
          tv[u] = st[i];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (j0 - u >= 0) {
            sT[(j0 - u) * P + threadIdx.x] = Tv[u] * (wv[u] - Q);
            Q = (wv[u] * av[u] + tv[u]) + (1.f - av[u]) * Q;
          }
        }
      }
    }
    wave_sync();
    for (int i = threadIdx.x; i < m; i += 64) ga[off + i] = sT[i];
    wave_sync();
  }
}

__global__ void __launch_bounds__(256)
patch_weight_fwd_kernel(const int32_t* __restrict__ packed_info, int32_t n_patches, int32_t P,
                        int64_t n_samples, const float* __restrict__ alphas, float* __restrict__ weights,
                        float* __restrict__ trans) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (g >= (int64_t)n_patches * P) return;
  const int32_t p = (int32_t)(g / P);
  const int32_t k = (int32_t)(g - (int64_t)p * P);
  const int32_t base = packed_info[2 * p];
  const int32_t steps = packed_info[2 * p + 1];
  if (steps <= 0 || base < 0 || (int64_t)base + steps > n_samples) return;
  const int64_t off = (int64_t)base * P + k;
  float T = 1.f;
  for (int32_t j0 = 0; j0 < steps; j0 += kAhead) {
    float a[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      a[u] = alphas[off + (int64_t)min(j0 + u, steps - 1) * P];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (j0 + u < steps) {
        const int64_t idx = off + (int64_t)(j0 + u) * P;
        if (trans) trans[idx] = T;
        if (weights) weights[idx] = a[u] * T;
        T *= (1.f - a[u]);
      }
    }
  }
}

// g_alpha[j] = T[j] * (gw[j] - Q[j]),
// Q[j] = (gw[j+1] a[j+1] + gT[j+1]) + (1 - a[j+1]) Q[j+1], Q[last] = 0.
// T[j] is first written into grad_alphas (pass 1), then scaled in place.
__global__ void __launch_bounds__(256)
patch_weight_bwd_kernel(const int32_t* __restrict__ packed_info, int32_t n_patches, int32_t P,
                        int64_t n_samples, const float* __restrict__ alphas, const float* __restrict__ gw,
                        const float* __restrict__ gT, float* __restrict__ ga) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (g >= (int64_t)n_patches * P) return;
  const int32_t p = (int32_t)(g / P);
  const int32_t k = (int32_t)(g - (int64_t)p * P);
  const int32_t base = packed_info[2 * p];
  const int32_t steps = packed_info[2 * p + 1];
  if (steps <= 0 || base < 0 || (int64_t)base + steps > n_samples) return;
  const int64_t off = (int64_t)base * P + k;
  float T = 1.f;
  for (int32_t j0 = 0; j0 < steps; j0 += kAhead) {
    float a[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      a[u] = alphas[off + (int64_t)min(j0 + u, steps - 1) * P];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (j0 + u < steps) {
        ga[off + (int64_t)(j0 + u) * P] = T;
        T *= (1.f - a[u]);
      }
    }
  }
  float Q = 0.f;
  for (int32_t j0 = steps - 1; j0 >= 0; j0 -= kAhead) {
    float a[kAhead], w[kAhead], t[kAhead], tj[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int64_t idx = off + (int64_t)max(j0 - u, 0) * P;
      a[u] = alphas[idx];
      w[u] = gw ? gw[idx] : 0.f;
      t[u] = gT ? gT[idx] : 0.f;
      tj[u] = ga[idx];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (j0 - u >= 0) {
        ga[off + (int64_t)(j0 - u) * P] = tj[u] * (w[u] - Q);
        Q = (w[u] * a[u] + t[u]) + (1.f - a[u]) * Q;
      }
    }
  }
}

// Per-ray exclusive product (csrc/render_transmittance.cu:85-112) and the
// visibility test of vol_rendering.py:744-747.
__global__ void __launch_bounds__(256)
visibility_kernel(const int32_t* __restrict__ packed_info, int32_t n_rays, int64_t n_samples,
                  const float* __restrict__ alphas, float eps, float alpha_thre,
                  uint8_t* __restrict__ keep) {
  const int32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_rays) return;
  const int32_t base = packed_info[2 * r];
  const int32_t steps = packed_info[2 * r + 1];
  if (steps <= 0 || base < 0 || (int64_t)base + steps > n_samples) return;
  float T = 1.f;
  for (int32_t j0 = 0; j0 < steps; j0 += kAhead) {
    float a[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) a[u] = alphas[base + min(j0 + u, steps - 1)];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (j0 + u < steps) {
        bool v = T >= eps;
        if (alpha_thre > 0.f) v = v && (a[u] >= alpha_thre);
        keep[base + j0 + u] = v ? 1 : 0;
        T *= (1.f - a[u]);
      }
    }
  }
}

// A thread takes one element of `run` consecutive rows and adds the rows of a
// run of equal indices before it issues their atomic: samples come sorted by
// ray, and fp32 atomics, ~2e10/s on the device, were all of its time.
// 131 k rows of 27 floats in runs of 64: 89 -> 9 us.
__global__ void __launch_bounds__(256)
scatter_add_rows_kernel(const int64_t* __restrict__ idx, int64_t n, int32_t row, int32_t run,
                        const float* __restrict__ src, float* __restrict__ out,
                        int32_t n_out_rows) {
  constexpr int kU = 4;
  const int64_t total = ceil_div(n, (int64_t)run) * row;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < total;
       g += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = g / row;
    const int32_t e = (int32_t)(g - c * row);
    const int64_t s0 = c * run, s1 = min(s0 + run, n);
    int64_t cur = -1;
    float sum = 0.f;
    for (int64_t s = s0; s < s1; s += kU) {
      int64_t r[kU];
      float v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t i = min(s + u, s1 - 1);
        r[u] = idx[i];
        v[u] = src[i * row + e];
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        if (s + u < s1 && r[u] >= 0 && r[u] < n_out_rows) {
          if (r[u] != cur) {
            if (cur >= 0) atomicAdd(&out[cur * row + e], sum);
            cur = r[u];
            sum = v[u];
          } else {
            sum += v[u];
          }
        }
      }
    }
    if (cur >= 0) atomicAdd(&out[cur * row + e], sum);
  }
}

}  // namespace sn

using namespace sn;

extern "C" {

int sn_patch_weight_fwd(const int32_t* packed_info, int32_t n_patches, int32_t patch_size,
                        int64_t n_samples, const float* alphas, float* weights,
                        float* transmittance, void* stream) {
  clear_error();
  SN_REQUIRE(n_patches >= 0 && patch_size > 0 && n_samples >= 0,
             "sn_patch_weight_fwd: bad sizes (%d, %d)", n_patches, patch_size);
  if (n_patches == 0 || n_samples == 0) return SN_OK;
  SN_REQUIRE(packed_info && alphas, "sn_patch_weight_fwd: null input");
  SN_REQUIRE(weights || transmittance, "sn_patch_weight_fwd: no output");
  if (patch_size <= 64) {
    patch_weight_fwd_lds_kernel<<<n_patches, 64, 0, as_stream(stream)>>>(
        packed_info, patch_size, n_samples, alphas, weights, transmittance);
    return check_launch("sn_patch_weight_fwd");
  }
  int64_t n = (int64_t)n_patches * patch_size;
  patch_weight_fwd_kernel<<<(unsigned)ceil_div(n, 256), 256, 0, as_stream(stream)>>>(
      packed_info, n_patches, patch_size, n_samples, alphas, weights, transmittance);
  return check_launch("sn_patch_weight_fwd");
}

int sn_patch_transmittance_fwd(const int32_t* packed_info, int32_t n_patches,
                               int32_t patch_size, int64_t n_samples, const float* alphas,
                               float* transmittance, void* stream) {
  return sn_patch_weight_fwd(packed_info, n_patches, patch_size, n_samples, alphas, nullptr,
                             transmittance, stream);
}

int sn_patch_weight_bwd(const int32_t* packed_info, int32_t n_patches, int32_t patch_size,
                        int64_t n_samples, const float* alphas, const float* grad_weights,
                        const float* grad_transmittance, float* grad_alphas, void* stream) {
  clear_error();
  SN_REQUIRE(n_patches >= 0 && patch_size > 0 && n_samples >= 0,
             "sn_patch_weight_bwd: bad sizes (%d, %d)", n_patches, patch_size);
  if (n_patches == 0 || n_samples == 0) return SN_OK;
  SN_REQUIRE(packed_info && alphas && grad_alphas, "sn_patch_weight_bwd: null pointer");
  if (patch_size <= 64) {
    patch_weight_bwd_lds_kernel<<<n_patches, 64, 0, as_stream(stream)>>>(
        packed_info, patch_size, n_samples, alphas, grad_weights, grad_transmittance,
        grad_alphas);
    return check_launch("sn_patch_weight_bwd");
  }
  int64_t n = (int64_t)n_patches * patch_size;
  patch_weight_bwd_kernel<<<(unsigned)ceil_div(n, 256), 256, 0, as_stream(stream)>>>(
      packed_info, n_patches, patch_size, n_samples, alphas, grad_weights, grad_transmittance,
      grad_alphas);
  return check_launch("sn_patch_weight_bwd");
}

int sn_visibility(const int32_t* packed_info, int32_t n_rays, int64_t n_samples,
                  const float* alphas, float early_stop_eps, float alpha_thre, uint8_t* keep,
                  void* stream) {
  clear_error();
  SN_REQUIRE(n_rays >= 0 && n_samples >= 0, "sn_visibility: negative size");
  if (n_rays == 0 || n_samples == 0) return SN_OK;
  SN_REQUIRE(packed_info && alphas && keep, "sn_visibility: null pointer");
  visibility_kernel<<<(unsigned)ceil_div(n_rays, 256), 256, 0, as_stream(stream)>>>(
      packed_info, n_rays, n_samples, alphas, early_stop_eps, alpha_thre, keep);
  return check_launch("sn_visibility");
}

int sn_scatter_add_rows(const int64_t* ray_indices, int64_t n, int32_t row_elems,
                        const float* src, float* out, int32_t n_out_rows, void* stream) {
  clear_error();
  SN_REQUIRE(n >= 0 && row_elems > 0 && n_out_rows >= 0, "sn_scatter_add_rows: bad sizes");
  if (n == 0) return SN_OK;
  SN_REQUIRE(ray_indices && src && out, "sn_scatter_add_rows: null pointer");
  // rows per thread: as many as leave 2^16 threads (4 wavefronts per CU), 16 at most
  const int64_t per = (n * row_elems) >> 16;
  const int32_t run = (int32_t)(per < 1 ? 1 : (per > 16 ? 16 : per));
  scatter_add_rows_kernel<<<grid_for(ceil_div(n, (int64_t)run) * row_elems, 256), 256, 0,
                            as_stream(stream)>>>(ray_indices, n, row_elems, run, src, out,
                                                 n_out_rows);
  return check_launch("sn_scatter_add_rows");
}

}  // extern "C"
