// Multiresolution hash-grid encoding, 3-D input, linear interpolation.
//
// Semantics follow tiny-cuda-nn's GridEncoding (commit 2ec562e8, the version
// pinned by the reference's create_env.sh:11; its source is not vendored in
// the reference) as restated from the Instant-NGP method:
//   scale_l = base * per_level_scale^l - 1      (computed once on the host, fp64 -> fp32)
//   res_l   = ceil(scale_l) + 1
//   size_l  = min(next_multiple(res_l^3, 8), 2^log2_hashmap_size)
//   pos     = fmaf(scale_l, x, 0.5); cell = floor(pos); frac = pos - cell
//   corner index: dense (x + y*res + z*res^2) when res^3 <= size_l, else
//   x ^ y*2654435761 ^ z*805459861 (uint32 wrap), modulo size_l.
// Cells of negative inputs wrap through uint32, which is what the reference
// gets when it feeds [-1, 1] positions (renderer.py:44) to tcnn.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sn {

constexpr int kMaxLevels = 32;

struct HashGridDesc {
  int32_t n_levels;
  int32_t n_active;  // levels >= n_active are masked (output 0, no gradient)
  // optional device copy of the active level count (read by the kernels,
  // bounded by n_active): lets a captured launch follow a changing count
  const int32_t* n_active_dev;
  uint32_t offset[kMaxLevels + 1];  // table entry offsets (not floats)
  uint32_t hsize[kMaxLevels];
  uint32_t res[kMaxLevels];
  float scale[kMaxLevels];
  uint32_t dense_mask;
};

// Host: fills the descriptor; returns total entries or -1 on bad arguments.
int64_t make_hashgrid_desc(int32_t n_levels, int32_t log2_T, int32_t base_res,
                           float per_level_scale, int32_t n_active, HashGridDesc* d);

#ifdef __HIPCC__
// Table rows of the 8 corners (order c = bx | by<<1 | bz<<2) of the cell with
// integer coordinates g.  One uniform branch per level; the hash's products
// are formed once per axis, and a dense level's rows from the first corner's:
// its row number is reduced modulo the level size once (only where some row
// number reaches it: cells of negative coordinates wrap through uint32), and a
// corner `off` rows further (off < size) is that remainder + off, less the
// size at most once -- or, where the uint32 sum wraps, the small wrapped
// number itself.  (A modulo per corner with its branches had made the corner
// indices a third of the gather and record kernels' instructions.)
__device__ __forceinline__ void hg_rows(const uint32_t g[3], uint32_t res, uint32_t hs, bool dense,
                                        uint32_t idx[8]) {
  if (dense) {  // uniform
    const uint32_t rr = res * res;
    const uint32_t base = g[0] + g[1] * res + g[2] * rr;
    const uint32_t far = 1u + res + rr;  // the last corner's offset
    if (base + far < base || base + far >= hs) {
      const uint32_t m = base % hs;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const uint32_t off = (c & 1) + ((c >> 1) & 1) * res + ((c >> 2) & 1) * rr;
        const uint32_t id = base + off, t = m + off;
        idx[c] = id < base ? id : (t < hs ? t : t - hs);
      }
      // (levels of fewer rows than a corner's offset: the plain form)
      if (far >= hs) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          idx[c] = (base + (c & 1) + ((c >> 1) & 1) * res + ((c >> 2) & 1) * rr) % hs;
      }
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        idx[c] = base + (c & 1) + ((c >> 1) & 1) * res + ((c >> 2) & 1) * rr;
    }
  } else {
    const uint32_t y0 = g[1] * 2654435761u, z0 = g[2] * 805459861u;
    const uint32_t y1 = y0 + 2654435761u, z1 = z0 + 805459861u, mask = hs - 1u;
    const uint32_t x0 = g[0], x1 = g[0] + 1u;
#pragma unroll
    for (int c = 0; c < 8; ++c)
      idx[c] = ((c & 1 ? x1 : x0) ^ ((c & 2 ? y1 : y0) ^ (c & 4 ? z1 : z0))) & mask;
  }
}

// Corner indices/weights of one level.  frac in [0,1); w[c] in corner order
// c = bx | by<<1 | bz<<2, computed as ((w_x) * w_y) * w_z like the reference loop;
// g = the cell's integer coordinates (corner 0).
__device__ __forceinline__ void hg_level(const float x[3], const HashGridDesc& d, int l,
                                         uint32_t idx[8], float w[8], float frac[3],
                                         uint32_t g[3]) {
  const float sc = d.scale[l];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float p = fmaf(sc, x[k], 0.5f);
    float fl = floorf(p);
    g[k] = (uint32_t)(int32_t)fl;
    frac[k] = p - fl;
  }
  hg_rows(g, d.res[l], d.hsize[l], (d.dense_mask >> l) & 1u, idx);
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float wt = (c & 1) ? frac[0] : 1.f - frac[0];
    wt *= ((c >> 1) & 1) ? frac[1] : 1.f - frac[1];
    wt *= ((c >> 2) & 1) ? frac[2] : 1.f - frac[2];
    w[c] = wt;
  }
}

__device__ __forceinline__ void hg_level(const float x[3], const HashGridDesc& d, int l,
                                         uint32_t idx[8], float w[8], float frac[3]) {
  uint32_t g[3];
  hg_level(x, d, l, idx, w, frac, g);
}

// Active levels seen by a kernel.
__device__ __forceinline__ int active_levels(const HashGridDesc& d) {
  if (!d.n_active_dev) return d.n_active;
  const int v = *d.n_active_dev;
  return v < 0 ? 0 : (v < d.n_active ? v : d.n_active);
}

// d w[c] / d frac[k]
__device__ __forceinline__ void hg_dweights(const float frac[3], float dw[8][3]) {
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float a0 = (c & 1) ? frac[0] : 1.f - frac[0];
    const float a1 = ((c >> 1) & 1) ? frac[1] : 1.f - frac[1];
    const float a2 = ((c >> 2) & 1) ? frac[2] : 1.f - frac[2];
    const float s0 = (c & 1) ? 1.f : -1.f;
    const float s1 = ((c >> 1) & 1) ? 1.f : -1.f;
    const float s2 = ((c >> 2) & 1) ? 1.f : -1.f;
    dw[c][0] = s0 * a1 * a2;
    dw[c][1] = a0 * s1 * a2;
    dw[c][2] = a0 * a1 * s2;
  }
}
#endif

}  // namespace sn
