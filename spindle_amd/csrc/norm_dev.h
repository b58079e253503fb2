// RMSNorm of fp32 rows as device code: the norm tail that a producer's last workgroup runs over the
// pass's rows (norm_rows) and the same norm of one row in a consumer's prologue (NormRow).
#pragma once
#include "attn.h"
#include "dev.h"
#include "fused.h"

namespace spx {

// ------------------------------------------------------------------ norm tail
// Rows [b0, b1) of a NormTail by all NW wavefronts of the workgroup. Wave w takes the
// 256-value blocks w, w+NW, ...; lane j holds values 4j..4j+3 of a block.
template <int NW>
__device__ __forceinline__ void norm_rows(const NormTail &t, int b0, int b1) {
  __shared__ float bsum[NORM_NT];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int dim = t.dim, n4 = dim >> 2, nblk = (n4 + 63) >> 6, nbq = dim >> 8;
  const rsrc_t ra = rsrc_of(t.add ? t.add : t.x);
  const float4 *x4 = reinterpret_cast<const float4 *>(t.x);
  const float4 *w4 = reinterpret_cast<const float4 *>(t.nw);
  float4 wn[NORM_NT / NW];  // the norm weights, loaded once with the first row's inputs
#pragma unroll
  for (int k = 0; k < NORM_NT / NW; k++) {
    const int f = (wave + NW * k) * 64 + lane;
    wn[k] = f < n4 ? w4[f] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  for (int b = b0; b < b1; b++) {
    float4 r[NORM_NT / NW];
#pragma unroll
    for (int k = 0; k < NORM_NT / NW; k++) {
      const int tb = wave + NW * k, f = tb * 64 + lane;
      r[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (tb < nblk) {
        if (f < n4) {
          float4 v = x4[(int64_t)b * n4 + f];
          if (t.add) {
            const f4v a = ld_coh4(ra, (b * n4 + f) * 16);
            v.x = v.x + t.rscale * a.x; v.y = v.y + t.rscale * a.y; v.z = v.z + t.rscale * a.z; v.w = v.w + t.rscale * a.w;
          }
          r[k] = v;
        }
        float p = r[k].x * r[k].x;
        p = fmaf(r[k].y, r[k].y, p);
        p = fmaf(r[k].z, r[k].z, p);
        p = fmaf(r[k].w, r[k].w, p);
        p = wave_sum(p);
        if (lane == 0) bsum[tb] = p;
      }
    }
    __syncthreads();
    float S = 0.0f;
    for (int k = 0; k < nblk; k++) S = S + bsum[k];
    const float inv = inv_rms(S, (float)dim, t.eps);
#pragma unroll
    for (int k = 0; k < NORM_NT / NW; k++) {
      const int tb = wave + NW * k, f = tb * 64 + lane;
      if (tb < nblk) {
        float4 v = r[k];
        if (f < n4) {
          if (t.x_out) reinterpret_cast<float4 *>(t.x_out)[(int64_t)b * n4 + f] = v;
          const float4 w = wn[k];
          v.x = v.x * inv * w.x; v.y = v.y * inv * w.y; v.z = v.z * inv * w.z; v.w = v.w * inv * w.w;
          if (t.xn_out) reinterpret_cast<float4 *>(t.xn_out)[(int64_t)b * n4 + f] = v;
        }
        if (t.q_out.q) {
          const float am = q8k_amax(v);
          const int64_t vb = (int64_t)b * nbq + tb;
          q8k_block_store(v, am, t.q_out.q + vb * 64, t.q_out.d + vb, reinterpret_cast<int *>(t.q_out.bs + vb * 8));
        }
      }
    }
    __syncthreads();
  }
}

// The same RMSNorm of one row (t.x, no residual add) computed by a consumer's workgroup for
// itself: the row and its weights loaded (load), then norm_rows's per-block fma chains and
// wavefront trees, the blocks in order, x * inv * w (finish) into LDS lx (and memory, xn_out).
// The bits are norm_rows's: a producer's residual epilogue plus this prologue replace its tail.
template <int NW>
struct NormRow {
  float4 r[NORM_NT / NW], w[NORM_NT / NW];
  __device__ __forceinline__ void load(const NormTail &t) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n4 = t.dim >> 2, nblk = (n4 + 63) >> 6;
#pragma unroll
    for (int k = 0; k < NORM_NT / NW; k++) {
      const int tb = wave + NW * k, f = tb * 64 + lane;
      r[k] = w[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (tb < nblk && f < n4) {
        r[k] = reinterpret_cast<const float4 *>(t.x)[f];
        w[k] = reinterpret_cast<const float4 *>(t.nw)[f];
      }
    }
  }
  __device__ __forceinline__ void finish(const NormTail &t, float *lx, float *xn_out) {
    __shared__ float bsum[NORM_NT];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n4 = t.dim >> 2, nblk = (n4 + 63) >> 6;
#pragma unroll
    for (int k = 0; k < NORM_NT / NW; k++) {
      const int tb = wave + NW * k;
      if (tb < nblk) {
        float p = r[k].x * r[k].x;
        p = fmaf(r[k].y, r[k].y, p);
        p = fmaf(r[k].z, r[k].z, p);
        p = fmaf(r[k].w, r[k].w, p);
        p = wave_sum(p);
        if (lane == 0) bsum[tb] = p;
      }
    }
    __syncthreads();
    float S = 0.0f;
    for (int k = 0; k < nblk; k++) S = S + bsum[k];
    const float inv = inv_rms(S, (float)t.dim, t.eps);
#pragma unroll
    for (int k = 0; k < NORM_NT / NW; k++) {
      const int tb = wave + NW * k, f = tb * 64 + lane;
      if (tb < nblk && f < n4) {
        float4 v = r[k];
        const float4 ww = w[k];
        v.x = v.x * inv * ww.x; v.y = v.y * inv * ww.y; v.z = v.z * inv * ww.z; v.w = v.w * inv * ww.w;
        reinterpret_cast<float4 *>(lx)[f] = v;
        if (xn_out) reinterpret_cast<float4 *>(xn_out)[f] = v;
      }
    }
    __syncthreads();
  }
};

// A launch output a norm tail will read is stored coherently.
__device__ __forceinline__ void out_store(float *p, float v, bool coh) {
  if (coh) st_dev(p, v);
  else *p = v;
}

}  // namespace spx
