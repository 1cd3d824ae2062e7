// prt_chain.h — one step of a Markov chain (Kelemen's Metropolis sampler,
// render.h:360-780, and energy redistribution, render.h:955-1008): the
// proposal's primary samples, its camera ray, and acceptance with the splats.
// The step kernels of prt_mlt.hip run it for all chains at a time, the path
// kernel for each chain by itself.
#pragma once
#include <hip/hip_runtime.h>

#include "prt_math.h"
#include "prt_mlt.h"
#include "prt_shade.h"

__device__ __forceinline__ uint32_t word_of(double x) {
  // x in [0, 1]; 1 wraps to 0 (the primary sample space is a torus)
  return x >= 1.0 ? 0u : (uint32_t)(x * 4294967296.0);
}

// Mutate0 (mlt.h:42-54), LuxRender's small step: an exponentially
// distributed offset between s1 / (s1/s2 + 1) and s2, up or down with equal
// probability, wrapped into [0, 1).  fabsf keeps the reference's float
// absolute value.
__device__ __forceinline__ uint32_t mutate0(uint32_t w, double r) {
  const double x = u01(w);
  const double s1 = 1.0 / 512.0, s2 = 1.0 / 16.0;
  const double dx = s1 / (s1 / s2 + (double)fabsf((float)(2.0 * r - 1.0))) - s1 / (s1 / s2 + 1.0);
  if (r < 0.5) {
    const double x1 = x + dx;
    return word_of((x1 < 1.0) ? x1 : x1 - 1.0);
  }
  const double x1 = x - dx;
  return word_of((x1 < 0.0) ? x1 + 1.0 : x1);
}

__device__ __forceinline__ bool large_step(const MltChains& C, uint32_t chain, uint32_t iter, double p_large) {
  uint32_t b[4];
  philox(chain, iter, MLT_TAG_LARGE, 0u, C.k0, C.k1, b);
  return u01(b[0]) < p_large;
}

// Words 4 blk .. 4 blk + 3 of a chain's proposal; v: its current path's.
__device__ __forceinline__ uint4 mlt_propose(const MltChains& C, uint32_t chain, uint32_t iter, uint32_t blk,
                                             double p_large, uint4 v) {
  uint32_t r[4];
  if (large_step(C, chain, iter, p_large)) {
    // large step: fresh primary samples (mlt.h:116-121)
    philox(chain, iter, MLT_TAG_FRESH, blk, C.k0, C.k1, r);
    return make_uint4(r[0], r[1], r[2], r[3]);
  }
  // small step: Mutate0 of every word (mlt.h:123-135; mutating the words a
  // path does not use changes nothing it evaluates, and the lazy catch-up
  // there applies the same mutations when a word is next used)
  philox(chain, iter, MLT_TAG_MUTATE, blk, C.k0, C.k1, r);
  return make_uint4(mutate0(v.x, u01(r[0])), mutate0(v.y, u01(r[1])), mutate0(v.z, u01(r[2])),
                    mutate0(v.w, u01(r[3])));
}

// Energy redistribution's proposal: every word moved by d (2u - 1), wrapped
// (erpt.h:29-34).  chain: within the sub-batch.
__device__ __forceinline__ uint4 erpt_propose(const ErptChains& C, uint32_t chain, uint32_t step, uint32_t blk,
                                              double d, uint4 v) {
  uint32_t r[4];
  philox(C.base + chain, step, ERPT_TAG_PERTURB, blk, C.k0, C.k1, r);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t o[4];
  for (int k = 0; k < 4; ++k) {
    double x = u01(w[k]) + d * (2.0 * u01(r[k]) - 1.0);
    if (x > 1.0) x -= 1.0;
    if (x < 0.0) x += 1.0;
    o[k] = word_of(x);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// generate_new_path's camera part (render.h:262-300) with the tent filter the
// MLT mode switches on (scene_env.h:1954): pixel (u0 W, u1 H), sub-pixel
// (u2 < 1/2, u3 < 1/2) of a 2x2 grid, tent offsets from u4, u5.  u: the
// proposal's words; returns its image element (render.h:585-586).
__device__ __forceinline__ uint32_t mlt_camera_ray(const Params& P, const uint32_t* u, d3& o, d3& d) {
  const int x = min((int)(u01(u[0]) * (double)P.W), P.W - 1);
  const int y = min((int)(u01(u[1]) * (double)P.H), P.H - 1);
  const int sx = u01(u[2]) < 0.5 ? 0 : 1;
  const int sy = u01(u[3]) < 0.5 ? 0 : 1;
  const double rr1 = 2.0 * u01(u[4]), rr2 = 2.0 * u01(u[5]);
  const double dx = rr1 < 1.0 ? sqrt(rr1) - 1.0 : 1.0 - sqrt(2.0 - rr1);
  const double dy = rr2 < 1.0 ? sqrt(rr2) - 1.0 : 1.0 - sqrt(2.0 - rr2);
  const double r1 = (sx + 0.5 + dx) * 0.5;
  const double r2 = (sy + 0.5 + dy) * 0.5;
  const d3 sp = ld3(P.center) + ld3(P.screen_x) * ((r1 + x) * P.iw - 0.5) + ld3(P.screen_y) * ((r2 + y) * P.ih - 0.5);
  o = ld3(P.cam_pos);
  d = normalize(sp - o);
  return (uint32_t)((P.H - y - 1) * P.W + x);
}

// mlt.h:171-174 with the Vector3d dot pairing
__device__ __forceinline__ double lum3(const double f[3]) { return (0.2126 * f[0] + 0.0722 * f[2]) + 0.7152 * f[1]; }

__device__ __forceinline__ void splat(uint64_t* img, uint32_t pix, double w, const double f[3]) {
  for (int k = 0; k < 3; ++k) {
    const double v = w * f[k];
    if (v > 0.0) atomicAdd((unsigned long long*)&img[3 * (size_t)pix + k], (unsigned long long)(v * MLT_FIX_ONE + 0.5));
  }
}

// render.h:574-630: a = min(1, L_new / L_old) (1 when L_old is ~0); the
// proposal gets (a + large) / (L_new / b + p_large) / M, the current path
// (1 - a) / (L_old / b + p_large) / M, each times the path weight 4*W*H and
// its radiance; then accept with probability a.  fn, p_new: the proposal's
// radiance and image element.  Returns whether it was accepted, which moves
// the chain's radiance and image element, not its words.
__device__ __forceinline__ bool mlt_accept(const MltChains& C, uint32_t c, uint32_t iter, double p_large, double b,
                                           double weight, double inv_m, const double fn[3], uint32_t p_new) {
  const double fo[3] = {C.f_old[3 * (size_t)c], C.f_old[3 * (size_t)c + 1], C.f_old[3 * (size_t)c + 2]};
  const double l_new = lum3(fn), l_old = lum3(fo);
  const double a = l_old > 1.0e-16 ? fmin(1.0, l_new / l_old) : 1.0;
  const double large = large_step(C, c, iter, p_large) ? 1.0 : 0.0;
  const double w_new = (a + large) / (l_new / b + p_large) * inv_m;
  const double w_old = (1.0 - a) / (l_old / b + p_large) * inv_m;
  splat(C.img, C.pix_old[c], w_old * weight, fo);
  splat(C.img, p_new, w_new * weight, fn);
  uint32_t r[4];
  philox(c, iter, MLT_TAG_ACCEPT, 0u, C.k0, C.k1, r);
  if (!(u01(r[0]) < a)) return false;
  for (int k = 0; k < 3; ++k) C.f_old[3 * (size_t)c + k] = fn[k];
  C.pix_old[c] = p_new;
  return true;
}

// Acceptance min(1, L_z / L_y) and the deposit of the current path, skipped
// once 20 deposits in a row fell on one pixel (render.h:975-1007).
__device__ __forceinline__ bool erpt_accept(const ErptChains& C, uint32_t j, uint32_t step, const double fz[3],
                                            uint32_t p_new) {
  double fy[3] = {C.f_y[3 * (size_t)j], C.f_y[3 * (size_t)j + 1], C.f_y[3 * (size_t)j + 2]};
  const double lz = lum3(fz), ly = lum3(fy);
  const double q = fmin(1.0, ly > 1.0e-16 ? lz / ly : 0.0);  // render.h:978-980
  uint32_t r[4];
  philox(C.base + j, step, ERPT_TAG_ACCEPT, 0u, C.k0, C.k1, r);
  uint32_t py = C.pix_y[j];
  const bool acc = q > u01(r[0]);
  if (acc) {
    for (int k = 0; k < 3; ++k) {
      fy[k] = fz[k];
      C.f_y[3 * (size_t)j + k] = fz[k];
    }
    py = p_new;
    C.pix_y[j] = py;
  }
  uint32_t run = C.run[j];
  if (C.pix_now[j] == py) {
    ++run;
  } else {
    C.pix_now[j] = py;
    run = 0;
  }
  C.run[j] = run;
  const double l = lum3(fy);
  if (run < ERPT_MAX_STACK && l > 0.0) splat(C.img, py, C.dep / l, fy);
  return acc;
}

// Random keys of path batches: batch idx of a phase whose hash is h takes
// splitmix64(h + idx).
__device__ __forceinline__ RngKey chain_key(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  x ^= x >> 31;
  return RngKey{(uint32_t)x, (uint32_t)(x >> 32)};
}
