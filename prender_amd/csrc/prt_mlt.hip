// prt_mlt.hip — kernels of the primary-sample-space Metropolis renderer
// (Render::RunMLT, render.h:360-780; KelemenMLT, mlt.h:70-170).  The paths
// themselves go through the wavefront kernels of prt_kernels.hip; these
// kernels mutate primary samples, make the proposals' camera rays, pick the
// chains' start paths and run the acceptance / splatting step.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "prt_chain.h"
#include "prt_math.h"
#include "prt_mlt.h"
#include "prt_shade.h"

namespace {

__device__ __forceinline__ void seed_words(const MltChains& C, uint32_t seed, uint32_t blk, uint32_t w[4]) {
  philox(seed, 0u, MLT_TAG_SEED, blk, C.k0, C.k1, w);
}

// One thread per (chain, block of 4 words).
__global__ __launch_bounds__(256) void k_mlt_mutate(MltChains C, int mode, uint32_t first, uint32_t n, uint32_t iter,
                                                    double p_large) {
  const uint32_t blocks = C.stride / 4u;
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)n * blocks) return;
  const uint32_t chain = (uint32_t)(t / blocks), blk = (uint32_t)(t % blocks);
  uint4* out = reinterpret_cast<uint4*>(C.prop + (size_t)chain * C.stride) + blk;
  if (mode == 0) {
    uint32_t w[4];
    seed_words(C, first + chain, blk, w);
    *out = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    const uint4 v = reinterpret_cast<const uint4*>(C.cur + (size_t)chain * C.stride)[blk];
    *out = mlt_propose(C, chain, iter, blk, p_large, v);
  }
}

__global__ __launch_bounds__(256) void k_mlt_gen(Params P, uint32_t n, RayQ q) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t* u = P.mlt_u + (size_t)i * (uint32_t)P.mlt_stride;
  d3 o, d;
  P.mlt_pix[i] = mlt_camera_ray(P, u, o, d);
  put_ray(q, i, o, d);
}

__global__ __launch_bounds__(256) void k_mlt_seed_record(const uint64_t* __restrict__ accum,
                                                         const uint32_t* __restrict__ pix_new, uint32_t first,
                                                         uint32_t n, MltSeeds S) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double f[3] = {accum_get(accum + 3 * (size_t)i), accum_get(accum + 3 * (size_t)i + 1),
                       accum_get(accum + 3 * (size_t)i + 2)};
  const size_t j = (size_t)first + i;
  S.f[3 * j] = f[0];
  S.f[3 * j + 1] = f[1];
  S.f[3 * j + 2] = f[2];
  // luminance in fixed point, capped so that 2^24 seeds cannot overflow
  const double l = lum3(f) * MLT_LUM_ONE + 0.5;
  S.lum[j] = l < 1099511627776.0 ? (uint64_t)l : 1099511627776ull;
  S.pix[j] = pix_new[i];
}

// Scan of MLT_SCAN_TILE-entry tiles: inclusive prefix within the tile, tile
// totals to tile_sums.
__global__ __launch_bounds__(256) void k_mlt_scan_tiles(MltSeeds S) {
  __shared__ uint64_t s_part[256];
  const uint32_t base = blockIdx.x * MLT_SCAN_TILE + threadIdx.x * 4u;
  uint64_t v[4];
  uint64_t run = 0;
  for (int k = 0; k < 4; ++k) {
    const uint32_t j = base + (uint32_t)k;
    run += j < S.n ? S.lum[j] : 0ull;
    v[k] = run;
  }
  s_part[threadIdx.x] = run;
  __syncthreads();
  for (uint32_t off = 1; off < 256; off <<= 1) {
    const uint64_t add = threadIdx.x >= off ? s_part[threadIdx.x - off] : 0ull;
    __syncthreads();
    s_part[threadIdx.x] += add;
    __syncthreads();
  }
  const uint64_t before = threadIdx.x ? s_part[threadIdx.x - 1] : 0ull;
  for (int k = 0; k < 4; ++k) {
    const uint32_t j = base + (uint32_t)k;
    if (j < S.n) S.cdf[j] = v[k] + before;
  }
  if (threadIdx.x == 255) S.tile_sums[blockIdx.x] = s_part[255];
}

// One block: exclusive prefix of the tile totals, in place.
__global__ __launch_bounds__(256) void k_mlt_scan_sums(MltSeeds S, uint32_t n_tiles) {
  __shared__ uint64_t s_part[256];
  uint64_t carry = 0;
  for (uint32_t b0 = 0; b0 < n_tiles; b0 += 256) {
    const uint32_t j = b0 + threadIdx.x;
    const uint64_t x = j < n_tiles ? S.tile_sums[j] : 0ull;
    s_part[threadIdx.x] = x;
    __syncthreads();
    for (uint32_t off = 1; off < 256; off <<= 1) {
      const uint64_t add = threadIdx.x >= off ? s_part[threadIdx.x - off] : 0ull;
      __syncthreads();
      s_part[threadIdx.x] += add;
      __syncthreads();
    }
    if (j < n_tiles) S.tile_sums[j] = carry + s_part[threadIdx.x] - x;
    const uint64_t total = s_part[255];
    __syncthreads();
    carry += total;
  }
}

__global__ __launch_bounds__(256) void k_mlt_scan_add(MltSeeds S) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= S.n) return;
  S.cdf[j] += S.tile_sums[j / MLT_SCAN_TILE];
}

// Start path of each chain: the first seed whose inclusive CDF exceeds
// u * total (mlt.h:201-220 picks the first with r <= accumulated, the same
// rule up to the boundary); then its primary samples, radiance and pixel.
__global__ __launch_bounds__(256) void k_mlt_init(MltChains C, MltSeeds S) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C.n) return;
  const uint64_t total = S.cdf[S.n - 1];
  uint32_t b[4];
  philox(c, 0u, MLT_TAG_INIT, 0u, C.k0, C.k1, b);
  uint64_t r = (uint64_t)(u01(b[0]) * (double)total);
  if (r >= total) r = total - 1;
  uint32_t lo = 0, hi = S.n - 1;  // smallest i with cdf[i] > r
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2u;
    if (S.cdf[mid] > r) hi = mid;
    else lo = mid + 1u;
  }
  const uint32_t seed = lo;
  uint4* cur = reinterpret_cast<uint4*>(C.cur + (size_t)c * C.stride);
  for (uint32_t blk = 0; blk < C.stride / 4u; ++blk) {
    uint32_t w[4];
    seed_words(C, seed, blk, w);
    cur[blk] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  C.f_old[3 * (size_t)c] = S.f[3 * (size_t)seed];
  C.f_old[3 * (size_t)c + 1] = S.f[3 * (size_t)seed + 1];
  C.f_old[3 * (size_t)c + 2] = S.f[3 * (size_t)seed + 2];
  C.pix_old[c] = S.pix[seed];
}

__global__ __launch_bounds__(256) void k_mlt_step(MltChains C, const uint64_t* __restrict__ accum, uint32_t iter,
                                                  double p_large, double b, double weight, double inv_m,
                                                  uint64_t* ctr) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  bool acc = false;
  if (c < C.n) {
    const double fn[3] = {accum_get(accum + 3 * (size_t)c), accum_get(accum + 3 * (size_t)c + 1),
                          accum_get(accum + 3 * (size_t)c + 2)};
    acc = mlt_accept(C, c, iter, p_large, b, weight, inv_m, fn, C.pix_new[c]);
    if (acc) {
      const uint4* src = reinterpret_cast<const uint4*>(C.prop + (size_t)c * C.stride);
      uint4* dst = reinterpret_cast<uint4*>(C.cur + (size_t)c * C.stride);
      for (uint32_t blk = 0; blk < C.stride / 4u; ++blk) dst[blk] = src[blk];
    }
  }
  const uint64_t n_acc = __popcll(__ballot(acc));
  if (lane_id() == 0) ctr_add(ctr, CTR_MLT_ACCEPT, n_acc);
}

__global__ __launch_bounds__(256) void k_mlt_resolve(const uint64_t* __restrict__ img, int64_t n, double scale,
                                                     void* out, int as_f64) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double v = (double)img[i] * MLT_FIX_INV * scale;
    if (as_f64) static_cast<double*>(out)[i] = v;
    else static_cast<float*>(out)[i] = (float)v;
  }
}

// ---------------------------------------------------------------- ERPT
// Block sums of the batch's path radiance (accumulators >> 8: 2^-24 fixed
// point), one atomic per block and channel.
__global__ __launch_bounds__(256) void k_erpt_sum(const uint64_t* __restrict__ accum, uint32_t n, uint64_t* sums) {
  __shared__ uint64_t s_sum[3][4];
  uint64_t v[3] = {0, 0, 0};
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    for (int k = 0; k < 3; ++k) v[k] += accum[3 * (size_t)i + k] >> 8;
  for (int k = 0; k < 3; ++k) {
    uint64_t x = v[k];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    if (lane_id() == 0) s_sum[k][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const uint64_t t = s_sum[threadIdx.x][0] + s_sum[threadIdx.x][1] + s_sum[threadIdx.x][2] + s_sum[threadIdx.x][3];
    if (t) atomicAdd((unsigned long long*)&sums[threadIdx.x], (unsigned long long)t);
  }
}

__global__ __launch_bounds__(256) void k_erpt_paths(const uint64_t* __restrict__ accum, ErptPaths E, uint32_t first,
                                                    uint64_t* img, double inv_samples, double ed, double mutation,
                                                    uint32_t k0, uint32_t k1) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= E.n) return;
  const double f[3] = {accum_get(accum + 3 * (size_t)i), accum_get(accum + 3 * (size_t)i + 1),
                       accum_get(accum + 3 * (size_t)i + 2)};
  const double l = lum3(f);
  E.f[3 * (size_t)i] = f[0];
  E.f[3 * (size_t)i + 1] = f[1];
  E.f[3 * (size_t)i + 2] = f[2];
  E.lum[i] = l;
  uint64_t chains = 0;
  if (E.direct[i]) {
    splat(img, E.pix[i], inv_samples, f);  // render.h:927-931
  } else if (l > 0.0 && ed > 0.0) {
    uint32_t r[4];
    philox(first + i, 0u, ERPT_TAG_CHAINS, 0u, k0, k1, r);
    const double c = floor(u01(r[0]) + l / (mutation * ed));  // render.h:938
    chains = c > 0.0 ? (uint64_t)c : 0ull;
  }
  E.count[i] = chains;
}

__global__ __launch_bounds__(256) void k_erpt_chain_init(ErptChains C, ErptPaths E, const uint32_t* __restrict__ path_u,
                                                         uint64_t j0, uint32_t first, int ss2, int width, int height) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= C.n) return;
  const uint64_t J = j0 + j;
  uint32_t lo = 0, hi = E.n - 1;  // the path whose chain range holds J
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2u;
    if (E.first[mid] > J) hi = mid;
    else lo = mid + 1u;
  }
  const uint32_t p = lo;
  const uint4* src = reinterpret_cast<const uint4*>(path_u + (size_t)p * C.stride);
  uint4* dst = reinterpret_cast<uint4*>(C.cur + (size_t)j * C.stride);
  for (uint32_t blk = 0; blk < C.stride / 4u; ++blk) dst[blk] = src[blk];
  C.f_y[3 * (size_t)j] = E.f[3 * (size_t)p];
  C.f_y[3 * (size_t)j + 1] = E.f[3 * (size_t)p + 1];
  C.f_y[3 * (size_t)j + 2] = E.f[3 * (size_t)p + 2];
  C.pix_y[j] = E.pix[p];
  // the loop pixel of initial path g = (y*W + x)*SS^2 + i (render.h:897-917)
  const uint32_t lp = (first + p) / (uint32_t)ss2;
  const int x = (int)(lp % (uint32_t)width), y = (int)(lp / (uint32_t)width);
  C.pix_now[j] = (uint32_t)((height - y - 1) * width + x);
  C.run[j] = 0u;
}

__global__ __launch_bounds__(256) void k_erpt_perturb(ErptChains C, uint32_t step, double d) {
  const uint32_t blocks = C.stride / 4u;
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)C.n * blocks) return;
  const uint32_t j = (uint32_t)(t / blocks), blk = (uint32_t)(t % blocks);
  const uint4 v = reinterpret_cast<const uint4*>(C.cur + (size_t)j * C.stride)[blk];
  reinterpret_cast<uint4*>(C.prop + (size_t)j * C.stride)[blk] = erpt_propose(C, j, step, blk, d, v);
}

__global__ __launch_bounds__(256) void k_erpt_step(ErptChains C, const uint64_t* __restrict__ accum, uint32_t step,
                                                   uint64_t* ctr) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  bool acc = false;
  if (j < C.n) {
    const double fz[3] = {accum_get(accum + 3 * (size_t)j), accum_get(accum + 3 * (size_t)j + 1),
                          accum_get(accum + 3 * (size_t)j + 2)};
    acc = erpt_accept(C, j, step, fz, C.pix_new[j]);
    if (acc) {
      const uint4* src = reinterpret_cast<const uint4*>(C.prop + (size_t)j * C.stride);
      uint4* dst = reinterpret_cast<uint4*>(C.cur + (size_t)j * C.stride);
      for (uint32_t blk = 0; blk < C.stride / 4u; ++blk) dst[blk] = src[blk];
    }
  }
  const uint64_t n_acc = __popcll(__ballot(acc));
  if (lane_id() == 0) ctr_add(ctr, CTR_MLT_ACCEPT, n_acc);
}

inline unsigned grid_of(uint64_t n, unsigned block = 256) { return (unsigned)((n + block - 1) / block); }

}  // namespace

hipError_t launch_mlt_mutate(const MltChains& C, int mode, uint32_t first, uint32_t n, uint32_t iter,
                             double p_large, hipStream_t s) {
  if (C.stride % 4u != 0 || n > C.n) return hipErrorInvalidValue;
  const uint64_t threads = (uint64_t)n * (C.stride / 4u);
  if (threads == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlt_mutate, dim3(grid_of(threads)), dim3(256), 0, s, C, mode, first, n, iter, p_large);
  return hipGetLastError();
}

hipError_t launch_mlt_gen(const Params& P, uint32_t n, const RayQ& q, hipStream_t s) {
  if (!P.mlt_u || !P.mlt_pix || n > q.cap) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlt_gen, dim3(grid_of(n)), dim3(256), 0, s, P, n, q);
  return hipGetLastError();
}

hipError_t launch_mlt_seed_record(const uint64_t* accum, const uint32_t* pix_new, uint32_t first, uint32_t n,
                                  const MltSeeds& S, hipStream_t s) {
  if ((uint64_t)first + n > S.n) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlt_seed_record, dim3(grid_of(n)), dim3(256), 0, s, accum, pix_new, first, n, S);
  return hipGetLastError();
}

hipError_t launch_mlt_scan(const MltSeeds& S, hipStream_t s) {
  if (S.n == 0) return hipErrorInvalidValue;
  const uint32_t tiles = (S.n + MLT_SCAN_TILE - 1) / MLT_SCAN_TILE;
  hipLaunchKernelGGL(k_mlt_scan_tiles, dim3(tiles), dim3(256), 0, s, S);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mlt_scan_sums, dim3(1), dim3(256), 0, s, S, tiles);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_mlt_scan_add, dim3(grid_of(S.n)), dim3(256), 0, s, S);
  return hipGetLastError();
}

hipError_t launch_mlt_init(const MltChains& C, const MltSeeds& S, hipStream_t s) {
  if (S.n == 0 || C.stride % 4u != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mlt_init, dim3(grid_of(C.n)), dim3(256), 0, s, C, S);
  return hipGetLastError();
}

hipError_t launch_mlt_step(const MltChains& C, const uint64_t* accum, uint32_t iter, double p_large, double b,
                           double weight, double inv_m, uint64_t* ctr, hipStream_t s) {
  hipLaunchKernelGGL(k_mlt_step, dim3(grid_of(C.n)), dim3(256), 0, s, C, accum, iter, p_large, b, weight, inv_m,
                     ctr);
  return hipGetLastError();
}

hipError_t launch_mlt_resolve(const uint64_t* img, int64_t n, double scale, void* out, int as_f64, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(k_mlt_resolve, dim3(g), dim3(256), 0, s, img, n, scale, out, as_f64);
  return hipGetLastError();
}

hipError_t launch_erpt_sum(const uint64_t* accum, uint32_t n, uint64_t* sums, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const unsigned g = (unsigned)std::min<uint64_t>(grid_of(n), 2048);
  hipLaunchKernelGGL(k_erpt_sum, dim3(g), dim3(256), 0, s, accum, n, sums);
  return hipGetLastError();
}

hipError_t launch_erpt_paths(const uint64_t* accum, const ErptPaths& E, uint32_t first, uint64_t* img,
                             double inv_samples, double ed, double mutation, uint32_t k0, uint32_t k1,
                             hipStream_t s) {
  if (E.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_erpt_paths, dim3(grid_of(E.n)), dim3(256), 0, s, accum, E, first, img, inv_samples, ed,
                     mutation, k0, k1);
  return hipGetLastError();
}

hipError_t launch_erpt_chain_init(const ErptChains& C, const ErptPaths& E, const uint32_t* path_u, uint64_t j0,
                                  uint32_t first, int ss2, int width, int height, hipStream_t s) {
  if (C.n == 0) return hipSuccess;
  if (E.n == 0 || C.stride % 4u != 0 || ss2 <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_erpt_chain_init, dim3(grid_of(C.n)), dim3(256), 0, s, C, E, path_u, j0, first, ss2, width,
                     height);
  return hipGetLastError();
}

hipError_t launch_erpt_perturb(const ErptChains& C, uint32_t step, double d, hipStream_t s) {
  if (C.stride % 4u != 0) return hipErrorInvalidValue;
  const uint64_t threads = (uint64_t)C.n * (C.stride / 4u);
  if (threads == 0) return hipSuccess;
  hipLaunchKernelGGL(k_erpt_perturb, dim3(grid_of(threads)), dim3(256), 0, s, C, step, d);
  return hipGetLastError();
}

hipError_t launch_erpt_step(const ErptChains& C, const uint64_t* accum, uint32_t step, uint64_t* ctr,
                            hipStream_t s) {
  if (C.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_erpt_step, dim3(grid_of(C.n)), dim3(256), 0, s, C, accum, step, ctr);
  return hipGetLastError();
}
