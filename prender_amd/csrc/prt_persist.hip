// prt_persist.hip — the path kernel: one launch follows every camera sample it
// is given along its whole path, with no ray queue and no launch per depth.
//
// It renders the samples of a batch of scenes (the batched renderer's
// persistent form and frames without light sampling), of one small frame or
// batch of Metropolis proposals (a depth-synchronous batch would pay two traversal launches
// per depth, each as long as its slowest ray), or the last rays of a
// depth-synchronous batch, from their queue.
//
// A wave keeps its 64 lanes on one path segment each.  Per trip: the light
// samples of the segments' origin vertices (three per diffuse vertex) and the
// segments' closest hits, then one radiance() vertex per segment (prt_shade.h),
// whose first child becomes the lane's next segment.  A light sample belongs
// to no lane: the three samples of every vertex are numbered through the wave
// and dealt out, first to the lanes without a segment (whose any-hit rays then
// run in the same traversal as the other lanes' closest hits), the rest 64 at
// a time, so a wave with few paths traces all rays of a vertex side by side and
// a full one wastes no lane on a vertex without light samples.  The second
// child of a glass vertex goes to the wave's pool, from which idle lanes take
// segments before they start new samples: a path's branches run side by side
// instead of one after the other.
//
// What bounds it: latency.  A trip of a wave is a traversal as long as its
// slowest ray (38,000 cycles with 7 paths of a 82k-triangle scene per wave,
// 29,000 per 64 rays of a full one), 6,000 to 10,000 cycles of dependent FP64
// chains in the vertices and 2,700 in 64 light samples.  So rays of one vertex
// run side by side, few samples are spread over all waves, records that
// every lane reads come from LDS, and scenes without light sampling have an
// instance without it (173 instead of 215 VGPRs).  Measured against one lane
// per sample that walks its glass tree and its light samples one after the
// other, and against depth-synchronous batches: spheres 32x24 x 8 spp 834 ->
// 175 us, 320x240 x 16 spp 1636 -> 951 us; mesh box 128x128 x 8 spp 2707 -> 926
// us; glass with light sampling 201x151 x 27 spp 5997 -> 3176 us; Metropolis
// batches of 15,360 chains 2.5 -> 0.41 ms.
//
// Markov chains of scenes without glass run here whole: a lane keeps a chain,
// accepts or rejects when its path has ended and goes on with the chain's next
// proposal, while the wave's other chains are wherever they are; the words of the
// proposals that are due are dealt over the lanes.  Chains in step cost the longest
// path of all chains per step: 15,360 chains x 64 steps 31.3 ms, each at its own
// pace 23.4 ms; 180,000 x 48 142.5 and 131.5 ms.
//
// A wave works on one scene at a time, so the scene's parameters are
// wave-uniform scalar loads: a lane starts a sample of another scene only
// after every lane of the wave has finished the previous scene's paths.
//
// The arithmetic is the queued renderers' (same vertex and NEE functions,
// segment throughput / pickup weight / NEE normal rounded to float as a queue
// stores them, contributions added in 32.32 fixed point), a sample's random
// numbers depend only on (pixel, sample, depth, branch), and integer sums do
// not depend on order, so every image equals the per-scene render bit for
// bit.  A lane sums its segments' light in LDS and adds it to the sample's
// accumulator (cleared before the launch) when its chain of segments ends.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "prt_chain.h"
#include "prt_device.h"
#include "prt_kernels.h"
#include "prt_math.h"
#include "prt_shade.h"
#include "prt_stream.h"
#include "prt_trace.h"

// 32.32 fixed-point value that accum_add would add for v.
__device__ __forceinline__ uint64_t fix_of(double v) {
  return v > 0.0 ? (uint64_t)(v * PRT_FIX_ONE + 0.5) : 0ull;
}

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ d3 shfl_d3(d3 v, int src) {
  return mk(__shfl(v.x, src, 64), __shfl(v.y, src, 64), __shfl(v.z, src, 64));
}

// materials a frame's blocks keep in LDS
#define PRT_PATH_MATERIALS 16

// Scene owning chunk c (c wave-uniform): the last s with chunk_base[s] <= c.
__device__ __forceinline__ int32_t scene_of_chunk(const Persist& st, uint32_t c) {
  int32_t lo = 0, hi = st.n_scenes;
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (st.chunk_base[mid] <= c) lo = mid;
    else hi = mid;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// SRC: PathSource.  NEE: some scene samples lights.  MANY: the analytic entities may
// be more than a block keeps in LDS.  NL: LDS stack entries; NTOP: BVH nodes kept
// in LDS; WAVES: waves per SIMD the registers are budgeted for.
template <int SRC, bool NEE, bool MANY, int NL, int NTOP, int WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void k_path(Persist st,
                                                                                                 Params P1) {
  const Params& P0 = SRC == PATH_BATCH ? st.scenes[0] : P1;
  PRT_DECLARE_STACK_N(S, P0, NL, 0);
  // the top-level node copy serves one scene only
  PRT_TOP_CACHE_N(S, P0.nodes, SRC != PATH_BATCH || st.n_scenes == 1 ? min(P0.n_wide, NTOP) : 0, NTOP);
  __shared__ uint64_t s_acc[3][256];  // light of each lane's chain so far
  __shared__ uint32_t s_pool[4];      // pool records of each wave
  __shared__ uint8_t s_map[256];      // lanes of each wave that hold a vertex to light, by rank
  // one scene's analytic entities and materials
  constexpr bool kCache = SRC != PATH_BATCH;
  __shared__ AnalyticSlot s_ana[kCache ? PRT_LDS_ANALYTIC : 1];
  __shared__ DevMaterial s_mats[kCache ? PRT_PATH_MATERIALS : 1];
  // its lights (at most NEE_LDS_LIGHTS); in a batch each wave's scene's, if it
  // has one light
  __shared__ LightSlot s_lights[!NEE ? 1 : kCache ? NEE_LDS_LIGHTS : 4];
  const LightSlot* lights = nullptr;
  const AnalyticSlot* slots = nullptr;
  const DevMaterial* lds_mats = nullptr;
  if (kCache) {
    slots = load_analytic_slots(P1, s_ana);
    if (!MANY) __builtin_assume(slots != nullptr);
    if (P1.n_materials <= PRT_PATH_MATERIALS) {
      if ((int)threadIdx.x < P1.n_materials) s_mats[threadIdx.x] = P1.mats[threadIdx.x];
      lds_mats = s_mats;
    }
    if (NEE && P1.n_lights <= NEE_LDS_LIGHTS) {
      if (threadIdx.x < 64u) load_light_slots(P1, s_lights);
      lights = s_lights;
    }
    __syncthreads();
  }
  const uint32_t lane = lane_id(), wib = threadIdx.x >> 6;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + wib));
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t wbase = wib * 64u;
  for (int c = 0; c < 3; ++c) s_acc[c][threadIdx.x] = 0ull;
  if (lane == 0) s_pool[wib] = 0u;
  wave_fence();
  PoolRec* pool = st.pool + (size_t)wave * PRT_PATH_POOL;
  TravStats tc{0, 0, 0}, tsh{0, 0, 0};
  uint32_t n_prim = 0, n_traced = 0, n_shadow = 0, truncated = 0, n_ext = 0, pickups = 0, dropped = 0;

  // wave-uniform work cursor: chunks [cb, ce), next sample co of chunk cb,
  // which belongs to scene cs (-1: not yet looked up) and holds cn samples; the
  // wave's current scene.  The first chunks are the wave's own (st.next starts
  // past them): one atomic per wave at the start would serialise the grid.
  const uint32_t n_chunks = SRC == PATH_QUEUE ? *st.cl.n : st.n_chunks;
  uint32_t cb = min(wave * st.claim, n_chunks), ce = min(cb + st.claim, n_chunks), co = 0, cn = 0;
  int32_t cs = -1, scene = SRC == PATH_BATCH ? -1 : 0;
  bool claims_left = n_chunks > gridDim.x * (blockDim.x >> 6) * st.claim;

  // the lane's segment
  bool act = false;
  d3 o = mk(0.0, 0.0, 0.0), d = o;
  float tr[3] = {1.0f, 1.0f, 1.0f}, pw[3] = {0.0f, 0.0f, 0.0f}, nr[3] = {0.0f, 0.0f, 0.0f};
  uint32_t meta = 0, slot = 0;  // slot: sample of the scene (frame, queue: of the batch), or chain
  // its chain: the step, that step's image element and Philox key; whether the
  // next proposal is due, and whether the last one was accepted
  uint32_t it = 0, element = 0, accepts = 0;
  RngKey key = SRC == PATH_CHAIN ? RngKey{0u, 0u} : key_of(P0);
  bool due = false, took = false;

  while (true) {
    // ---- idle lanes take the wave's waiting segments, then new samples
    uint64_t need = __ballot(!act);
    const uint32_t waiting = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(s_pool[wib], PRT_PATH_POOL));
    uint32_t left = waiting;
    if (need && waiting) {
      const uint32_t take = min((uint32_t)__popcll(need), waiting), rank = (uint32_t)__popcll(need & below);
      if (!act && rank < take) {
        const PoolRec& r = pool[waiting - 1u - rank];
        o = mk(r.o[0], r.o[1], r.o[2]);
        d = mk(r.d[0], r.d[1], r.d[2]);
        for (int j = 0; j < 3; ++j) {
          tr[j] = r.t[j];
          pw[j] = r.p[j];
        }
        meta = r.meta;
        slot = r.slot;
        act = true;
      }
      left = waiting - take;
      if (lane == 0) s_pool[wib] = left;
      wave_fence();
      need = __ballot(!act);
    }
    uint32_t room = 64u - (uint32_t)__popcll(need);  // segments held
    room = left == 0u && st.quota > room ? st.quota - room : 0u;
    while (need && room) {
      if (cb >= ce) {
        if (!claims_left) break;
        uint32_t c0 = 0;
        if (lane == 0) c0 = atomicAdd(st.next, st.claim);
        c0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)__shfl((int)c0, 0, 64));
        if (c0 >= n_chunks) {
          claims_left = false;
          break;
        }
        cb = c0;
        ce = min(c0 + st.claim, n_chunks);
        co = 0;
        cs = -1;
      }
      if (cs < 0) {
        if (SRC == PATH_BATCH) {
          cs = scene_of_chunk(st, cb);
          const uint64_t first = (uint64_t)(cb - st.chunk_base[cs]) * 64u;
          const uint64_t n_s = st.sample_base[cs + 1] - st.sample_base[cs];
          cn = (uint32_t)__builtin_amdgcn_readfirstlane((int)(n_s - first < 64u ? n_s - first : 64u));
        } else if (SRC == PATH_FRAME || SRC == PATH_CHAIN) {
          cs = 0;
          cn = min(st.unit, st.n_samples - cb * st.unit);
        } else {
          cs = 0;
          cn = (uint32_t)__builtin_amdgcn_readfirstlane((int)st.cl.desc[cb].y);
        }
      }
      if (SRC == PATH_BATCH && cs != scene) {
        if (__any(act)) break;  // the wave finishes its scene's paths first
        scene = cs;
        const Params& P = scene_params(st.scenes, scene);
        lights = nullptr;
        if (NEE && P.nee && P.n_lights == 1) {
          load_light_slots(P, s_lights + wib);
          lights = s_lights + wib;
        }
      }
      const uint32_t take = min(min((uint32_t)__popcll(need), room), cn - co);
      const uint32_t rank = (uint32_t)__popcll(need & below);
      if (!act && rank < take) {
        const Params& P = SRC == PATH_BATCH ? scene_params(st.scenes, scene) : P1;
        if (SRC == PATH_QUEUE) {
          const uint32_t i = st.cl.desc[cb].x + co + rank;
          d3 T, Pw;
          get_ray(st.q, i, o, d);
          get_segment(st.q, i, T, Pw, meta, slot);
          tr[0] = (float)T.x; tr[1] = (float)T.y; tr[2] = (float)T.z;
          pw[0] = (float)Pw.x; pw[1] = (float)Pw.y; pw[2] = (float)Pw.z;
          meta &= ~(META_NEE | META_PICK);
        } else {
          if (SRC == PATH_BATCH) slot = (cb - st.chunk_base[scene]) * 64u + co + rank;
          else slot = cb * st.unit + co + rank;
          if (SRC == PATH_CHAIN) {
            it = st.chain.it0;
            due = true;
          } else if (SRC == PATH_FRAME && P.mlt_u != nullptr) {  // a Metropolis proposal's own camera ray
            get_ray(st.q, slot, o, d);
          } else {
            const int64_t pixel = st.batch.pixel_base + (int64_t)(slot / (uint32_t)P.spp);
            const int sub = (int)(slot % (uint32_t)P.spp % (uint32_t)(P.SS * P.SS));
            camera_ray(P, (int)(pixel % P.W), (int)(pixel / P.W), sub % P.SS, sub / P.SS, o, d);
          }
          tr[0] = tr[1] = tr[2] = 1.0f;
          pw[0] = pw[1] = pw[2] = 0.0f;
          meta = rng_c2(0, 1u);
          if (SRC != PATH_CHAIN) ++n_prim;
        }
        act = true;
      }
      co += take;
      room -= take;
      if (co >= cn) {
        ++cb;
        co = 0;
        cs = -1;
      }
      need = __ballot(!act);
    }
    if (!__any(act)) {
      if (!claims_left && cb >= ce) break;
      continue;
    }
    const Params& P = SRC == PATH_BATCH ? scene_params(st.scenes, scene) : P1;
    if (SRC == PATH_CHAIN) {
      // ---- proposals that are due, their words dealt over the wave's lanes
      const ChainRun& R = st.chain;
      const uint64_t due_m = __ballot(due);
      if (due_m) {
        const uint32_t stride = (uint32_t)P.mlt_stride, blocks = stride / 4u;
        const uint32_t n_items = blocks * (uint32_t)__popcll(due_m);
        uint32_t* words = R.erpt_on ? R.erpt.cur : R.mlt.cur;
        uint32_t* prop = R.erpt_on ? R.erpt.prop : R.mlt.prop;
        if (due) s_map[wbase + (uint32_t)__popcll(due_m & below)] = (uint8_t)lane;
        wave_fence();
        for (uint32_t base = 0; base < n_items; base += 64u) {
          const uint32_t item = base + lane, blk = item % blocks;
          const int src = item < n_items ? (int)s_map[wbase + item / blocks] : (int)lane;
          const uint32_t chain = (uint32_t)__shfl((int)slot, src, 64), step = (uint32_t)__shfl((int)it, src, 64);
          const bool moved = __shfl((int)took, src, 64) != 0;
          if (item < n_items) {
            uint4* cur = reinterpret_cast<uint4*>(words + (size_t)chain * stride) + blk;
            uint4* out = reinterpret_cast<uint4*>(prop + (size_t)chain * stride) + blk;
            const uint4 v = moved ? *out : *cur;
            if (moved) *cur = v;
            if (step < R.it1)
              *out = R.erpt_on ? erpt_propose(R.erpt, chain, step, blk, R.d, v)
                               : mlt_propose(R.mlt, chain, step, blk, R.p_large, v);
          }
        }
        wave_fence();
        if (due) {
          due = took = false;
          if (it < R.it1) {
            element = mlt_camera_ray(P, prop + (size_t)slot * stride, o, d);
            key = chain_key(R.key0 + it);
            tr[0] = tr[1] = tr[2] = 1.0f;
            pw[0] = pw[1] = pw[2] = 0.0f;
            meta = rng_c2(0, 1u);
            ++n_prim;
          } else {
            act = false;
          }
        }
        if (!__any(act)) continue;
      }
    }
    const uint32_t pixel =
        SRC == PATH_CHAIN ? slot : (uint32_t)(st.batch.pixel_base + (int64_t)(slot / (uint32_t)P.spp));
    const uint32_t k = SRC == PATH_CHAIN ? 0u : slot % (uint32_t)P.spp;
    if (SRC != PATH_CHAIN) key = key_of(P);
    // ---- light samples and closest hits
    double t = PS_INF;
    int32_t id = -1;
    if (!NEE) {
      if (act) {
        (void)trace_lane(P, slots, o + d * 0.000001, d, false, t, id, S, tc, tsh);
        ++n_traced;
      }
    } else {
      const bool lit = act && (meta & META_NEE);
      const uint64_t lit_m = __ballot(lit);
      const uint32_t n_items = 3u * (uint32_t)__popcll(lit_m);
      if (lit) s_map[wbase + (uint32_t)__popcll(lit_m & below)] = (uint8_t)lane;
      wave_fence();
      const uint32_t n_idle = 64u - (uint32_t)__popcll(__ballot(act));
      uint32_t item = act ? 0xFFFFFFFFu : (uint32_t)__popcll(__ballot(!act) & below);  // this round's light sample
      for (uint32_t base = n_idle;; base += 64u) {
        const bool first = base == n_idle;
        const bool has = item < n_items;
        bool shadow = false;
        ShadowRay sr{};
        int src = (int)lane;
        if (__any(has)) {
          if (has) src = (int)s_map[wbase + item / 3u];
          const d3 x = shfl_d3(o, src);
          const d3 nrm = mk(__shfl(nr[0], src, 64), __shfl(nr[1], src, 64), __shfl(nr[2], src, 64));
          const d3 ct = mk(__shfl(tr[0], src, 64), __shfl(tr[1], src, 64), __shfl(tr[2], src, 64));
          const uint32_t sp = (uint32_t)__shfl((int)pixel, src, 64), sk = (uint32_t)__shfl((int)k, src, 64);
          const uint32_t sm = (uint32_t)__shfl((int)meta, src, 64);
          RngKey sample_key = key;
          if (SRC == PATH_CHAIN)
            sample_key = RngKey{(uint32_t)__shfl((int)key.k0, src, 64), (uint32_t)__shfl((int)key.k1, src, 64)};
          if (has) {
            uint32_t w[3];
            nee_words_of(sample_key, sp, sk, (int)(sm & 0xFFu) - 1, META_BRANCH(sm), (int)(item % 3u), w);
            int32_t l = -1;
            shadow = lights ? nee_one_slots(P, lights, w, 0, x, nrm, ct, sr, l) : nee_one(P, w, 0, x, nrm, ct, sr, l);
          }
        }
        const bool closest = first && act;
        if (closest || shadow) {
          double tt = closest ? PS_INF : sr.tmax;
          int32_t hid = -1;
          const bool blocked = trace_lane(P, slots, closest ? o + d * 0.000001 : sr.o2, closest ? d : sr.dir, !closest, tt, hid,
                                          S, tc, tsh);
          if (closest) {
            t = tt;
            id = hid;
            ++n_traced;
          } else {
            ++n_shadow;
            if (!blocked) {
              for (int c = 0; c < 3; ++c)
                if (const uint64_t v = fix_of(sr.c[c]))
                  atomicAdd((unsigned long long*)&s_acc[c][wbase + (uint32_t)src], (unsigned long long)v);
            }
          }
        }
        if (base >= n_items) break;
        item = base + lane;
      }
    }
    wave_fence();
    // ---- the segments' vertices
    if (act) {
      LaneCtx C;
      C.has0 = false;
      C.pool = pool;
      C.pool_n = &s_pool[wib];
      C.slot = slot;
      C.truncated = C.n_ext = C.pickups = C.dropped = C.direct = 0;
      VertexAdj va;
      const int depth = (int)(meta & 0xFFu);
      const d3 add = shade_vertex(P, lds_mats ? lds_mats : P.mats, C, o, d, t, id, mk(tr[0], tr[1], tr[2]), mk(pw[0], pw[1], pw[2]), key, pixel,
                                  k, depth, META_BRANCH(meta), va);
      uint64_t acc[3] = {fix_of(add.x), fix_of(add.y), fix_of(add.z)};
      truncated += C.truncated;
      n_ext += C.n_ext;
      pickups += C.pickups;
      dropped += C.dropped;
      if (SRC == PATH_FRAME && depth == 0 && P.mlt_flags != nullptr) P.mlt_flags[slot] = C.direct;
      if (C.has0) {
        for (int c = 0; c < 3; ++c)
          if (acc[c]) s_acc[c][threadIdx.x] += acc[c];
        o = C.o0;
        d = C.d0;
        for (int j = 0; j < 3; ++j) {
          tr[j] = C.t0[j];
          pw[j] = C.p0[j];
          nr[j] = C.n0[j];
        }
        meta = C.meta0;
      } else if (SRC == PATH_CHAIN) {
        double f[3];
        for (int c = 0; c < 3; ++c) {
          acc[c] += s_acc[c][threadIdx.x];
          s_acc[c][threadIdx.x] = 0ull;
          f[c] = accum_get(&acc[c]);
        }
        const ChainRun& R = st.chain;
        took = R.erpt_on ? erpt_accept(R.erpt, slot, it, f, element)
                         : mlt_accept(R.mlt, slot, it, R.p_large, R.b, R.weight, R.inv_m, f, element);
        accepts += took ? 1u : 0u;
        ++it;
        due = true;
      } else {
        const uint64_t at = (SRC == PATH_BATCH ? st.sample_base[scene] : 0ull) + slot;
        for (int c = 0; c < 3; ++c) {
          acc[c] += s_acc[c][threadIdx.x];
          s_acc[c][threadIdx.x] = 0ull;
          if (acc[c]) atomicAdd((unsigned long long*)&st.accum[3 * at + c], (unsigned long long)acc[c]);
        }
        act = false;
      }
    }
  }
  flush_stats(st.ctr, CTR_NODES, tc);
  flush_stats(st.ctr, CTR_SNODES, tsh);
  const uint64_t s_prim = wave_sum_u32(n_prim), s_tr = wave_sum_u32(n_traced), s_sh = wave_sum_u32(n_shadow);
  const uint64_t s_ext = wave_sum_u32(n_ext), s_pick = wave_sum_u32(pickups), s_trunc = wave_sum_u32(truncated);
  const uint64_t s_drop = wave_sum_u32(dropped), s_acc_n = SRC == PATH_CHAIN ? wave_sum_u32(accepts) : 0ull;
  if (lane == 0) {
    auto count = [&](int c, uint64_t v) { ctr_add(st.ctr, c, v); };
    count(CTR_QUEUED, s_prim + s_ext);
    count(CTR_TRACED, s_tr);
    count(CTR_SHADOW, s_sh);
    count(CTR_STRACED, s_sh);
    count(CTR_EXT, s_ext);
    count(CTR_PICKUP, s_pick);
    count(CTR_TRUNC, s_trunc);
    count(CTR_DROP, s_drop);
    if (SRC == PATH_CHAIN) count(CTR_MLT_ACCEPT, s_acc_n);
  }
}
// Every pixel of every scene of the batch: fold its samples' accumulators
// into the scene's image (fold_pixel: 1/spp scale, luminance clamp,
// sensor_response, variance of the mean).  pixel_base[s]: first pixel of
// scene s in the batch's pixel numbering ([n_scenes + 1]).
__global__ __launch_bounds__(256) void k_persist_resolve(Persist st, int64_t n_pix, const int64_t* pixel_base) {
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n_pix; g += (int64_t)gridDim.x * blockDim.x) {
    int32_t lo = 0, hi = st.n_scenes;
    while (hi - lo > 1) {
      const int32_t mid = (lo + hi) >> 1;
      if (pixel_base[mid] <= g) lo = mid;
      else hi = mid;
    }
    const Params& P = st.scenes[lo];
    const int64_t pix = g - pixel_base[lo];
    const int x = (int)(pix % P.W), y = (int)(pix / P.W);
    const size_t ii = (size_t)(P.H - y - 1) * P.W + x;  // render.h:1234
    double c[3], v[3];
    fold_pixel(P, st.accum + 3 * (st.sample_base[lo] + (uint64_t)pix * (uint64_t)P.spp), c, v);
    float* rgb = st.out_rgb[lo];
    float* var = st.out_var[lo];
    for (int j = 0; j < 3; ++j) {
      rgb[3 * ii + j] = (float)c[j];
      if (var) var[3 * ii + j] = (float)v[j];
    }
  }
}

// ------------------------------------------------------------ launchers
// Two register budgets, neither of which spills vector registers: 2 waves per
// SIMD, and without light sampling 3 (168 VGPRs), for launches that fill them
// (spheres 320x240 x 16 spp 1033 -> 951 us).  A smaller launch gains nothing
// from more waves and loses the LDS.  An instance for 4 waves with light sampling
// (128 VGPRs, 151 spilled to scratch memory) gave wrong sums for a reason not
// found, so the build refuses an instance that spills vector registers
// (build.py, check_spills).
// LDS of the instances: at 2 waves (two blocks per CU) 12 stack entries and
// five BVH levels, so that the tree's top costs an LDS access instead of an L2
// one, or for a batch of scenes, which shares no tree, 32 entries; at 3 waves 14
// entries and four levels, or 20.
// Frames without light sampling have an instance without the loop over more
// analytic entities than the LDS copy holds: its scalars raised the three-wave
// one's spills from 139 to 154 (spheres 320x240 x 16 spp 934 -> 955 us).
template <int SRC, bool NEE, bool MANY, class F>
static hipError_t with_path_waves(int waves, F&& f) {
  constexpr bool batch = SRC == PATH_BATCH;
  if constexpr (!NEE)
    if (waves >= 3) return f(k_path<SRC, NEE, MANY, batch ? 20 : 14, batch ? PRT_TOP_NODES : 85, 3>);
  return f(k_path<SRC, NEE, MANY, batch ? 32 : 12, batch ? PRT_TOP_NODES : PRT_WIDE_NODES, 2>);
}
template <class F>
static hipError_t with_path_kernel(PathSource src, bool nee, bool many, int waves, F&& f) {
  if (src == PATH_BATCH)
    return nee ? with_path_waves<PATH_BATCH, true, true>(waves, f) : with_path_waves<PATH_BATCH, false, true>(waves, f);
  if (src == PATH_CHAIN) return with_path_waves<PATH_CHAIN, true, true>(waves, f);
  if (src == PATH_QUEUE) return with_path_waves<PATH_QUEUE, true, true>(waves, f);
  if (nee) return with_path_waves<PATH_FRAME, true, true>(waves, f);
  return many ? with_path_waves<PATH_FRAME, false, true>(waves, f) : with_path_waves<PATH_FRAME, false, false>(waves, f);
}

hipError_t launch_path(PathSource src, const Persist& p, const Params& P, int waves, int blocks, hipStream_t s) {
  return with_path_kernel(src, p.nee != 0, P.n_analytic > PRT_LDS_ANALYTIC, waves, [&](void (*k)(Persist, Params)) {
    hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, s, p, P);
    return hipGetLastError();
  });
}

hipError_t launch_persist_resolve(const Persist& p, int64_t n_pixels_total, const int64_t* d_pixel_base,
                                  hipStream_t s) {
  int64_t g = (n_pixels_total + 255) / 256;
  if (g < 1) g = 1;
  if (g > 8192) g = 8192;
  hipLaunchKernelGGL(k_persist_resolve, dim3((unsigned)g), dim3(256), 0, s, p, n_pixels_total, d_pixel_base);
  return hipGetLastError();
}
