// prt_trace.h — BVH traversal on gfx950: closest hit and any hit over the
// 4-wide node records, with a per-lane stack in LDS.
//
// Semantics are those of intersect_scene_ (scene.cpp:83-214) over the
// reference's QBVH (QBVH.cpp:17-159): the 1e-6 origin nudge, hits accepted at
// t > 1e-6, the nearest hit kept.  The float box test differs from the
// reference's only in being conservative (boxes carry a margin and NaN slabs
// impose no bound), so it never prunes a box that holds the closest hit.
#pragma once
#include "prt_kernels.h"
#include "prt_math.h"

struct TravStats {
  uint32_t nodes, tris;
  uint32_t rays;  // queries finished (traverse_pool)
};

// Per-lane traversal stack of (node, t) entries: the first NL in LDS (lane
// interleaved, one 64-bit entry per level, bank-conflict free), deeper ones
// in a global overflow area of Params::ovf_words words per thread (enough for
// the scene's BVH depth), thread interleaved as well: entry k of every
// thread of a region lies together (k * ovf_threads + thread), so the lanes
// of a wave that spill at the same depth write 512 contiguous bytes instead
// of 64 lines.
//
// An entry is a 64-bit key, t in the high word and the node in the low one, as
// node_keys sorts them.  The levels of all lanes of a wave are usually in LDS,
// which a wave-uniform branch finds out: entries are then written without a
// branch per child (a miss is overwritten by the next entry), and read two at a
// time.
//
// The overflow area, the nodes and the triangles lie in device memory, which
// their pointers' type says: a pointer that a kernel reads from memory (the
// scenes of a batch) is a flat one otherwise, whose loads wait for LDS accesses
// as well and take no scalar base.
#define PRT_GLOBAL __attribute__((address_space(1)))
// memory that nothing writes during the kernel: uniform reads are scalar loads
#define PRT_CONST __attribute__((address_space(4)))
// four floats as a native vector (copyable out of an address-space-qualified
// object, unlike float4)
typedef float prt_f4 __attribute__((ext_vector_type(4)));

template <int NL>
struct StackN {
  static constexpr int stride = 256;  // threads per block of every traversal kernel
  static constexpr int levels = NL;
  uint64_t* lds;                      // [NL][256]
  PRT_GLOBAL uint64_t* ovf;           // this thread's first overflow entry
  size_t ostride;                     // entries between its consecutive overflow entries
  // (3 * BVH depth + 1 - NL overflow entries used at most)
  // the block's LDS copy of BVH nodes 0..n_top-1 (PRT_TOP_CACHE)
  const __attribute__((address_space(3))) prt_f4* top = nullptr;
  int n_top = 0;
  __device__ __forceinline__ void put(int k, uint64_t key) {
    if (k < NL) lds[k * stride] = key;
    else ovf[(size_t)(k - NL) * ostride] = key;
  }
  __device__ __forceinline__ uint64_t get(int k) const {
    return k < NL ? lds[k * stride] : ovf[(size_t)(k - NL) * ostride];
  }
};
typedef StackN<PRT_STACK_LDS> Stack;

// Blocks of 256 threads; a thread's overflow area is picked by its global
// index modulo ovf_threads (the host sizes the area for the largest grid)
// within one of PRT_OVF_REGIONS regions: closest-hit and path kernels use region
// 0, shadow kernels region 1, because the two run at the same time on two
// streams.  Two launches that use one region must have an order between them.
#define PRT_DECLARE_STACK_N(S, P, NL, REGION)                                                             \
  __shared__ uint64_t s_stack_[(NL) * 256];                                                               \
  StackN<NL> S{s_stack_ + threadIdx.x,                                                                    \
               (PRT_GLOBAL uint64_t*)((P).stack_ovf +                                                     \
                                      (size_t)(REGION) * (size_t)(P).ovf_threads * (size_t)(P).ovf_words) + \
                   (size_t)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) % (P).ovf_threads),          \
               (size_t)(P).ovf_threads}
#define PRT_DECLARE_STACK(S, P, REGION) PRT_DECLARE_STACK_N(S, P, PRT_STACK_LDS, REGION)

// Copies BVH nodes 0..NTOP-1 (the top levels, numbered first by the builder;
// NTOP <= PRT_TOP_NODES, or <= CAP) into the block's LDS for stack S.  Every thread of
// the block must reach it.
#define PRT_TOP_CACHE(S, NODES, NTOP) PRT_TOP_CACHE_N(S, NODES, NTOP, PRT_TOP_NODES)
#define PRT_TOP_CACHE_N(S, NODES, NTOP, CAP)                                                 \
  __shared__ float4 s_top_[(CAP) * 8];                                                       \
  {                                                                                          \
    const int nt_ = (NTOP);                                                                  \
    const float4* g_ = reinterpret_cast<const float4*>(NODES);                               \
    for (int k_ = (int)threadIdx.x; k_ < nt_ * 8; k_ += (int)blockDim.x) s_top_[k_] = g_[k_]; \
    __syncthreads();                                                                         \
    S.top = (const __attribute__((address_space(3))) prt_f4*)s_top_;                         \
    S.n_top = nt_;                                                                           \
  }

// a float >= t (t > 0): the culling bound never drops below the double hit
__device__ __forceinline__ float fup(double t) {
  const float f = (float)t;
  return (double)f < t ? __uint_as_float(__float_as_uint(f) + 1u) : f;
}

// Byte offsets within a 128-byte node record of the row holding each axis'
// entry planes, packed x | y << 8 | z << 16: the lo row (x 0, y 16, z 32)
// where the ray's inverse direction on that axis is >= 0, else the hi row
// (x 48, y 64, z 80).  The exit planes are in the other row, at the entry
// offset XOR 48, 80 or 112.  ix, iy, iz are never zero (|1 / d| >= 1 for a
// unit direction, and an infinite one is clamped to +-1e30).
__device__ __forceinline__ uint32_t entry_rows(float ix, float iy, float iz) {
  return (ix < 0.0f ? 48u : 0u) | ((iy < 0.0f ? 64u : 16u) << 8) | ((iz < 0.0f ? 80u : 32u) << 16);
}

// 1 / d for the float slab test; where that overflows, +-1e30.  An approximate
// reciprocal and two Newton steps, which gave the quotient's float for every one
// of 4.3e9 d in each of four ranges from 2^-125 to 2^120 (the double's error was
// nil there; after one step it was up to 2.2e-15, and 10 floats differed).
__device__ __forceinline__ float ray_inverse(double d) {
  const double y0 = __builtin_amdgcn_rcp(d);
  const double y = __builtin_fma(__builtin_fma(-d, y0, 1.0), y0, y0);
  const float i = (float)__builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  return fabsf(i) < __builtin_inff() ? i : __builtin_copysignf(1.0e30f, (float)d);
}

// Smaller of two keys into a, larger into b.  A key's high word is a float in
// [0, +inf], so as a double it is positive and finite (0x7F800000 is no
// double's infinity) and its order is the keys' order as integers; the 64-bit
// minimum leaves its operand's bits alone, denormals included.
__device__ __forceinline__ void key_order(uint64_t& a, uint64_t& b) {
  const double x = __longlong_as_double((long long)a), y = __longlong_as_double((long long)b);
  double lo, hi;
  asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(x), "v"(y));
  asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(x), "v"(y));
  a = (uint64_t)__double_as_longlong(lo);
  b = (uint64_t)__double_as_longlong(hi);
}
#define PRT_KEY_MISS 0x7F800000u
__device__ __forceinline__ bool key_hit(uint64_t key) { return (uint32_t)(key >> 32) != PRT_KEY_MISS; }

// Slab test of the 4 children of node `cur` against the ray's float slabs: a key
// per child, entry distance (+inf: miss) over child reference, ascending.
// Each axis reads its entry and exit planes from the rows entry_rows picks:
// fma(c, i, -oi) is monotonic in the plane coordinate c and every child has
// lo <= hi (an empty slot lo = hi = +inf), so the entry plane's distance is
// exactly the smaller of the two, without a min / max per axis.
// The keys' sort is ten 64-bit minima and maxima (25 instructions as exchanges
// by selects, 45 as 32-bit keys whose children are picked afterwards).
// Nodes of the top levels come from the block's LDS copy (without it the
// 82k-triangle box took 34.0 instead of 33.3 ms a frame), others at a 32-bit
// offset from a scalar base while that reaches all nodes (2^25 of them).
template <class Stk>
__device__ __forceinline__ void node_keys(const Stk& S, const DevNode* nodes, int32_t n_nodes, int32_t cur, uint32_t rows,
                                          float ix, float iy, float iz, float oix, float oiy, float oiz, float tb,
                                          uint64_t key[4]) {
  const uint32_t nx = rows & 0xFFu, ny = (rows >> 8) & 0xFFu, nz = rows >> 16;
  // entry x, y, z rows, exit x, y, z rows, children
  const uint32_t off[7] = {nx, ny, nz, nx ^ 48u, ny ^ 80u, nz ^ 112u, 96u};
  prt_f4 nd[7];
  if (cur < S.n_top) {
    typedef const __attribute__((address_space(3))) char lds_c;
    typedef const __attribute__((address_space(3))) prt_f4 lds_f4;
    lds_c* t = reinterpret_cast<lds_c*>(S.top);
#pragma unroll
    for (int k = 0; k < 7; ++k) nd[k] = *reinterpret_cast<lds_f4*>(t + (((uint32_t)cur << 7) + off[k]));
  } else {
    typedef const PRT_GLOBAL char glb_c;
    typedef const PRT_GLOBAL prt_f4 glb_f4;
    glb_c* g = (glb_c*)nodes;
    if (n_nodes <= (1 << 25)) {
#pragma unroll
      for (int k = 0; k < 7; ++k) nd[k] = *reinterpret_cast<glb_f4*>(g + (((uint32_t)cur << 7) | off[k]));
    } else {
      g += (size_t)cur << 7;
#pragma unroll
      for (int k = 0; k < 7; ++k) nd[k] = *reinterpret_cast<glb_f4*>(g + off[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float x0 = __builtin_fmaf(nd[0][k], ix, -oix), x1 = __builtin_fmaf(nd[3][k], ix, -oix);
    const float y0 = __builtin_fmaf(nd[1][k], iy, -oiy), y1 = __builtin_fmaf(nd[4][k], iy, -oiy);
    const float z0 = __builtin_fmaf(nd[2][k], iz, -oiz), z1 = __builtin_fmaf(nd[5][k], iz, -oiz);
    const float tnear = fmaxf(fmaxf(x0, y0), fmaxf(z0, 0.0f));
    const float tfar = fminf(fminf(x1, y1), fminf(z1, tb));
    const uint32_t t = (tnear <= tfar) ? __float_as_uint(tnear) : PRT_KEY_MISS;
    key[k] = ((uint64_t)t << 32) | __float_as_uint(nd[6][k]);
  }
  key_order(key[0], key[1]);
  key_order(key[2], key[3]);
  key_order(key[0], key[2]);
  key_order(key[1], key[3]);
  key_order(key[1], key[2]);
}

// Pushes keys 3, 2, 1 of a node (farthest first) that are hits.
template <class Stk>
__device__ __forceinline__ void push_keys(Stk& S, int& sp, const uint64_t key[4]) {
  if (!__any(sp > Stk::levels - 3)) {
#pragma unroll
    for (int j = 3; j >= 1; --j) {
      S.lds[sp * Stk::stride] = key[j];
      sp += key_hit(key[j]) ? 1 : 0;
    }
  } else {
#pragma unroll
    for (int j = 3; j >= 1; --j)
      if (key_hit(key[j])) S.put(sp++, key[j]);
  }
}

// A lane's place in the tree: an internal node (0 <= cur < PRT_TRAV_POP), a leaf
// code (< 0), PRT_TRAV_POP (its next node is on the stack, which is not empty) or
// PRT_TRAV_DONE.
#define PRT_TRAV_DONE 0x7FFFFFFF
#define PRT_TRAV_POP 0x7FFFFFFE
__device__ __forceinline__ int32_t next_entry(int sp) { return sp > 0 ? PRT_TRAV_POP : PRT_TRAV_DONE; }

// Takes the top two entries of a lane at PRT_TRAV_POP, as far as it needs them:
// an entry beyond tb is dropped, a first leaf is parked in lf (>= 0: none).  A lane
// that finds nothing stays at PRT_TRAV_POP.  A loop until every lane of the wave
// has its node ran as often as the lane with the most stale entries: after a hit
// that is most of the stack, at some 25 instructions an entry for one lane.
template <class Stk>
__device__ __forceinline__ void pop_two(const Stk& S, int& sp, float tb, int32_t& cur, int32_t& lf) {
  uint64_t e[2];
  const int k1 = max(sp - 2, 0);
  if (!__any(sp > Stk::levels)) {
    e[0] = S.lds[(sp - 1) * Stk::stride];
    e[1] = S.lds[k1 * Stk::stride];
  } else {
    e[0] = S.get(sp - 1);
    e[1] = S.get(k1);
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (cur == PRT_TRAV_POP) {
      const int32_t node = (int32_t)(uint32_t)e[k];
      const bool open = __uint_as_float((uint32_t)(e[k] >> 32)) <= tb, park = open && node < 0 && lf >= 0;
      --sp;
      lf = park ? node : lf;
      cur = open && !park ? node : next_entry(sp);
    }
  }
}

// While-while traversal with speculative leaf postponement (Aila & Laine,
// "Understanding the Efficiency of Ray Traversal on GPUs", HPG 2009): a lane
// walks internal nodes until it meets a leaf, parks that leaf and keeps
// walking until every lane of the wave holds a parked leaf (or is done);
// then the whole wave tests triangles together.  Node visits and triangle
// tests thus run with most lanes active instead of interleaving a node
// step of some lanes with a leaf loop of others in every trip.
//
// intersect_scene_ (scene.cpp:83-214) tests the entities in index order and
// keeps a hit only when strictly nearer, so of hits at exactly the same t the
// one of the lowest entity index wins (a box standing on the ground mesh
// meets it in a shared plane).  Within one mesh the QBVH keeps the first
// triangle it finds; that order is the reference tree's, which this BVH does
// not reproduce.
__device__ __forceinline__ bool nearer_hit(double t, int32_t ent, double t_best, int32_t ent_best) {
  return t < t_best || (t == t_best && ent < ent_best);
}
// Entity of a hit id (>= 0 triangle slot, <= -2 analytic entity, -1 none:
// above every entity).
__device__ __forceinline__ int32_t hit_entity(const PRT_GLOBAL prt_f4* tris4, int32_t id) {
  return id >= 0 ? __float_as_int(tris4[(size_t)id * 3].w) : (id <= -2 ? -2 - id : 0x7FFFFFFF);
}

// The analytic entities of a scene (at most PRT_LDS_ANALYTIC) as a block
// keeps them in LDS, spheres first.
struct AnalyticSlot {
  double p0[3], radius;  // sphere; uvplane: p0
  double u_axis[3], v_axis[3], u_len, v_len, u_max, v_max;  // uvplane
  double normal[3];      // uvplane: with the entity's sign
  int32_t ei, pad_;
};
// Copies them into slots (block-wide, a barrier follows); null if they are too
// many.
__device__ __forceinline__ const AnalyticSlot* load_analytic_slots(const Params& P, AnalyticSlot* slots) {
  if (P.n_analytic > PRT_LDS_ANALYTIC) return nullptr;
  if ((int)threadIdx.x < P.n_analytic) {
    AnalyticSlot& a = slots[threadIdx.x];
    a.ei = P.analytic[threadIdx.x];
    const DevEntity& e = P.ents[a.ei];
    const double sign = e.ninv < 0 ? -1.0 : 1.0;
    for (int j = 0; j < 3; ++j) {
      a.p0[j] = e.p0[j];
      a.u_axis[j] = e.u_axis[j];
      a.v_axis[j] = e.v_axis[j];
      a.normal[j] = e.normal[j] * sign;
    }
    a.radius = e.radius;
    a.u_len = e.u_len;
    a.v_len = e.v_len;
    // above these the plane coordinate's quotient by its length exceeds the
    // length whatever its rounding
    a.u_max = e.u_len * e.u_len * (1.0 + 1.0e-12);
    a.v_max = e.v_len * e.v_len * (1.0 + 1.0e-12);
  }
  return slots;
}
// uvplane_t of a slot: its answer and its t.  The quotients that bound the plane
// coordinates are formed only near the rectangle.
__device__ __forceinline__ bool uvplane_slot(const AnalyticSlot& e, d3 o, d3 d, double& t) {
  const d3 n2 = ld3(e.normal);
  const double dd = dot(d, n2), num = dot(ld3(e.p0) - o, n2);
  // behind the origin, whatever the quotient's rounding; NaN goes on
  if (fabs(dd) < PS_EPS14 || (num < 0.0 && dd > 0.0) || (num > 0.0 && dd < 0.0)) return false;
  t = num / dd;
  const d3 pos = d * t + o;
  if (t < PS_EPS) return false;
  const d3 rel = pos - ld3(e.p0);
  const double a = dot(rel, ld3(e.u_axis)), b = dot(rel, ld3(e.v_axis));
  if (a < -1.0e-200 || b < -1.0e-200 || a > e.u_max || b > e.v_max) return false;
  const double hu = a / e.u_len, hv = b / e.v_len;
  if (hu < 0 || hu > e.u_len) return false;
  if (hv < 0 || hv > e.v_len) return false;
  return true;
}

// The analytic part of a ray's hit: updates a closest hit (t, id) or tells
// whether an any hit lies below t.  slots: the scene's analytic entities in
// LDS, or null.  The tests are chains of dependent FP64 operations run by lanes
// that have just started a ray, so their records come from LDS instead of
// through three dependent global loads each, and the spheres are tested
// without branches, so that several chains overlap (nine spheres: 13,800 ->
// 6,400 cycles).
__device__ __forceinline__ bool analytic_hits(const Params& P, const AnalyticSlot* slots, d3 o, d3 d, bool any,
                                              double& t, int32_t& id) {
  bool blocked = false;
  int32_t e_best = 0x7FFFFFFF;
  auto meet = [&](bool hit, double tt, int32_t ei) {
    const bool near = hit && (any ? tt < t : nearer_hit(tt, ei, t, e_best));
    if (near && !any) {
      t = tt;
      id = -2 - ei;
      e_best = ei;
    }
    blocked |= near && any;
  };
  if (__builtin_expect(slots != nullptr, 1)) {
#pragma unroll 3
    for (int k = 0; k < P.n_spheres; ++k) {
      const AnalyticSlot& e = slots[k];
      double tt;
      const bool hit = sphere_root(ld3(e.p0), e.radius, o, d, tt);
      meet(hit, tt, e.ei);
    }
    for (int k = P.n_spheres; k < P.n_analytic; ++k) {
      const AnalyticSlot& e = slots[k];
      double tt;
      const bool hit = uvplane_slot(e, o, d, tt);
      meet(hit, tt, e.ei);
    }
  } else {
    // More of them than a block's LDS copy, or a batch of scenes.  Most of many
    // spheres are met by no ray of the wave: no square root without a lane that
    // needs it, and the records, which the host alone writes, by scalar loads (the
    // loop waited for vector loads and their addresses).  It runs at the lanes of a
    // refill alone, so without that it cost more than voted steps gave.  With 400
    // entities and 60k triangles, 2.5 M samples, ms before voted steps / with them /
    // with this loop: depth-synchronous 46.2 / 51.6 / 23.7, tile queue 48.6 / 52.9 /
    // 25.6; 2^20 rays against 400 entities 635 / 651 / 460 us; batch of 8 scenes 38.7
    // -> 37.2 ms.
    const PRT_CONST int32_t* list = (const PRT_CONST int32_t*)P.analytic;
    const PRT_CONST DevEntity* ents = (const PRT_CONST DevEntity*)P.ents;
#pragma unroll 2
    for (int k = 0; k < P.n_spheres; ++k) {
      const int32_t ei = list[k];
      const PRT_CONST DevEntity& e = ents[ei];
      const d3 p_o = mk(e.p0[0], e.p0[1], e.p0[2]) - o;
      const double b = dot(p_o, d);
      const double D4 = b * b - dot(p_o, p_o) + e.radius * e.radius;
      if (D4 < 0.0) continue;
      const double s = sqrt(D4);
      const double t1 = b - s, t2 = b + s;
      meet(!((t1 < PS_EPS) & (t2 < PS_EPS)), (t1 > PS_EPS) ? t1 : t2, ei);
    }
    for (int k = P.n_spheres; k < P.n_analytic; ++k) {
      const int32_t ei = list[k];
      double tt;
      const bool hit = uvplane_t(P.ents[ei], o, d, tt);
      meet(hit, tt, ei);
    }
  }
  return blocked;
}

// Every triangle a ray tests is one whose box the conservative culling
// leaves open (a box whose entry equals the best t stays open), so the
// closest hit is the one over all triangles, with the tie rule of
// nearer_hit.
// any (the same for every ray of a launch, or a lane's own): stop at the first
// hit below t_best instead.
template <class Stk>
__device__ __forceinline__ bool traverse_ww(const Params& P, bool any, d3 o, d3 d, double& t_best, int32_t& id_best,
                                            double& ub, double& vb, Stk& S, TravStats& ts) {
  if (P.n_nodes <= 0) return false;
  const float ox = (float)o.x, oy = (float)o.y, oz = (float)o.z;
  const float ix = ray_inverse(d.x), iy = ray_inverse(d.y), iz = ray_inverse(d.z);
  const float oix = ox * ix, oiy = oy * iy, oiz = oz * iz;
  const uint32_t rows = entry_rows(ix, iy, iz);
  float tb = t_best < 1.0e30 ? fup(t_best) : __builtin_inff();
  bool found = false;
  int sp = 0;
  const PRT_GLOBAL prt_f4* tris4 = (const PRT_GLOBAL prt_f4*)P.tris;
  int32_t e_best = any ? 0 : hit_entity(tris4, id_best);
  int32_t cur = 0, lf = 0;  // lf: parked leaf (< 0) or none (>= 0)
  while (true) {
    while ((uint32_t)cur < (uint32_t)PRT_TRAV_DONE) {
      if (cur == PRT_TRAV_POP) pop_two(S, sp, tb, cur, lf);
      if ((uint32_t)cur < (uint32_t)PRT_TRAV_POP) {
        uint64_t key[4];
        node_keys(S, P.nodes, P.n_nodes, cur, rows, ix, iy, iz, oix, oiy, oiz, tb, key);
        ts.nodes++;
        push_keys(S, sp, key);
        cur = key_hit(key[0]) ? (int32_t)(uint32_t)key[0] : next_entry(sp);
        if (cur < 0 && lf >= 0) {  // park the first leaf and keep walking
          lf = cur;
          cur = next_entry(sp);
        }
      }
      if (!__any(lf >= 0)) break;  // every lane still walking holds a leaf
    }
    while (lf < 0) {
      const uint32_t code = ~(uint32_t)lf;
      const uint32_t first = code & 0x07FFFFFFu;
      const uint32_t count = (code >> 27) + 1u;
      // triangle k + 1 is loaded before triangle k is tested
      const PRT_GLOBAL prt_f4* tr0 = tris4 + (size_t)first * 3;
      prt_f4 na = tr0[0], nb = tr0[1], nc = tr0[2];
      for (uint32_t k = 0; k < count; ++k) {
        const prt_f4 a = na, b = nb, c = nc;
        if (k + 1 < count) {
          const PRT_GLOBAL prt_f4* tr = tris4 + (size_t)(first + k + 1) * 3;
          na = tr[0];
          nb = tr[1];
          nc = tr[2];
        }
        ts.tris++;
        double t, u, v;
        if (mt_test(a, b, c, o, d, t, u, v) &&
            (any ? t < t_best : nearer_hit(t, __float_as_int(a.w), t_best, e_best))) {
          if (any) {
            id_best = (int32_t)(first + k);
            return true;
          }
          t_best = t;
          ub = u;
          vb = v;
          id_best = (int32_t)(first + k);
          e_best = __float_as_int(a.w);
          tb = fup(t);
          found = true;
        }
      }
      lf = cur;  // a second leaf met while walking is tested next
      if (cur < 0) cur = next_entry(sp);
    }
    if (cur == PRT_TRAV_DONE) break;
  }
  return found;
}

// One ray per lane (o: its already-nudged origin), closest and any hits side by
// side.  Without `any`: the closest hit over analytic entities and the BVH, t
// (entered as PS_INF) and id (>= 0: triangle slot; <= -2: analytic entity
// -2 - id; -1: miss).  With it: whether anything lies in (1e-6, t).  slots: the
// scene's analytic entities in LDS, or null.
template <class Stk>
__device__ __forceinline__ bool trace_lane(const Params& P, const AnalyticSlot* slots, d3 o, d3 d, bool any, double& t,
                                           int32_t& id, Stk& S, TravStats& tc, TravStats& tsh) {
  bool blocked = analytic_hits(P, slots, o, d, any, t, id);
  if (blocked) return true;
  TravStats ts{0, 0, 0};
  double u, v;
  blocked = traverse_ww(P, any, o, d, t, id, u, v, S, ts) && any;
  (any ? tsh : tc).nodes += ts.nodes;
  (any ? tsh : tc).tris += ts.tris;
  return blocked;
}

// *p, p the same for every lane, through the scalar cache (nothing may write it
// during the kernel).
__device__ __forceinline__ uint2 uniform_load(const uint2* p) {
  const uint64_t a = (uint64_t)p;
  const uint64_t au = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a);
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  const u2 v = *(const __attribute__((address_space(4))) u2*)au;
  return make_uint2(v.x, v.y);
}

// ------------------------------------------------ chunk claims
// The chunks [0, n_chunks) of a queue are split into PRT_FETCH_COUNTERS
// sub-ranges (fewer when the grid has fewer waves: every sub-range needs a
// wave that drains it), each with its own claim counter on its own 128-byte
// line, so no counter is shared by the whole device.  A wave draws from the
// sub-range wave % n_sub.
struct ClaimRange {
  uint32_t* counter;
  uint32_t b, e;
};
#ifndef PRT_XCD_CLAIMS
#define PRT_XCD_CLAIMS 0
#endif
__device__ __forceinline__ ClaimRange claim_range(uint32_t* fetch, uint32_t n_chunks) {
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  const uint32_t n_waves = (gridDim.x * blockDim.x) >> 6;
  const uint32_t n_sub = n_waves < (uint32_t)PRT_FETCH_COUNTERS ? n_waves : (uint32_t)PRT_FETCH_COUNTERS;
  uint32_t sub = wave % n_sub;
  if (PRT_XCD_CLAIMS && n_sub == (uint32_t)PRT_FETCH_COUNTERS && (gridDim.x & 7u) == 0) {
    // blocks go round-robin to the 8 XCDs: the waves of XCD x draw from
    // sub-ranges x * n_sub / 8 .. (x + 1) * n_sub / 8 - 1, one eighth of
    // the queue, so each XCD's L2 sees the rays of one part of the image
    const uint32_t per = n_sub / 8u, xcd = blockIdx.x & 7u;
    const uint32_t local = (blockIdx.x >> 3) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    sub = (uint32_t)__builtin_amdgcn_readfirstlane((int)(xcd * per + local % per));
  }
  ClaimRange r;
  r.counter = fetch + (size_t)sub * PRT_FETCH_STRIDE;
  r.b = (uint32_t)((uint64_t)sub * n_chunks / n_sub);
  r.e = (uint32_t)((uint64_t)(sub + 1) * n_chunks / n_sub);
  return r;
}
// Claims up to k chunks [c0, c1) of the wave's sub-range (one atomic);
// false once it is drained.  Every lane of the wave must call it.
__device__ __forceinline__ bool claim(const ClaimRange& r, uint32_t k, uint32_t& c0, uint32_t& c1) {
  uint32_t x = 0;
  if (lane_id() == 0) x = atomicAdd(r.counter, k);
  x = (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)x, 0, 64));
  c0 = r.b + x;
  if (c0 >= r.e) return false;
  c1 = min(c0 + k, r.e);
  return true;
}

// ------------------------------------------------ queue traversal with refill
//
// Closest or any hit for the rays that a source hands out, with lanes
// refilled as their rays finish: without refill a wave lives as long as its
// slowest ray and the other lanes idle meanwhile.  Each step of a wave is a
// node visit or a triangle test, whichever more of its lanes wait for (a node
// visit counting PRT_VOTE_NODE times), so that both run with most lanes
// active; a lane that has found a leaf keeps walking until it finds a second
// one, as in traverse_ww.  Once PRT_REFILL_MIN rays have finished they are
// handed over and their lanes take new ones.  A ray's hit is traverse_ww's.
//
// What bounds it: vector instructions, issued in 80 % of a SIMD's cycles, and
// so the lanes that share each of them.  Walking until every lane holds a
// leaf and then testing all leaves ran 23.8 lanes per node visit and 30.8 per
// triangle test (closest hits of the 82k-triangle box); the vote runs 43 and
// 38.  A refill is some 250 instructions at the refilled lanes only, plus the
// reads of the new rays, so it waits for half the wave: 38.0, 37.0, 36.4 ms a
// frame at 16, 24, 32 lanes (32, 24 and 40 are alike on other scenes).  The
// registers have to stay within 96 for five waves per SIMD: counts are kept per
// wave, and a hit's entity, needed only for equal distances, is read again.
// Frame of that box 41.5 -> 34.7 ms, with the analytic entities in LDS and the
// shorter tests; the field of 2.1 M triangles 72.8 -> 60.1 ms and the batch of
// eight scenes 54.4 -> 42.3 ms, whose tile queue had no refill.  Steps without a
// loop or a branch per child (pop_two, push_keys), keys sorted by 64-bit minima
// and scalar node bases: 34.4 -> 33.2, 59.6 -> 55.8 and 42.4 -> 41.1 ms.
//
// Source: next(base, n, idle) gives the wave's next rays base .. base + n - 1
// (n > 0; idle: no lane of the wave holds a ray), false when there are none
// now; params() the scene of the rays handed out last.  Every lane of the wave
// calls next together.
// Load(j, o, d, tmax): ray j's origin (before the 1e-6 nudge for a closest
// hit, already nudged for an any hit), direction and t bound.
// Done(j, t, id, blocked, o, d): the finished ray (closest hit t / id as
// trace_lane; any hit: blocked; o the nudged origin).
#ifndef PRT_REFILL_MIN
#define PRT_REFILL_MIN 32
#endif
#ifndef PRT_VOTE_NODE
#define PRT_VOTE_NODE 2
#endif
#ifndef PRT_FETCH_RAYS
#define PRT_FETCH_RAYS 128
#endif

// Chunks claimed from a chunk list (claim_range), PRT_FETCH_RAYS rays per
// atomic.
struct ChunkSource {
  const Params& P;
  const uint2* desc;
  ClaimRange cr;
  uint32_t c, c1;
  bool more;
  __device__ __forceinline__ ChunkSource(const Params& p, const ChunkList& cl, uint32_t* fetch)
      : P(p), desc(cl.desc), cr(claim_range(fetch, *cl.n)), c(0), c1(0), more(cr.b < cr.e) {}
  __device__ __forceinline__ const Params& params() const { return P; }
  __device__ __forceinline__ bool next(uint32_t& base, uint32_t& n, bool) {
    if (c >= c1) {
      if (!more || !claim(cr, (uint32_t)PRT_FETCH_RAYS / 64u, c, c1)) {
        more = false;
        return false;
      }
      more = c1 < cr.e;
    }
    const uint2 d = uniform_load(desc + c);
    ++c;
    base = d.x;
    n = d.y;
    return true;
  }
};

// An even share of the rays 0 .. n - 1 per wave of the grid, no counter.
struct ShareSource {
  const Params& P;
  uint32_t b, e;
  __device__ __forceinline__ ShareSource(const Params& p, uint32_t n) : P(p) {
    const uint64_t wave = (uint64_t)__builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const uint32_t n_waves = (gridDim.x * blockDim.x) >> 6;
    b = (uint32_t)(wave * n / n_waves);
    e = (uint32_t)((wave + 1) * n / n_waves);
  }
  __device__ __forceinline__ const Params& params() const { return P; }
  __device__ __forceinline__ bool next(uint32_t& base, uint32_t& n, bool) {
    if (b >= e) return false;
    base = b;
    n = e - b;
    b = e;
    return true;
  }
};

template <bool ANY, class Stk, class Source, class Load, class Done>
__device__ __forceinline__ void traverse_pool(Source& src, const AnalyticSlot* slots, Stk& S, TravStats& ts, Load&& load,
                                              Done&& done) {
  const uint32_t lane = lane_id();
  const uint64_t below = (1ull << lane) - 1ull;
  d3 o = mk(0.0, 0.0, 0.0), d = o;
  float ix = 0.0f, iy = 0.0f, iz = 0.0f, oix = 0.0f, oiy = 0.0f, oiz = 0.0f, tb = 0.0f;
  uint32_t rows = 0;
  double t_best = 0.0;
  int32_t id_best = -1, cur = PRT_TRAV_DONE, lf = 0;
  int sp = 0;
  uint32_t ri = 0;
  bool act = false, blocked = false;
  uint32_t base = 0, left = 0;  // wave-uniform: rays handed out and not yet started
  uint32_t n_nodes = 0, n_tris = 0, n_rays = 0;  // wave-uniform counts
  while (true) {
    // ---- idle lanes take new rays
    const uint64_t idle = __ballot(!act);
    const uint32_t n_idle = (uint32_t)__popcll(idle);
    if (n_idle >= (uint32_t)PRT_REFILL_MIN) {
      const uint32_t rank = (uint32_t)__popcll(idle & below);
      uint32_t got = 0;
      bool has = false;
      while (got < n_idle) {
        if (left == 0 && !src.next(base, left, n_idle == 64u && got == 0u)) break;
        const uint32_t take = min(n_idle - got, left);
        if (!act && rank >= got && rank < got + take) {
          ri = base + (rank - got);
          has = true;
        }
        base += take;
        left -= take;
        got += take;
      }
      if (got == 0u && n_idle == 64u) break;  // nothing running and nothing left
      if (has) {
        // analytic entities first
        const Params& P = src.params();
        act = true;
        load(ri, o, d, t_best);
        if (!ANY) o = o + d * 0.000001;
        id_best = -1;
        blocked = analytic_hits(P, slots, o, d, ANY, t_best, id_best);
        lf = 0;
        sp = 0;
        cur = PRT_TRAV_DONE;
        if (!blocked && P.n_nodes > 0) {
          ix = ray_inverse(d.x);
          iy = ray_inverse(d.y);
          iz = ray_inverse(d.z);
          oix = (float)o.x * ix;
          oiy = (float)o.y * iy;
          oiz = (float)o.z * iz;
          rows = entry_rows(ix, iy, iz);
          tb = t_best < 1.0e30 ? fup(t_best) : __builtin_inff();
          cur = 0;
        }
      }
    }
    const Params& P = src.params();
    const PRT_GLOBAL prt_f4* tris4 = (const PRT_GLOBAL prt_f4*)P.tris;
    const DevNode* nodes = P.nodes;
    const int32_t count = P.n_nodes;
    // ---- node and triangle steps until enough rays have finished
    while (true) {
      const bool walk = (uint32_t)cur < (uint32_t)PRT_TRAV_DONE;
      const uint32_t nw = (uint32_t)__popcll(__ballot(walk)), nl = (uint32_t)__popcll(__ballot(lf < 0));
      if (nw + nl == 0u) break;
      if (nw * (uint32_t)PRT_VOTE_NODE >= nl) {
        if (cur == PRT_TRAV_POP) pop_two(S, sp, tb, cur, lf);
        const bool visit = (uint32_t)cur < (uint32_t)PRT_TRAV_POP;
        n_nodes += (uint32_t)__popcll(__ballot(visit));
        if (visit) {
          uint64_t key[4];
          node_keys(S, nodes, count, cur, rows, ix, iy, iz, oix, oiy, oiz, tb, key);
          push_keys(S, sp, key);
          cur = key_hit(key[0]) ? (int32_t)(uint32_t)key[0] : next_entry(sp);
          if (cur < 0 && lf >= 0) {  // park the first leaf and keep walking
            lf = cur;
            cur = next_entry(sp);
          }
        }
      } else {
        n_tris += nl;
        if (lf < 0) {
          const uint32_t code = ~(uint32_t)lf;
          const uint32_t tri = code & 0x07FFFFFFu;
          const PRT_GLOBAL prt_f4* tr = tris4 + (size_t)tri * 3;
          const prt_f4 a = tr[0], b = tr[1], c = tr[2];
          double t, u, v;
          if (mt_test(a, b, c, o, d, t, u, v) &&
              (ANY ? t < t_best
                   : (t < t_best || (t == t_best && __float_as_int(a.w) < hit_entity(tris4, id_best))))) {
            if (ANY) {
              blocked = true;
            } else {
              t_best = t;
              id_best = (int32_t)tri;
              tb = fup(t);
            }
          }
          if (ANY && blocked) {
            lf = 0;
            cur = PRT_TRAV_DONE;
          } else if ((code >> 27) != 0u) {
            lf = (int32_t)~(code + 1u - (1u << 27));  // the leaf's next triangle
          } else {
            lf = cur < 0 ? cur : 0;  // a second leaf met while walking
            if (cur < 0) cur = next_entry(sp);
          }
        }
      }
      if ((uint32_t)__popcll(__ballot(act && cur == PRT_TRAV_DONE && lf >= 0)) >= (uint32_t)PRT_REFILL_MIN) break;
    }
    // ---- hand over finished rays
    const bool fin = act && cur == PRT_TRAV_DONE && lf >= 0;
    n_rays += (uint32_t)__popcll(__ballot(fin));
    if (fin) {
      done(ri, t_best, id_best, blocked, o, d);
      act = false;
    }
  }
  if (lane == 0) {
    ts.nodes += n_nodes;
    ts.tris += n_tris;
    ts.rays += n_rays;
  }
}

__device__ __forceinline__ void flush_stats(uint64_t* ctr, int idx_nodes, TravStats ts, int idx_rays = -1) {
  const uint64_t n = wave_sum_u32(ts.nodes), t = wave_sum_u32(ts.tris);
  const uint64_t r = idx_rays >= 0 ? wave_sum_u32(ts.rays) : 0;
  if (lane_id() == 0) {
    ctr_add(ctr, idx_nodes, n);
    ctr_add(ctr, idx_nodes + 1, t);
    ctr_add(ctr, idx_rays, r);
  }
}
