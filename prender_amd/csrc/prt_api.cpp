// prt_api.cpp — the C ABI of include/prt.h: scene upload, closest-hit
// queries and the wavefront render loop on one HIP stream.
//
// Scene semantics follow SceneEnv::Load (proj/scene_env.h:357-1990): the
// light list holds the light-material spheres and uvplanes in entity order,
// sorted by power = area * |emission| descending (light.h:95-99,
// scene_env.h:1567-1719); the camera is CameraScreenPram (render.h:100-146)
// after SceneEnv's CAMERA_ANGLE handling and normalisation
// (scene_env.h:1881-1886, 1920).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/prt.h"
#include "bvh.h"
#include "prt_mlt.h"
#include "prt_device.h"
#include "prt_internal.h"
#include "prt_kernels.h"
#include "prt_stream.h"

// 256-thread blocks per CU of the traversal grids
#ifndef PRT_TRAV_BLOCKS_PER_CU
#define PRT_TRAV_BLOCKS_PER_CU 8
#endif
// camera samples per depth-synchronous batch: 2^PRT_BATCH_LOG2 (half with
// glass).  2^24 holds a 512x512x64 frame whole: one drain of the depth tail
// per frame instead of eight (cfg2 216 -> 294 M samples/s against 2^21), for
// about 7.5 GB of queues, accumulators and hit records.
#ifndef PRT_BATCH_LOG2
#define PRT_BATCH_LOG2 24
#endif
// Per-scene renders of NEE scenes: where a depth's shadow rays are traced.
// 0: on the main stream after the depth's NEE; 1: on a second stream, while
// the next depth's extension rays are traced; 2: NEE and shadow rays both on
// the second stream, after the shade that wrote the NEE input; 3: the NEE on
// the main stream into one of two shadow queues, and its shadow rays on the
// second stream once the next depth's extension rays are done, so that they
// share the chip with that depth's shade and NEE (queue-streaming kernels)
// rather than with another traversal.
#ifndef PRT_OVERLAP_SHADOW
#define PRT_OVERLAP_SHADOW 3
#endif

// Shadow-ray blocks per CU.  The traversal kernels' LDS stacks allow 4
// resident blocks per CU; 3 leave room for the shade and NEE blocks that run
// beside the shadow rays in the alternating schedule (cfg2 348 -> 353 M
// samples/s; 2 let the shadow rays run into the next closest-hit launch).
#ifndef PRT_SHADOW_BLOCKS_PER_CU
#define PRT_SHADOW_BLOCKS_PER_CU 3
#endif
// the traversal-stack overflow areas hold one slot per thread of the
// closest-hit grid; a larger shadow grid would share slots between threads
static_assert(PRT_SHADOW_BLOCKS_PER_CU <= PRT_TRAV_BLOCKS_PER_CU,
              "shadow traversal grid must not exceed the closest-hit grid");

namespace prt {

thread_local std::string g_err;

int dev_alloc(DevBuf& b, size_t bytes) {
  if (b.bytes >= bytes && b.p) return PRT_OK;
  b.release();
  if (bytes == 0) return PRT_OK;
  hipError_t e = hipMalloc(&b.p, bytes);
  if (e != hipSuccess) {
    b.p = nullptr;
    (void)hipGetLastError();  // not left for the next launch's error check
    return fail(PRT_E_NOMEM, std::string("hipMalloc of ") + std::to_string(bytes) + " bytes: " + hipGetErrorString(e));
  }
  b.bytes = bytes;
  return PRT_OK;
}

namespace {
constexpr int kMaxPoolDevices = 64;
std::mutex g_pool_mu;
DevicePool* g_pools[kMaxPoolDevices] = {};
}  // namespace

DevicePool* acquire_device_pool(int device) {
  if (device < 0 || device >= kMaxPoolDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_pool_mu);
  if (!g_pools[device]) g_pools[device] = new (std::nothrow) DevicePool();
  if (g_pools[device]) g_pools[device]->scenes++;
  return g_pools[device];
}

void release_device_pool(int device) {
  if (device < 0 || device >= kMaxPoolDevices) return;
  std::lock_guard<std::mutex> lk(g_pool_mu);
  DevicePool* p = g_pools[device];
  if (!p || --p->scenes > 0) return;
  // the last handle on the device is gone: free the memory (the pool object,
  // whose lock another thread could still name, stays)
  std::lock_guard<std::recursive_mutex> l2(p->m);
  p->ws.release();
  release_stream_workspace(p->sws);
  p->sws = nullptr;
}

void Workspace::release() {
  for (auto& a : q)
    for (auto& b : a) b.release();
  hit_t.release();
  hit_id.release();
  for (auto& b : sq) b.release();
  for (auto& b : sq2) b.release();
  for (auto& b : desc) b.release();
  slabs.release();
  accum.release();
  accum2.release();
  for (auto& b : recs) b.release();
  counts.release();
  fetch.release();
  ctr.release();
  pool.release();
  if (h_counts) (void)hipHostFree(h_counts);
  h_counts = nullptr;
  batch_samples = queue_cap = shadow_cap = 0;
}

static const size_t kRayColBytes[RAYQ_COLS] = {16, 16, 16, 16, 16, 16};
static const size_t kShadowColBytes[SHADOWQ_COLS] = {16, 16, 16, 8, 16, 4};
size_t ray_entry_bytes() {
  size_t b = 0;
  for (size_t v : kRayColBytes) b += v;
  return b;
}
size_t shadow_entry_bytes() {
  size_t b = 0;
  for (size_t v : kShadowColBytes) b += v;
  return b;
}

int alloc_ray_queue(DevBuf* cols, int64_t cap) {
  const size_t* dsz = kRayColBytes;
  for (int k = 0; k < RAYQ_COLS; ++k) {
    const int rc = dev_alloc(cols[k], (size_t)cap * dsz[k]);
    if (rc) return rc;
  }
  return PRT_OK;
}

int alloc_shadow_queue(DevBuf* cols, int64_t cap) {
  const size_t* ssz = kShadowColBytes;
  for (int k = 0; k < SHADOWQ_COLS; ++k) {
    const int rc = dev_alloc(cols[k], (size_t)cap * ssz[k]);
    if (rc) return rc;
  }
  return PRT_OK;
}

RayQ ray_queue(DevBuf* b, int64_t cap) {
  RayQ q;
  q.a = (double2*)b[0].p; q.b = (double2*)b[1].p; q.c = (double2*)b[2].p;
  q.t = (float4*)b[3].p;
  q.n = (float4*)b[4].p;
  q.p = (float4*)b[5].p;
  q.cap = (uint32_t)cap;
  return q;
}

ShadowQ shadow_queue(DevBuf* b, int64_t cap) {
  ShadowQ q;
  q.a = (double2*)b[0].p; q.b = (double2*)b[1].p; q.c = (double2*)b[2].p;
  q.tmax = (double*)b[3].p;
  q.l = (float4*)b[4].p;
  q.light = (int32_t*)b[5].p;
  q.cap = (uint32_t)cap;
  return q;
}

}  // namespace prt

using namespace prt;

namespace {

// Host Vector3d with the reference's operation order (vector3d.h).
struct V3 {
  double x, y, z;
};
V3 mk(double a, double b, double c) { return V3{a, b, c}; }
V3 operator+(V3 a, V3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
V3 operator-(V3 a, V3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
V3 operator*(V3 a, double s) { return mk(a.x * s, a.y * s, a.z * s); }
double dot(V3 a, V3 b) { return (a.x * b.x + a.z * b.z) + a.y * b.y; }
double length(V3 a) { return std::sqrt((a.x * a.x + a.z * a.z) + a.y * a.y); }
V3 normalize(V3 a) { return a * (1.0 / length(a)); }
V3 cross(V3 a, V3 b) { return mk((a.y * b.z) - (a.z * b.y), (a.z * b.x) - (a.x * b.z), (a.x * b.y) - (a.y * b.x)); }
V3 from(const double* p) { return mk(p[0], p[1], p[2]); }
void put(double* d, V3 v) { d[0] = v.x; d[1] = v.y; d[2] = v.z; }

}  // namespace

extern "C" {

int prt_abi_version(void) { return PRT_ABI_VERSION; }
const char* prt_last_error(void) { return g_err.c_str(); }

int prt_device_info(char* name, int name_len, int* cu_count, int* arch_major, int* arch_minor) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(PRT_E_NODEVICE, hipGetErrorString(e));
  hipDeviceProp_t p;
  HIPCHK(hipGetDeviceProperties(&p, dev));
  if (name && name_len > 0) {
    std::snprintf(name, name_len, "%s", p.gcnArchName);
  }
  if (cu_count) *cu_count = p.multiProcessorCount;
  if (arch_major) *arch_major = p.major;
  if (arch_minor) *arch_minor = p.minor;
  return PRT_OK;
}

void prt_scene_destroy(prt_scene* s) {
  if (!s) return;
  (void)hipSetDevice(s->device);
  if (s->stream) (void)hipStreamSynchronize(s->stream);
  if (s->stream2) (void)hipStreamSynchronize(s->stream2);
  s->nodes.release(); s->tris.release(); s->tri_nrm.release(); s->tri_alb.release();
  s->ents.release(); s->mats.release(); s->analytic.release(); s->lights.release(); s->ovf.release();
  if (s->pool) release_device_pool(s->device);
  s->pool = nullptr;
  s->out_rgb.release();
  s->out_var.release();
  s->d_slot_of_tri.release();
  s->grad_buf.release();
  s->tri_alb_rr.release();
  s->mlt.release();
  s->timer_events.release();
  for (hipEvent_t e : s->ev_nee)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : s->ev_sh)
    if (e) (void)hipEventDestroy(e);
  if (s->ev_shadow) (void)hipEventDestroy(s->ev_shadow);
  if (s->ev_shade) (void)hipEventDestroy(s->ev_shade);
  if (s->stream2) (void)hipStreamDestroy(s->stream2);
  if (s->stream) (void)hipStreamDestroy(s->stream);
  delete s;
}

static int scene_build(prt_scene* s, const prt_scene_desc* d) {
  if (!d) return fail(PRT_E_INVALID, "null scene description");
  const prt_camera& cam = d->camera;
  const prt_sampling& smp = d->sampling;
  if (cam.image_width <= 0 || cam.image_height <= 0) return fail(PRT_E_INVALID, "image size must be positive");
  if (smp.samples <= 0 || smp.supersamples <= 0) return fail(PRT_E_INVALID, "samples and supersamples must be positive");
  if ((int64_t)smp.samples * smp.supersamples * smp.supersamples > (1 << 20))
    return fail(PRT_E_INVALID, "samples per pixel above 2^20");
  if (d->n_materials <= 0 || !d->materials) return fail(PRT_E_INVALID, "no materials");
  if ((uint32_t)d->n_materials > TRI_SHADE_MAT_MASK + 1u) return fail(PRT_E_INVALID, "more than 2^24 materials");
  if (d->n_entities < 0 || (d->n_entities > 0 && !d->entities)) return fail(PRT_E_INVALID, "bad entity list");

  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(PRT_E_NODEVICE, hipGetErrorString(e));
  hipDeviceProp_t prop;
  HIPCHK(hipGetDeviceProperties(&prop, dev));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(PRT_E_NODEVICE, std::string("libprt is built for gfx950, device is ") + prop.gcnArchName);
  s->device = dev;
  s->cu_count = prop.multiProcessorCount;
  s->pool = acquire_device_pool(dev);
  if (!s->pool) return fail(PRT_E_NOMEM, "no render memory pool for this device");
  HIPCHK(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
  HIPCHK(hipStreamCreateWithFlags(&s->stream2, hipStreamNonBlocking));
  HIPCHK(hipEventCreateWithFlags(&s->ev_nee[0], hipEventDisableTiming));
  HIPCHK(hipEventCreateWithFlags(&s->ev_nee[1], hipEventDisableTiming));
  HIPCHK(hipEventCreateWithFlags(&s->ev_shadow, hipEventDisableTiming));
  HIPCHK(hipEventCreateWithFlags(&s->ev_shade, hipEventDisableTiming));
  HIPCHK(hipEventCreateWithFlags(&s->ev_sh[0], hipEventDisableTiming));
  HIPCHK(hipEventCreateWithFlags(&s->ev_sh[1], hipEventDisableTiming));

  // materials (Material::isLight, material.h:195-210)
  s->h_mats.resize(d->n_materials);
  for (int i = 0; i < d->n_materials; ++i) {
    const prt_material& pm = d->materials[i];
    DevMaterial& m = s->h_mats[i];
    std::memcpy(m.color, pm.color, sizeof(m.color));
    std::memcpy(m.emission, pm.emission, sizeof(m.emission));
    m.roughness = pm.roughness;
    m.ior = pm.refractive_index;
    m.type = pm.reflection_type;
    if (m.type < PRT_REFLECTION_DIFFUSE || m.type > PRT_REFLECTION_REFRACTION)
      return fail(PRT_E_UNSUPPORTED, "reflection_type outside diffuse/specular/refraction");
    m.is_light = (m.type == PRT_REFLECTION_DIFFUSE && length(from(pm.color)) < 0.001 &&
                  length(from(pm.emission)) > 0.001) ? 1 : 0;
    if (m.type == PRT_REFLECTION_REFRACTION) s->has_glass = true;
  }

  // entities, triangles
  std::vector<int32_t> analytic;
  std::vector<float> v9;         // per input triangle: v0 v1 v2
  std::vector<int32_t> t_ent, t_face;
  std::vector<float> t_nrm, t_alb;
  bool any_albedo = false;
  s->h_ents.resize(d->n_entities);
  s->ent_first_tri.assign(d->n_entities, -1);
  s->ent_n_tris.assign(d->n_entities, 0);
  for (int i = 0; i < d->n_entities; ++i) {
    const prt_entity& pe = d->entities[i];
    DevEntity& de = s->h_ents[i];
    std::memset(&de, 0, sizeof(de));
    de.type = pe.type;
    de.material = pe.material;
    de.ninv = pe.normal_vector_inverse < 0 ? -1 : 1;
    if (pe.material < 0 || pe.material >= d->n_materials) return fail(PRT_E_INVALID, "entity material out of range");
    de.light = s->h_mats[pe.material].is_light;
    if (pe.type == PRT_ENTITY_SPHERE) {
      if (!(pe.radius > 0)) return fail(PRT_E_INVALID, "sphere radius must be positive");
      std::memcpy(de.p0, pe.p0, sizeof(de.p0));
      de.radius = pe.radius;
      de.area = (12.5663706143591729538505735331180115 * pe.radius * pe.radius);  // sphere.h:23-27
      analytic.push_back(i);
    } else if (pe.type == PRT_ENTITY_UVPLANE) {
      // UVPlane ctor + CalcArea, plane.h:143-166
      const V3 U = from(pe.p1), V = from(pe.p2);
      de.u_len = length(U);
      de.v_len = length(V);
      if (!(de.u_len > 0) || !(de.v_len > 0)) return fail(PRT_E_INVALID, "uvplane axes must be non-zero");
      const V3 ua = normalize(U), va = normalize(V);
      put(de.u_axis, ua);
      put(de.v_axis, va);
      put(de.normal, normalize(cross(ua, va)));
      std::memcpy(de.p0, pe.p0, sizeof(de.p0));
      de.area = length(ua * de.u_len) * length(va * de.v_len) * (1.0 - std::pow(dot(ua, va), 2.0));
      analytic.push_back(i);
    } else if (pe.type == PRT_ENTITY_POLYGON) {
      if (pe.n_faces <= 0 || pe.n_vertices <= 0 || !pe.vertices || !pe.indices)
        return fail(PRT_E_INVALID, "polygon entity without vertices or faces");
      if (de.light && smp.next_event_estimation)
        return fail(PRT_E_UNSUPPORTED, "POLYGON lights cannot be sampled by NEE (directLight_radiance.h:329)");
      de.has_albedo = pe.face_albedo ? 1 : 0;
      any_albedo |= (pe.face_albedo != nullptr);
      s->ent_first_tri[i] = (int64_t)t_ent.size();
      s->ent_n_tris[i] = pe.n_faces;
      for (int64_t f = 0; f < pe.n_faces; ++f) {
        const int32_t* ix = pe.indices + 3 * f;
        for (int k = 0; k < 3; ++k)
          if (ix[k] < 0 || ix[k] >= pe.n_vertices) return fail(PRT_E_INVALID, "triangle index out of range");
        const float* a = pe.vertices + 3 * (size_t)ix[0];
        const float* b = pe.vertices + 3 * (size_t)ix[1];
        const float* c = pe.vertices + 3 * (size_t)ix[2];
        v9.insert(v9.end(), {a[0], a[1], a[2], b[0], b[1], b[2], c[0], c[1], c[2]});
        t_ent.push_back(i);
        t_face.push_back((int32_t)f);
        // f32 face normal, ObjLoader.cpp:577-602 + 688-698
        const float dx1 = b[0] - a[0], dy1 = b[1] - a[1], dz1 = b[2] - a[2];
        const float dx2 = c[0] - a[0], dy2 = c[1] - a[1], dz2 = c[2] - a[2];
        float nx = dy1 * dz2 - dz1 * dy2;
        float ny = dz1 * dx2 - dx1 * dz2;
        float nz = dx1 * dy2 - dy1 * dx2;
        const float len = std::sqrt(nx * nx + ny * ny + nz * nz);
        if (len != 0.0f) { nx /= len; ny /= len; nz /= len; }
        t_nrm.insert(t_nrm.end(), {nx, ny, nz});
        if (pe.face_albedo) {
          const float* al = pe.face_albedo + 3 * f;
          t_alb.insert(t_alb.end(), {al[0], al[1], al[2]});
        } else {
          t_alb.insert(t_alb.end(), {0.0f, 0.0f, 0.0f});
        }
      }
    } else {
      return fail(PRT_E_UNSUPPORTED, "entity type outside sphere/uvplane/polygon");
    }
  }
  s->n_tris = (int64_t)t_ent.size();
  // spheres, then uvplanes (of equal hits the lowest entity index wins in any
  // order, nearer_hit)
  const size_t n_spheres = std::stable_partition(analytic.begin(), analytic.end(),
                                                 [&](int32_t i) { return s->h_ents[i].type == PRT_ENTITY_SPHERE; }) -
                           analytic.begin();

  // lights: light-material spheres and uvplanes, power-descending (stable)
  struct L { int32_t ent; double power; };
  std::vector<L> ls;
  for (int i = 0; i < d->n_entities; ++i) {
    const DevEntity& de = s->h_ents[i];
    if (!de.light || de.type == PRT_ENTITY_POLYGON) continue;
    ls.push_back(L{i, de.area * length(from(s->h_mats[de.material].emission))});
  }
  std::stable_sort(ls.begin(), ls.end(), [](const L& a, const L& b) { return a.power > b.power; });
  s->h_lights.clear();
  for (const L& l : ls) s->h_lights.push_back(l.ent);

  // BVH over all triangles, leaf-ordered triangle records
  BvhOutput bo;
  if (s->n_tris > 0) {
    BvhInput bi{v9.data(), s->n_tris, 0};
    const char* err = nullptr;
    if (!prt_build_bvh(bi, bo, &err)) return fail(PRT_E_UNSUPPORTED, err ? err : "bvh build failed");
  }
  s->bvh_depth = bo.depth;
  s->n_top = bo.n_top;
  s->bvh_ms = bo.build_ms;
  std::vector<float> tri4((size_t)s->n_tris * 12);
  std::vector<float> nrm((size_t)s->n_tris * 4), alb(any_albedo ? (size_t)s->n_tris * 3 : 0);
  s->slot_of_tri.assign(s->n_tris, 0);
  for (int64_t slot = 0; slot < s->n_tris; ++slot) {
    const uint32_t t = bo.order[slot];
    s->slot_of_tri[t] = (uint32_t)slot;
    float* r = &tri4[12 * slot];
    const float* v = &v9[9 * (size_t)t];
    int32_t ent = t_ent[t], face = t_face[t];
    const DevEntity& de = s->h_ents[ent];
    const uint32_t shade = ((uint32_t)de.material & TRI_SHADE_MAT_MASK) | (de.ninv < 0 ? TRI_SHADE_NINV : 0u) |
                           (de.light ? TRI_SHADE_LIGHT : 0u) | (de.has_albedo ? TRI_SHADE_ALBEDO : 0u);
    r[0] = v[0]; r[1] = v[1]; r[2] = v[2]; std::memcpy(&r[3], &ent, 4);
    r[4] = v[3]; r[5] = v[4]; r[6] = v[5]; std::memcpy(&r[7], &face, 4);
    r[8] = v[6]; r[9] = v[7]; r[10] = v[8]; r[11] = 0.0f;
    for (int k = 0; k < 3; ++k) nrm[4 * slot + k] = t_nrm[3 * (size_t)t + k];
    std::memcpy(&nrm[4 * slot + 3], &shade, 4);
    if (any_albedo)
      for (int k = 0; k < 3; ++k) alb[3 * slot + k] = t_alb[3 * (size_t)t + k];
  }

  hipStream_t st = s->stream;
  int rc;
  if ((rc = dev_upload(s->nodes, bo.nodes, st))) return rc;
  if ((rc = dev_upload(s->tris, tri4, st))) return rc;
  if ((rc = dev_upload(s->tri_nrm, nrm, st))) return rc;
  if (any_albedo && (rc = dev_upload(s->tri_alb, alb, st))) return rc;
  if ((rc = dev_upload(s->ents, s->h_ents, st))) return rc;
  if ((rc = dev_upload(s->mats, s->h_mats, st))) return rc;
  if ((rc = dev_upload(s->analytic, analytic, st))) return rc;
  if ((rc = dev_upload(s->lights, s->h_lights, st))) return rc;
  if (any_albedo && (rc = dev_upload(s->d_slot_of_tri, s->slot_of_tri, st))) return rc;
  // traversal stack overflow: one area per thread of the largest grid
  s->max_trav_blocks = std::max(1, s->cu_count) * PRT_TRAV_BLOCKS_PER_CU;
  const int64_t ovf_threads = (int64_t)s->max_trav_blocks * 256;
  const int ovf_words = ovf_words_for(s->bvh_depth);
  if ((rc = dev_alloc(s->ovf, (size_t)PRT_OVF_REGIONS * ovf_threads * ovf_words * sizeof(uint32_t))))
    return rc;
  HIPCHK(hipStreamSynchronize(st));

  // Params: camera (CameraScreenPram, render.h:100-146; scene_env.h:1881-1886, 1920)
  Params& P = s->P;
  std::memset(&P, 0, sizeof(P));
  V3 cpos = from(cam.camera_position), cdir = normalize(from(cam.camera_dir)), cup = from(cam.camera_up);
  double wsw = cam.world_screen_width, wsh = cam.world_screen_height;
  if (cam.camera_angle > 0.0) {
    wsw = 2.0 * cam.world_screen_dist * std::tan(cam.camera_angle * (3.14159265358979323846264338327950288 / 180.0) / 2.0);
    wsh = wsw;
  }
  const double PI = 3.14159265358979323846264338327950288;
  double cam_phi = std::atan2(cdir.y, cdir.x);
  if (cam_phi < 0.0) cam_phi += 2.0 * PI;
  if (std::fabs(cam_phi - PI) < 1.0e-6 || cam_phi < 1.0e-6 || std::fabs(cam_phi - 2.0 * PI) < 1.0e-6) {
    cdir.y += 1.0e-6;
    const double len = std::sqrt(cdir.x * cdir.x + cdir.y * cdir.y + cdir.z * cdir.z);
    cdir.x /= len; cdir.y /= len; cdir.z /= len;
  }
  const double screen_width = wsw * cam.image_width / cam.image_height;
  const double screen_height = wsh;
  const V3 sx = normalize(cross(cdir, cup)) * screen_width;
  const V3 sy = normalize(cross(sx, cdir)) * screen_height;
  put(P.cam_pos, cpos);
  put(P.screen_x, sx);
  put(P.screen_y, sy);
  put(P.center, cpos + cdir * cam.world_screen_dist);
  P.iw = 1.0 / cam.image_width;
  P.ih = 1.0 / cam.image_height;
  P.W = cam.image_width;
  P.H = cam.image_height;
  P.SS = smp.supersamples;
  P.samples = smp.samples;
  P.spp = smp.samples * smp.supersamples * smp.supersamples;
  P.depth = smp.depth;
  P.depth_limit = smp.depth_limit;
  P.nee = smp.next_event_estimation ? 1 : 0;
  P.max_vertices = 128;
  P.n_lights = (int32_t)s->h_lights.size();
  P.n_materials = (int32_t)s->h_mats.size();
  P.n_analytic = (int32_t)analytic.size();
  P.n_spheres = (int32_t)n_spheres;
  P.n_nodes = (int32_t)bo.nodes.size();
  P.smp = 1.0 / smp.samples / (smp.supersamples * smp.supersamples);
  P.sensor_response = smp.sensor_response;
  P.cutoff = (float)smp.luminance_cutoff;  // a float in SceneEnv (scene_env.h:221)
  std::memcpy(P.background, smp.background_color, sizeof(P.background));
  std::memcpy(P.env_light, smp.environment_light, sizeof(P.env_light));
  P.nodes = (const DevNode*)s->nodes.p;
  P.tris = (const float*)s->tris.p;
  P.tri_nrm = (const float*)s->tri_nrm.p;
  P.tri_alb = any_albedo ? (const float*)s->tri_alb.p : nullptr;
  P.ents = (const DevEntity*)s->ents.p;
  P.mats = (const DevMaterial*)s->mats.p;
  P.analytic = (const int32_t*)s->analytic.p;
  P.lights = (const int32_t*)s->lights.p;
  P.stack_ovf = (uint32_t*)s->ovf.p;
  P.ovf_threads = (int32_t)ovf_threads;
  P.ovf_words = ovf_words;
  P.n_top = P.n_nodes > 0 ? std::min(bo.n_top, PRT_TOP_NODES) : 0;
  P.n_wide = P.n_nodes > 0 ? std::min(bo.n_wide, PRT_WIDE_NODES) : 0;
  P.n_tris = (int32_t)s->n_tris;
  return PRT_OK;
}

prt_scene* prt_scene_create(const prt_scene_desc* desc) {
  prt_scene* s = new (std::nothrow) prt_scene();
  if (!s) { g_err = "out of host memory"; return nullptr; }
  int rc;
  try {
    rc = scene_build(s, desc);
  } catch (const std::bad_alloc&) {
    rc = fail(PRT_E_NOMEM, "out of host memory while building the scene");
  }
  if (rc != PRT_OK) {
    std::string keep = g_err;
    prt_scene_destroy(s);
    g_err = keep;
    return nullptr;
  }
  return s;
}

int prt_scene_info(const prt_scene* s, int64_t* n_nodes, int64_t* n_tris, int64_t* n_lights, int64_t* bvh_bytes) {
  if (!s) return fail(PRT_E_INVALID, "null scene");
  if (n_nodes) *n_nodes = s->P.n_nodes;
  if (n_tris) *n_tris = s->n_tris;
  if (n_lights) *n_lights = (int64_t)s->h_lights.size();
  if (bvh_bytes) *bvh_bytes = (int64_t)s->P.n_nodes * (int64_t)sizeof(DevNode) + s->n_tris * 48;
  return PRT_OK;
}

extern "C++" void prt::fill_stats(prt_stats* st, const uint64_t* c) {
  st->node_visits += c[CTR_NODES] + c[CTR_SNODES];
  st->tri_tests += c[CTR_TRIS] + c[CTR_STRIS];
  st->shadow_node_visits += c[CTR_SNODES];
  st->shadow_tri_tests += c[CTR_STRIS];
  st->pickup_hits += c[CTR_PICKUP];
  st->truncated_paths += c[CTR_TRUNC];
}

extern "C++" int prt::check_traced(const uint64_t* c, uint64_t primary_rays) {
  if (c[CTR_DROP] != 0) return fail(PRT_E_INVALID, "ray queue overflow (" + std::to_string(c[CTR_DROP]) + " rays)");
  if (c[CTR_QUEUED] != primary_rays + c[CTR_EXT])
    return fail(PRT_E_INTERNAL, std::to_string(c[CTR_QUEUED]) + " rays came from " + std::to_string(primary_rays) +
                                    " camera rays and " + std::to_string(c[CTR_EXT]) + " children");
  if (c[CTR_TRACED] != c[CTR_QUEUED] || c[CTR_STRACED] != c[CTR_SHADOW])
    return fail(PRT_E_INTERNAL, "traversal finished " + std::to_string(c[CTR_TRACED]) + " of " +
                                    std::to_string(c[CTR_QUEUED]) + " rays and " +
                                    std::to_string(c[CTR_STRACED]) + " of " + std::to_string(c[CTR_SHADOW]) +
                                    " shadow rays");
  return PRT_OK;
}

static int trace_device(prt_scene* s, const prt_ray* d_rays, int64_t n, prt_hit* d_hits, prt_stats* stats) {
  HIPCHK(hipSetDevice(s->device));
  std::lock_guard<std::recursive_mutex> pool_lock(s->pool->m);
  int rc;
  if ((rc = dev_alloc(s->pool->ws.ctr, CTR_WORDS * sizeof(uint64_t)))) return rc;
  HIPCHK(launch_fill_u64((uint64_t*)s->pool->ws.ctr.p, 0ull, CTR_WORDS, s->stream));
  ScopedEvent e0, e1;
  HIPCHK(hipEventCreate(&e0.e));
  HIPCHK(hipEventCreate(&e1.e));
  HIPCHK(hipEventRecord(e0.e, s->stream));
  if (n > 0)
    HIPCHK(launch_trace(s->P, (const prt_ray_dev*)d_rays, n, (prt_hit_dev*)d_hits, (uint64_t*)s->pool->ws.ctr.p,
                        std::max(1, s->cu_count), s->stream));
  HIPCHK(hipEventRecord(e1.e, s->stream));
  uint64_t raw[CTR_WORDS], c[CTR_COUNT];
  HIPCHK(hipMemcpyAsync(raw, s->pool->ws.ctr.p, sizeof(raw), hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  sum_counters(raw, c);
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, e0.e, e1.e));
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    fill_stats(stats, c);
    stats->extension_rays = (uint64_t)n;
    stats->ms_total = ms;
    stats->ms_extend = ms;
    stats->launches_extend = 1;
    stats->bytes_extend = 128 * stats->node_visits + 48 * stats->tri_tests + 48 * (uint64_t)n;
    stats->bytes_algorithmic = stats->bytes_extend;
  }
  return PRT_OK;
}

int prt_trace_closest_device(prt_scene* s, const prt_ray* d_rays, int64_t n, prt_hit* d_hits, prt_stats* stats) {
  if (!s || n < 0 || (n > 0 && (!d_rays || !d_hits))) return fail(PRT_E_INVALID, "bad arguments");
  return trace_device(s, d_rays, n, d_hits, stats);
}

// The same traversal as prt_trace_closest_device with nothing allocated in
// the call: the counters are the library's per-GPU scratch array (cleared by
// a fill kernel, so every call starts from zero whatever the last call left)
// and no timing events are created.  Calls that overlap on one GPU share
// those counters (their hits stay exact; their counts mix).
int prt_trace_closest_device_noalloc(prt_scene* s, const prt_ray* d_rays, int64_t n, prt_hit* d_hits,
                                     prt_stats* stats) {
  if (!s || n < 0 || (n > 0 && (!d_rays || !d_hits))) return fail(PRT_E_INVALID, "bad arguments");
  HIPCHK(hipSetDevice(s->device));
  uint64_t* ctr = nullptr;
  HIPCHK(noalloc_scratch(s->device, &ctr));
  HIPCHK(launch_fill_u64(ctr, 0, CTR_WORDS, s->stream));
  if (n > 0)
    HIPCHK(launch_trace(s->P, (const prt_ray_dev*)d_rays, n, (prt_hit_dev*)d_hits, ctr,
                        std::max(1, s->cu_count), s->stream));
  uint64_t raw[CTR_WORDS], c[CTR_COUNT];
  HIPCHK(hipMemcpyAsync(raw, ctr, sizeof(raw), hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  sum_counters(raw, c);
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    fill_stats(stats, c);
    stats->extension_rays = (uint64_t)n;
    stats->launches_extend = n > 0 ? 1 : 0;
    stats->bytes_extend = 128 * stats->node_visits + 48 * stats->tri_tests + 48 * (uint64_t)n;
    stats->bytes_algorithmic = stats->bytes_extend;
  }
  return PRT_OK;
}

int prt_trace_closest(prt_scene* s, const prt_ray* rays, int64_t n, prt_hit* hits, prt_stats* stats) {
  if (!s || n < 0 || (n > 0 && (!rays || !hits))) return fail(PRT_E_INVALID, "bad arguments");
  HIPCHK(hipSetDevice(s->device));
  void *dr = nullptr, *dh = nullptr;
  if (n > 0) {
    HIPCHK(hipMalloc(&dr, (size_t)n * sizeof(prt_ray)));
    hipError_t e = hipMalloc(&dh, (size_t)n * sizeof(prt_hit));
    if (e != hipSuccess) { (void)hipFree(dr); return fail(PRT_E_NOMEM, hipGetErrorString(e)); }
    e = hipMemcpyAsync(dr, rays, (size_t)n * sizeof(prt_ray), hipMemcpyHostToDevice, s->stream);
    if (e != hipSuccess) { (void)hipFree(dr); (void)hipFree(dh); return fail(PRT_E_HIP, hipGetErrorString(e)); }
  }
  int rc = trace_device(s, (const prt_ray*)dr, n, (prt_hit*)dh, stats);
  if (rc == PRT_OK && n > 0) {
    hipError_t e = hipMemcpyAsync(hits, dh, (size_t)n * sizeof(prt_hit), hipMemcpyDeviceToHost, s->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
    if (e != hipSuccess) rc = fail(PRT_E_HIP, hipGetErrorString(e));
  }
  if (dr) (void)hipFree(dr);
  if (dh) (void)hipFree(dh);
  return rc;
}

// ---------------------------------------------------------------- render
extern "C++" int prt::ensure_workspace(prt_scene* s, int64_t batch_samples, bool two_accum) {
  Workspace& w = s->pool->ws;
  // A slab writer over input chunks [c0, c1) owns fan * 64 * (c1 - c0)
  // entries from fan * 64 * c0 on, so a launch's outputs span fan * 64 *
  // (input chunks) <= fan * (input rays + 64 * PRT_SLAB_WAVES).  With glass a
  // vertex at depth <= 2 spawns two children (fan 2), deeper ones one, so
  // fan * input rays <= 8x the samples (2 * 4x at depth 2); without glass 1x.
  // Shadow rays: three per ray of the NEE input.
  const int64_t grow = s->has_glass ? 8 : 1;
  const int64_t W = PRT_SLAB_WAVES;
  int64_t qcap = grow * batch_samples + 2 * 64 * W + 64;
  int64_t scap = 3 * (grow * batch_samples + 64 * W);
  if (qcap >= ((int64_t)1 << 32) || scap >= ((int64_t)1 << 32)) return fail(PRT_E_INVALID, "batch too large");
  // the second shadow queue of the alternating schedule (NEE scenes only)
  bool two_sq = PRT_OVERLAP_SHADOW == 3 && s->P.nee && s->P.n_lights > 0;
  if (w.batch_samples >= batch_samples && w.queue_cap >= qcap && w.shadow_cap >= scap && w.h_counts &&
      (!two_accum || w.accum2.p) && (!two_sq || w.sq2[0].p))
    return PRT_OK;
  // The device's workspace serves every scene: it only grows (to the largest
  // sizes any call needed, keeping the optional buffers once they exist), so
  // scenes of different sizes in turn do not reallocate it back and forth.
  batch_samples = std::max(batch_samples, w.batch_samples);
  qcap = std::max(qcap, w.queue_cap);
  scap = std::max(scap, w.shadow_cap);
  two_sq = two_sq || w.sq2[0].p != nullptr;
  two_accum = two_accum || w.accum2.p != nullptr;
  // recorded sizes only once every buffer holds them: a failed allocation
  // has released its buffer, and the next call must not take the old sizes
  // for granted
  w.batch_samples = w.queue_cap = w.shadow_cap = 0;
  int rc;
  for (int qi = 0; qi < 2; ++qi)
    if ((rc = alloc_ray_queue(w.q[qi], qcap))) return rc;
  if ((rc = dev_alloc(w.hit_t, (size_t)qcap * 8))) return rc;
  if ((rc = dev_alloc(w.hit_id, (size_t)qcap * 4))) return rc;
  if ((rc = alloc_shadow_queue(w.sq, scap))) return rc;
  if (two_sq && (rc = alloc_shadow_queue(w.sq2, scap))) return rc;
  // chunks: a slab's last chunk may be partly filled
  for (int k = 0; k < (two_sq ? 4 : 3); ++k)
    if ((rc = dev_alloc(w.desc[k], (size_t)((k < 2 ? qcap : scap) / 64 + W + 1) * sizeof(uint2)))) return rc;
  if ((rc = dev_alloc(w.slabs, (size_t)3 * W * sizeof(uint2)))) return rc;
  if ((rc = dev_alloc(w.accum, (size_t)batch_samples * 3 * sizeof(uint64_t)))) return rc;
  if (two_accum && (rc = dev_alloc(w.accum2, (size_t)batch_samples * 3 * sizeof(uint64_t)))) return rc;
  if ((rc = dev_alloc(w.counts, 16 * sizeof(uint32_t)))) return rc;
  if ((rc = dev_alloc(w.fetch, (size_t)FETCH_LAUNCHES * PRT_FETCH_COUNTERS * PRT_FETCH_STRIDE * sizeof(uint32_t))))
    return rc;
  if ((rc = dev_alloc(w.ctr, CTR_WORDS * sizeof(uint64_t)))) return rc;
  if (!w.h_counts) HIPCHK(hipHostMalloc((void**)&w.h_counts, 16 * sizeof(uint32_t), hipHostMallocDefault));
  w.batch_samples = batch_samples;
  w.queue_cap = qcap;
  w.shadow_cap = scap;
  return PRT_OK;
}

// The part of the workspace a frame of the path kernel needs.
static int ensure_path_workspace(prt_scene* s, int64_t samples) {
  Workspace& w = s->pool->ws;
  // the queued renders use the same accumulators: a failed allocation has
  // released them, so they are not recorded until it has succeeded
  const int64_t recorded = w.batch_samples;
  w.batch_samples = 0;
  int rc;
  if ((rc = dev_alloc(w.accum, (size_t)samples * 3 * sizeof(uint64_t)))) return rc;
  w.batch_samples = recorded;
  if ((rc = dev_alloc(w.counts, 16 * sizeof(uint32_t)))) return rc;
  return dev_alloc(w.ctr, CTR_WORDS * sizeof(uint64_t));
}

// Settings of one render call derived from the scene and the options.
struct RenderSetup {
  Params P;
  int64_t n_pix = 0, bp = 0;
};

static int setup_render(prt_scene* s, const prt_render_opts* o, RenderSetup& R) {
  prt_render_opts opts{};
  if (o) opts = *o;
  Params P = s->P;
  if (opts.samples_override > 0) {
    P.samples = opts.samples_override;
    P.spp = P.samples * P.SS * P.SS;
    P.smp = 1.0 / P.samples / (P.SS * P.SS);
  }
  if (P.spp > (1 << 20)) return fail(PRT_E_INVALID, "samples per pixel above 2^20");
  P.max_vertices = opts.max_depth > 0 ? std::min(opts.max_depth, 255) : 128;
  P.key0 = (uint32_t)opts.seed;
  P.key1 = (uint32_t)(opts.seed >> 32);
  R.n_pix = (int64_t)P.W * P.H;
  // 2^PRT_BATCH_LOG2 camera samples per batch; half with glass, whose queues
  // are sized for up to 8 path segments per sample
  const int64_t batch_samples = (int64_t)1 << (s->has_glass ? PRT_BATCH_LOG2 - 1 : PRT_BATCH_LOG2);
  int64_t bp = opts.batch_pixels > 0 ? opts.batch_pixels : std::max<int64_t>(1, batch_samples / P.spp);
  bp = std::min(bp, R.n_pix);
  // queues hold up to 16x (glass splits into slabs) and 24x (shadow rays)
  // the batch, indexed by uint32
  while (bp > 1 && bp * P.spp * 32 >= ((int64_t)1 << 32)) bp /= 2;
  R.bp = bp;
  R.P = P;
  return PRT_OK;
}

// Depths enqueued between host reads of the ray count (a depth with an
// empty queue costs only near-empty launches).
#ifndef PRT_DEPTHS_PER_SYNC
#define PRT_DEPTHS_PER_SYNC 4
#endif

// Largest batches of scenes with next-event estimation that the path kernel
// traces alone (camera samples), and the queue size at which it takes over a
// batch's tail (rays).  A depth-synchronous depth or a tile-queue iteration
// costs two traversal launches however few its rays; the path kernel pays no
// launch per depth, but its waves wait for their slowest ray in every trip.
// Measured (path kernel / the queued engine of such scenes, ms):
//   box, 104 triangles: 0.26 M samples 1.26 / 1.47, 0.39 M 1.73 / 1.68, 0.52 M 2.25 /
//   1.92; 82k: 2.12 / 2.51, 2.85 / 2.87, 3.54 / 3.21; 1.3 M: 2.88 / 3.48, 3.87 / 4.11,
//   4.62 / 4.62;
//   with glass, where the tile queue drains through long tails, spheres 2.1 M samples
//   4.41 / 6.27, 2.6 M 5.45 / 8.47; and 60k triangles 1.6 M 6.27 / 6.43, 2.1 M 8.21 /
//   7.88, 2.6 M 10.2 / 10.8; field of 103k triangles 2.1 M 2.10 / 2.77, of 564k 1.0 M
//   3.53 / 3.88, 1.6 M 4.33 / 4.26, 2.1 M 5.13 / 4.72, of 2.1 M 1.0 M 4.37 / 4.57, 1.6 M
//   5.87 / 5.09, 2.1 M 6.93 / 5.61: for the largest meshes the line lies too high.
#ifndef PRT_PATH_SAMPLES
#define PRT_PATH_SAMPLES (3 << 17)
#endif
#ifndef PRT_PATH_SAMPLES_GLASS
#define PRT_PATH_SAMPLES_GLASS (1 << 21)
#endif
// Every ray tests every analytic entity, in the path kernel two waves per SIMD
// and at the lanes that have a ray then: with more entities than the LDS copy
// holds it is the faster one for fewer samples, about as the number of the others.
// Measured as above: spheres with glass, 40 entities, 0.61 M samples 2.69 / 3.19, 0.86 M
// 3.65 / 3.87, 1.6 M 6.16 / 5.60; 100: 0.24 M 2.58 / 2.63, 0.38 M 3.10 / 2.98, 0.61 M 4.83
// / 3.64; 400: 7 k 1.42 / 3.05, 55 k 4.04 / 3.20, 0.13 M 8.66 / 3.98; without glass, 100:
// 0.13 M 1.46 / 1.57, 0.24 M 1.88 / 1.85, 0.38 M 2.77 / 2.16; 400: 55 k 1.98 / 2.88, 0.13 M
// 5.43 / 3.18.
#ifndef PRT_PATH_ENTITIES
#define PRT_PATH_ENTITIES ((int64_t)1 << 25)
#endif
#ifndef PRT_PATH_TAIL
#define PRT_PATH_TAIL (1 << 16)
#endif

extern "C++" PathGrid prt::path_grid(int cu_count, int waves, uint64_t n, bool nee, bool whole_chunks) {
  PathGrid g;
  if (waves == 0) waves = n >= (uint64_t)std::max(1, cu_count) * 2 * 256 ? 3 : 2;
  waves = path_waves(waves, nee);
  g.waves = waves;
  g.blocks = std::max(1, cu_count) * waves;  // one 256-thread block per CU puts one wave on each SIMD
  const uint64_t per_wave = (n + g.n_waves() - 1) / g.n_waves();
  if (!whole_chunks && per_wave < 64) {
    // fewer samples than lanes: every wave gets the same few, so that a wave's
    // free lanes trace the light samples and glass branches of its own
    g.unit = g.quota = (uint32_t)std::max<uint64_t>(1, per_wave);
    g.blocks = (int)std::max<uint64_t>(1, ((n + g.unit - 1) / g.unit + 3) / 4);
  }
  // 256 samples per claim atomic once that leaves every wave 64 claims to even
  // out what samples cost.  From 4 claims a wave on, as it was, a field of 2.1 M
  // triangles, 8 spp, light sampling took at 2^21, 2^22, 2^23, 2^24 samples 10.6,
  // 14.6, 25.0, 44.5 ms against 7.0, 11.9, 22.1, 42.2 ms with one chunk per claim,
  // the spheres 4.41, 8.94, 17.1, 33.6 against 4.41, 8.52, 16.7, 33.2; at 2^26
  // samples without light sampling 62.3 and 64.1 ms, 41.2 and 41.0.
  if (per_wave >= 64 * 256) g.claim = 4;
  return g;
}

extern "C++" int prt::ensure_path_pool(DevBuf& b, const PathGrid& g, bool glass) {
  return dev_alloc(b, glass ? (size_t)g.n_waves() * PRT_PATH_POOL * sizeof(PoolRec) : 256);
}

static int64_t path_samples_most(const prt_scene* s) { return s->has_glass ? PRT_PATH_SAMPLES_GLASS : PRT_PATH_SAMPLES; }
static int64_t path_samples(const prt_scene* s) {
  const int64_t more = s->P.n_analytic - PRT_LDS_ANALYTIC;
  return more > 0 ? std::min(path_samples_most(s), PRT_PATH_ENTITIES / more) : path_samples_most(s);
}

// One batch's samples (src PATH_FRAME), or the rays of q[k] (PATH_QUEUE),
// through the path kernel.
static int run_path(prt_scene* s, PathSource src, const Params& P, const Batch& B, int k, uint64_t* accum,
                    const PathGrid& g) {
  Workspace& w = s->pool->ws;
  hipStream_t st = s->stream;
  uint32_t* counts = (uint32_t*)w.counts.p;
  const int64_t ns = B.n_pixels * P.spp;
  Persist a{};
  a.next = counts + 12;
  a.accum = accum;
  a.pool = (PoolRec*)w.pool.p;
  a.ctr = (uint64_t*)w.ctr.p;
  a.n_chunks = (uint32_t)((ns + g.unit - 1) / g.unit);
  a.claim = g.claim;
  a.n_scenes = 1;
  a.quota = g.quota;
  a.unit = g.unit;
  a.n_samples = (uint32_t)ns;
  a.nee = P.nee && P.n_lights > 0;
  a.batch = B;
  a.q = ray_queue(w.q[k], w.queue_cap);
  a.cl = ChunkList{(const uint2*)w.desc[k].p, counts + k};
  HIPCHK(launch_fill_u32(a.next, g.n_waves() * g.claim, 1, st));
  HIPCHK(launch_path(src, a, P, g.waves, g.blocks, st));
  return PRT_OK;
}

// Steps per launch of the chains: short enough that one launch stays well
// under a second, long enough that its end (the last chains finish alone) is
// a small part of it.
#ifndef PRT_CHAIN_STEPS
#define PRT_CHAIN_STEPS 256u
#endif

// n Markov chains at their own pace, one lane of the path kernel each, or step by
// step with all chains' proposals as one batch.  A step of all chains lasts as
// long as its longest path, and a chain's path ends the trip before its next
// begins.  A glass vertex's second segment runs on another lane, so no lane knows
// when the proposal is complete: those scenes go step by step.
// Measured (in step / own pace, ms): 15,360 chains 31.3 / 23.4, 65,536 64.3 / 53.9,
// 180,000 142.5 / 131.5, 360,000 187.4 / 178.9.
extern "C++" bool prt::chains_async(const prt_scene* s, uint32_t n) { return !s->has_glass && n <= PRT_PATH_SAMPLES; }

extern "C++" int prt::run_chains(prt_scene* s, const Params& P, const ChainRun& R, uint32_t n, uint32_t steps, Timer& tm,
                    CallTotals& tot) {
  Workspace& w = s->pool->ws;
  hipStream_t st = s->stream;
  const PathGrid g = path_grid(s->cu_count, 0, n, true, false);
  int rc = ensure_path_pool(w.pool, g, false);
  if (rc) return rc;
  Persist a{};
  a.next = (uint32_t*)w.counts.p + 12;
  a.pool = (PoolRec*)w.pool.p;
  a.ctr = (uint64_t*)w.ctr.p;
  a.n_chunks = (n + g.unit - 1) / g.unit;
  a.claim = g.claim;
  a.n_scenes = 1;
  a.quota = g.quota;
  a.unit = g.unit;
  a.n_samples = n;
  a.nee = 1;
  a.chain = R;
  if ((rc = tm.mark(T_OTHER))) return rc;
  for (uint32_t it = 0; it < steps; it += PRT_CHAIN_STEPS) {
    a.chain.it0 = it;
    a.chain.it1 = it + std::min<uint32_t>(PRT_CHAIN_STEPS, steps - it);
    HIPCHK(launch_fill_u32(a.next, g.n_waves() * g.claim, 1, st));
    HIPCHK(launch_path(PATH_CHAIN, a, P, g.waves, g.blocks, st));
    tot.primary_rays += (uint64_t)n * (a.chain.it1 - it);
    tot.launches++;
  }
  return tm.mark(T_EXTEND);
}

// One batch through the wavefront: generate, then extend / shade / NEE /
// shadow per path depth until no ray is left.  Sample radiance accumulates
// into `accum` (fixed point, 3 per camera sample of the batch).  Each
// slab-writing kernel is followed by k_slab_index, which lists the chunks
// of the queue it wrote for the kernels that read it.  The host reads the
// ray count once per PRT_DEPTHS_PER_SYNC depths.  A depth's shadow rays are
// traced on the scene's second stream as PRT_OVERLAP_SHADOW selects (an
// adjoint's replay, which reads the partial sums of a sample in path order, keeps
// one stream; its recording pass waits for them before the next shade); a NEE
// that rewrites a shadow queue waits for the shadow launch that read it, a
// shadow launch on the main stream for the one before it (they share the stack
// area), and the batch's end for every shadow launch.
static int run_batch_on(prt_scene* s, const Params& P, const Batch& B, uint64_t* accum, Adjoint A,
                        BatchForm form, Timer& tm, CallTotals& tot, uint32_t* n_records) {
  Workspace& w = s->pool->ws;
  hipStream_t st = s->stream;
  const int64_t ns = B.n_pixels * P.spp;
  if (form == FORM_PATH || (form == FORM_AUTO && ns <= path_samples(s))) {
    const PathGrid g = path_grid(s->cu_count, 0, (uint64_t)ns, P.nee && P.n_lights > 0, false);
    int rc = ensure_path_pool(w.pool, g, s->has_glass);
    if (rc) return rc;
    HIPCHK(launch_fill_u64(accum, 0ull, 3 * ns, st));
    if (P.mlt_u) HIPCHK(launch_mlt_gen(P, (uint32_t)ns, ray_queue(w.q[0], w.queue_cap), st));
    if ((rc = tm.mark(T_OTHER))) return rc;
    if ((rc = run_path(s, PATH_FRAME, P, B, 0, accum, g))) return rc;
    if ((rc = tm.mark(T_EXTEND))) return rc;
    tot.primary_rays += (uint64_t)ns;
    tot.launches++;
    return PRT_OK;
  }
  const int overlap = A.on == ADJ_REPLAY || (A.on && PRT_OVERLAP_SHADOW != 3) ? 0 : PRT_OVERLAP_SHADOW;
  hipStream_t st_sh = overlap ? s->stream2 : st;
  uint32_t* counts = (uint32_t*)w.counts.p;
  uint32_t* fetch = (uint32_t*)w.fetch.p;
  uint2* slabs = (uint2*)w.slabs.p;
  uint64_t* ctr = (uint64_t*)w.ctr.p;
  RayQ q[2] = {ray_queue(w.q[0], w.queue_cap), ray_queue(w.q[1], w.queue_cap)};
  ShadowQ sq = shadow_queue(w.sq, w.shadow_cap);
  const int tb = s->max_trav_blocks;
  // the shadow grid on the second stream leaves room on each CU; on the main
  // stream (no overlap) it is the closest-hit grid
  const int tb_sh = overlap ? std::max(1, s->cu_count) * PRT_SHADOW_BLOCKS_PER_CU : tb;
  const bool nee = P.nee && P.n_lights > 0;
  const uint32_t W = PRT_SLAB_WAVES;
  const size_t fetch_launch = (size_t)PRT_FETCH_COUNTERS * PRT_FETCH_STRIDE;
  // children per shaded vertex: glass splits in two up to depth 2
  auto fan = [&](int depth) { return (uint32_t)(s->has_glass && depth <= 2 ? 2 : 1); };
  auto chunks = [&](int k) { return ChunkList{(const uint2*)w.desc[k].p, counts + k}; };
  auto index = [&](int k, uint32_t n_slabs, const uint2* sl, hipStream_t on) {
    const uint32_t max_chunks = (uint32_t)(w.desc[k].bytes / sizeof(uint2));
    return launch_slab_index(sl, n_slabs, (uint2*)w.desc[k].p, max_chunks, counts + k, counts + 4 + k, ctr,
                             k < 2 ? CTR_QUEUED : -1, on);
  };
  int fi = 0;  // traversal launches so far; each takes fresh claim counters
  auto next_fetch = [&](uint32_t** f) -> int {
    if (fi >= FETCH_LAUNCHES) return fail(PRT_E_INVALID, "too many wavefront launches in one batch");
    if (fi % FETCH_GROUP == 0) HIPCHK(launch_fill_u32(fetch + fi * fetch_launch, 0u, FETCH_GROUP * fetch_launch, st));
    *f = fetch + fi++ * fetch_launch;
    return PRT_OK;
  };
  int rc;
  uint32_t* f;
  // NEE of the rays in q[k] and the any-hit tests of its shadow rays
  auto nee_and_shadow = [&](int k) -> int {
    if (overlap == 2) {
      // both on the second stream, after the shade that wrote q[k]; the
      // claim counters are cleared on the main stream before the hand-over
      if ((rc = next_fetch(&f))) return rc;
      HIPCHK(hipEventRecord(s->ev_shade, st));
      HIPCHK(hipStreamWaitEvent(st_sh, s->ev_shade, 0));
      if ((rc = tm.begin_side(st_sh))) return rc;
      HIPCHK(launch_nee(P, B, q[k], chunks(k), sq, slabs + 2 * W, ctr, st_sh));
      HIPCHK(index(2, W, slabs + 2 * W, st_sh));
      if ((rc = tm.end_side(st_sh, T_NEE))) return rc;
      HIPCHK(hipEventRecord(s->ev_nee[k], st_sh));
      if ((rc = tm.begin_side(st_sh))) return rc;
      HIPCHK(launch_shadow(P, B, sq, chunks(2), f, accum, A, ctr, tb_sh, st_sh));
      if ((rc = tm.end_side(st_sh, T_SHADOW))) return rc;
      HIPCHK(hipEventRecord(s->ev_shadow, st_sh));
      return PRT_OK;
    }
    if (overlap) HIPCHK(hipStreamWaitEvent(st, s->ev_shadow, 0));  // the last shadow launch has read sq
    HIPCHK(launch_nee(P, B, q[k], chunks(k), sq, slabs + 2 * W, ctr, st));
    HIPCHK(index(2, W, slabs + 2 * W, st));
    if ((rc = tm.mark(T_NEE))) return rc;
    if ((rc = next_fetch(&f))) return rc;
    if (overlap) {
      HIPCHK(hipEventRecord(s->ev_shade, st));
      HIPCHK(hipStreamWaitEvent(st_sh, s->ev_shade, 0));
      if ((rc = tm.begin_side(st_sh))) return rc;
    }
    HIPCHK(launch_shadow(P, B, sq, chunks(2), f, accum, A, ctr, tb_sh, st_sh));
    if (overlap) {
      if ((rc = tm.end_side(st_sh, T_SHADOW))) return rc;
      HIPCHK(hipEventRecord(s->ev_shadow, st_sh));
    } else if ((rc = tm.mark(T_SHADOW))) {
      return rc;
    }
    return PRT_OK;
  };
  // Alternating schedule (overlap 3): the NEE of q[k] on the main stream
  // into shadow queue sh_next, whose shadow rays are traced on the second
  // stream after the next depth's closest-hit launch (shadow_alt).
  const bool alt = overlap == 3 && nee;
  const ShadowQ sqs[2] = {sq, alt ? shadow_queue(w.sq2, w.shadow_cap) : sq};
  int sh_next = 0, sh_pending = -1;
  bool sh_used[2] = {false, false};
  auto nee_alt = [&](int k) -> int {
    const int b = sh_next;
    sh_next ^= 1;
    if (sh_used[b]) HIPCHK(hipStreamWaitEvent(st, s->ev_sh[b], 0));  // its last shadow launch has read it
    HIPCHK(launch_nee(P, B, q[k], chunks(k), sqs[b], slabs + 2 * W, ctr, st));
    HIPCHK(index(2 + b, W, slabs + 2 * W, st));
    if ((rc = tm.mark(T_NEE))) return rc;
    sh_pending = b;
    return PRT_OK;
  };
  // the pending shadow queue's rays, after everything enqueued so far on the
  // main stream (on the main stream itself when `side` is false)
  auto shadow_alt = [&](bool side) -> int {
    if (sh_pending < 0) return PRT_OK;
    const int b = sh_pending;
    sh_pending = -1;
    if ((rc = next_fetch(&f))) return rc;  // a fill clearing its counters goes on st first
    hipStream_t on = side ? st_sh : st;
    // never beside another shadow launch: they share a stack area
    if (!side && sh_used[b ^ 1]) HIPCHK(hipStreamWaitEvent(on, s->ev_sh[b ^ 1], 0));
    if (side) {
      HIPCHK(hipEventRecord(s->ev_shade, st));
      HIPCHK(hipStreamWaitEvent(on, s->ev_shade, 0));
      if ((rc = tm.begin_side(on))) return rc;
    }
    HIPCHK(launch_shadow(P, B, sqs[b], chunks(2 + b), f, accum, A, ctr, side ? tb_sh : tb, on));
    if (side) {
      if ((rc = tm.end_side(on, T_SHADOW))) return rc;
      HIPCHK(hipEventRecord(s->ev_sh[b], on));
      sh_used[b] = true;
    } else if ((rc = tm.mark(T_SHADOW))) {
      return rc;
    }
    return PRT_OK;
  };
  const int64_t np = B.n_pixels * P.SS * P.SS;
  int shades = 0;
  HIPCHK(launch_fill_u64(accum, 0ull, 3 * ns, st));
  HIPCHK(launch_fill_u32(counts, 0u, 16, st));
  // the primary rays: one slab of np rays at the start of q[0]
  HIPCHK(launch_fill_u32((uint32_t*)slabs, 0u, 1, st));
  HIPCHK(launch_fill_u32((uint32_t*)slabs + 1, (uint32_t)np, 1, st));
  if (P.mlt_u) HIPCHK(launch_mlt_gen(P, (uint32_t)np, q[0], st));
  else HIPCHK(launch_gen_primary(P, B, q[0], st));
  HIPCHK(index(0, 1, slabs, st));
  if ((rc = tm.mark(T_OTHER))) return rc;
  if ((rc = next_fetch(&f))) return rc;
  HIPCHK(launch_extend(P, q[0], chunks(0), np, f, (double*)w.hit_t.p, (int32_t*)w.hit_id.p, ctr, tb, st));
  if ((rc = tm.mark(T_EXTEND0))) return rc;
  tot.primary_rays += (uint64_t)np;
  tot.launches++;
  // Shade q[kin] (primary: every camera sample against its sub-pixel's
  // primary hit) into q[kout], then the NEE of the children.
  auto shade_nee = [&](int primary, int kin, int kout, uint32_t fn) -> int {
    A.recs.first = counts + 8 + (shades & 1);
    A.recs.next = counts + 8 + (++shades & 1);
    HIPCHK(launch_shade(P, B, primary, q[kin], chunks(kin), (const double*)w.hit_t.p, (const int32_t*)w.hit_id.p,
                        q[kout], fn, slabs + kout * W, accum, A, ctr, st));
    HIPCHK(index(kout, W, slabs + kout * W, st));
    if ((rc = tm.mark(T_SHADE))) return rc;
    return nee ? (alt ? nee_alt(kout) : nee_and_shadow(kout)) : PRT_OK;
  };
  if ((rc = shade_nee(1, 0, 1, fan(0)))) return rc;
  int cur = 1;
  for (int depth = 1;; ++depth) {  // depth of the rays in q[cur]
    if ((depth - 1) % PRT_DEPTHS_PER_SYNC == 0) {
      HIPCHK(hipMemcpyAsync(w.h_counts, counts, 16 * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      const uint32_t rays = w.h_counts[4 + cur];
      if (n_records) *n_records = w.h_counts[8 + (shades & 1)];
      if (rays == 0) break;
      if (form == FORM_AUTO && rays <= PRT_PATH_TAIL) {
        // the rest of the batch in one launch, alongside the shadow rays of q[cur]'s NEE
        if (alt && (rc = shadow_alt(true))) return rc;
        const PathGrid g = path_grid(s->cu_count, 2, rays, true, true);
        if ((rc = ensure_path_pool(w.pool, g, s->has_glass))) return rc;
        if ((rc = run_path(s, PATH_QUEUE, P, B, cur, accum, g))) return rc;
        if ((rc = tm.mark(T_EXTEND))) return rc;
        tot.launches++;
        break;
      }
    }
    const int nxt = cur ^ 1;
    // a recording pass: alongside this depth's closest hits, because the shade
    // reads the samples' sums so far
    if (alt && A.on && (rc = shadow_alt(true))) return rc;
    if ((rc = next_fetch(&f))) return rc;
    if ((rc = tm.mark(T_OTHER))) return rc;
    HIPCHK(launch_extend(P, q[cur], chunks(cur), (int64_t)tb * 256, f, (double*)w.hit_t.p, (int32_t*)w.hit_id.p, ctr,
                         tb, st));
    if ((rc = tm.mark(T_EXTEND))) return rc;
    tot.launches++;
    // the shadow rays of q[cur]'s NEE, alongside this depth's shade and NEE
    if (alt && !A.on && (rc = shadow_alt(true))) return rc;
    if (alt && A.on) HIPCHK(hipStreamWaitEvent(st, s->ev_sh[sh_next ^ 1], 0));
    // the NEE two depths back read q[nxt] and its chunk list
    if (overlap == 2 && nee) HIPCHK(hipStreamWaitEvent(st, s->ev_nee[nxt], 0));
    if ((rc = shade_nee(0, cur, nxt, fan(depth)))) return rc;
    cur = nxt;
  }
  if (alt) {
    if ((rc = shadow_alt(false))) return rc;
    for (int b = 0; b < 2; ++b)
      if (sh_used[b]) HIPCHK(hipStreamWaitEvent(st, s->ev_sh[b], 0));
  } else if (overlap) {
    HIPCHK(hipStreamWaitEvent(st, s->ev_shadow, 0));
  }
  return PRT_OK;
}

extern "C++" int prt::run_batch(prt_scene* s, const Params& P, const Batch& B, uint64_t* accum, const Adjoint& A,
                                BatchForm form, Timer& tm, CallTotals& tot, uint32_t* n_records) {
  const int rc = run_batch_on(s, P, B, accum, A, form, tm, tot, n_records);
  // a failed batch may have left shadow work queued on the second stream
  if (rc != PRT_OK) (void)hipStreamSynchronize(s->stream2);
  return rc;
}

static int finish_stats(prt_scene* s, const RenderSetup& R, Timer& tm, const CallTotals& tot, prt_stats* stats,
                        uint64_t* c) {
  hipStream_t st = s->stream;
  uint64_t raw[CTR_WORDS];
  HIPCHK(hipMemcpyAsync(raw, s->pool->ws.ctr.p, sizeof(raw), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  sum_counters(raw, c);
  if (const int rc = check_traced(c, tot.primary_rays)) return rc;
  double cat[T_NCAT] = {0, 0, 0, 0, 0, 0};
  double trav = 0.0;
  const double wall = tm.collect(cat, &trav, 1u << T_EXTEND | 1u << T_EXTEND0 | 1u << T_SHADOW);
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    fill_stats(stats, c);
    stats->camera_samples = (uint64_t)R.n_pix * R.P.spp;
    stats->primary_rays = tot.primary_rays;
    stats->extension_rays = c[CTR_QUEUED] - tot.primary_rays;
    stats->shadow_rays = c[CTR_SHADOW];
    stats->ms_extend = cat[T_EXTEND] + cat[T_EXTEND0];
    stats->ms_shade = cat[T_SHADE];
    stats->ms_shadow = cat[T_SHADOW];
    stats->ms_other = cat[T_OTHER];
    stats->ms_extend_primary = cat[T_EXTEND0];
    stats->ms_nee = cat[T_NEE];
    stats->ms_total = wall;
    stats->ms_traversal = trav;
    stats->launches_extend = tot.launches;
    // per ray query: 128 B per node record, 48 B per triangle record, 48 B
    // of ray in + hit out
    stats->bytes_extend = 128 * c[CTR_NODES] + 48 * c[CTR_TRIS] + 48 * c[CTR_QUEUED];
    stats->bytes_shadow = 128 * c[CTR_SNODES] + 48 * c[CTR_STRIS] + 48 * c[CTR_SHADOW];
    stats->bytes_algorithmic = stats->bytes_extend + stats->bytes_shadow;
  }
  return PRT_OK;
}

// Progress images of a render with prt_dump_opts (Render::Run's periodic
// OutputBmp, render.h:1390-1401): the device image is copied to the host
// between batches once the interval has passed.
struct ImageDumper {
  const prt_dump_opts* d = nullptr;
  std::chrono::steady_clock::time_point last;
  int32_t index = 0;
  std::vector<float> host;
  std::vector<double> host64;

  bool on() const { return d != nullptr && d->seconds >= 0.0; }
  bool due() const {
    const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - last).count();
    return d->seconds == 0.0 || el >= d->seconds;
  }
  int dump(prt_scene* s, const void* d_rgb, int f64, double fraction) {
    const int W = s->P.W, H = s->P.H;
    const size_t n = (size_t)W * H * 3;
    host.resize(n);
    HIPCHK(hipStreamSynchronize(s->stream));
    if (f64) {
      host64.resize(n);
      HIPCHK(hipMemcpy(host64.data(), d_rgb, n * sizeof(double), hipMemcpyDeviceToHost));
      for (size_t i = 0; i < n; ++i) host[i] = (float)host64[i];
    } else {
      HIPCHK(hipMemcpy(host.data(), d_rgb, n * sizeof(float), hipMemcpyDeviceToHost));
    }
    if (d->callback) d->callback(d->user, host.data(), W, H, index, fraction);
    if (d->directory) {
      char name[32];
      std::snprintf(name, sizeof(name), "output_W%06d.bmp", (int)index);
      const std::string path = std::string(d->directory) + "/" + name;
      const int rc = prt_write_bmp(path.c_str(), host.data(), W, H, d->gamma_offset);
      if (rc != PRT_OK) return rc;
    }
    ++index;
    last = std::chrono::steady_clock::now();
    return PRT_OK;
  }
};

static int render_device(prt_scene* s, const prt_render_opts* o, float* d_rgb, float* d_var, prt_stats* stats,
                         ImageDumper* dumper = nullptr) {
  HIPCHK(hipSetDevice(s->device));
  std::lock_guard<std::recursive_mutex> pool_lock(s->pool->m);
  // Scenes with glass stream through the batched renderer's tile queue: a
  // depth-synchronous batch of them drains through long, thin tails after
  // the glass splits, which the stream keeps filled with new tiles.  Same
  // image bits either way (fixed-point sums, counter-based random numbers).
  if (o && o->reserved_ != 0) return fail(PRT_E_INVALID, "prt_render_opts.reserved_ must be 0");
  const int engine = o ? o->engine : 0;
  const bool stream_ok = !o || (o->image_f64 == 0 && o->samples_override <= 0 && o->batch_pixels <= 0);
  if (engine == 2 && !stream_ok)
    return fail(PRT_E_INVALID, "the streaming engine writes float images without samples_override / batch_pixels");
  const bool dumping = dumper && dumper->on();
  if (dumping && (engine == 2 || engine == 3))
    return fail(PRT_E_INVALID, "progress images need the depth-synchronous engine");
  if (engine < 0 || engine > 3) return fail(PRT_E_INVALID, "engine must be 0..3");
  // Scenes without next-event estimation take the path kernel at any size, others
  // up to path_samples.  Measured without it (path kernel / the faster of the
  // queued engines, ms, 16 spp): spheres 0.26 M samples 0.39 / 0.78, 16.8 M 10.4 / 12.7;
  // and 60k triangles 1.0 M 1.68 / 2.57, 4.2 M 5.55 / 5.62, 16.8 M 21.2 / 18.8; box of 82k
  // triangles 1.0 M 2.25 / 2.72, 4.2 M 7.56 / 5.88, 16.8 M 28.8 / 18.0, of 1.3 M 2.97 / 4.04,
  // 10.2 / 7.59, 38.9 / 21.1; field of 2.1 M triangles 0.26 M 1.98 / 2.08, 16.8 M 17.1 /
  // 14.5.  From some 3 M samples on, then, meshes are faster depth-synchronous
  // (engine 1) at the price of its queues, 700 bytes a sample against 24.
  const bool nee_scene = s->P.nee && s->P.n_lights > 0;
  const bool persist_ok = stream_ok && (uint64_t)s->P.W * s->P.H * s->P.spp <= ((uint64_t)1 << 28);
  if (engine == 3 && !persist_ok)
    return fail(PRT_E_INVALID, "the persistent engine writes float images of at most 2^28 samples, without "
                               "samples_override / batch_pixels");
  const int64_t frame = (int64_t)s->P.W * s->P.H * s->P.spp;
  bool path = engine == 3 || (engine == 0 && persist_ok && !dumping && (!nee_scene || frame <= path_samples(s)));
  // a frame that only its scene's entities keep from the path kernel takes it all
  // the same where there is no memory for queues
  const bool path_fits = engine == 0 && persist_ok && !dumping && frame <= path_samples_most(s);
  int rc;
  if (engine == 2 || (engine == 0 && !path && s->has_glass && stream_ok && !dumping)) {
    prt_batch_opts b{};
    b.seed = o ? o->seed : 0;
    b.max_depth = o ? o->max_depth : 0;
    b.timing = o ? o->timing : 0;
    b.use_graph = -1;            // plain launches (faster than graph replay; timed renders need them)
    // samples in flight: a whole frame of up to 2^21, else the batched
    // renderer's automatic size (the most, up to 2^24, whose workspace fits
    // its share of the device memory)
    b.tile_samples = 4096;
    b.inflight_tiles = frame <= ((int64_t)1 << 21) ? (int32_t)std::max<int64_t>(1, (frame + 4095) / 4096) : 0;
    prt_scene* const one[1] = {s};
    float* const rgb[1] = {d_rgb};
    float* const var[1] = {d_var};
    rc = prt_render_batch_device(one, 1, &b, rgb, var, stats);
    if (rc != PRT_E_NOMEM || !path_fits) return rc;
    path = true;
  }
  RenderSetup R;
  if ((rc = setup_render(s, o, R))) return rc;
  if (!path && (rc = ensure_workspace(s, R.bp * R.P.spp, false))) {
    if (rc != PRT_E_NOMEM || !path_fits) return rc;
    path = true;
  }
  if (path) {
    R.bp = R.n_pix;  // one launch, which needs no queues
    if ((rc = ensure_path_workspace(s, R.n_pix * R.P.spp))) return rc;
  }
  hipStream_t st = s->stream;
  HIPCHK(launch_fill_u64((uint64_t*)s->pool->ws.ctr.p, 0ull, CTR_WORDS, st));
  Timer tm;
  if ((rc = tm.begin(path || (o && o->timing != 0), st, &s->timer_events))) return rc;
  CallTotals tot;
  Adjoint none{};
  // engine 1 and renders with progress images or a batch size are asked to be
  // depth-synchronous
  const BatchForm form = path ? FORM_PATH : engine == 1 || dumping || (o && o->batch_pixels > 0) ? FORM_WAVEFRONT : FORM_AUTO;
  const int f64 = o && o->image_f64;
  if (dumping) {
    // pixels not yet rendered read as 0 in the progress images
    const int64_t n = R.n_pix * 3;
    if (f64)
      HIPCHK(launch_fill_u64((uint64_t*)d_rgb, 0ull, n, st));
    else
      HIPCHK(launch_fill_f32(d_rgb, 0.0f, n, st));
    dumper->last = std::chrono::steady_clock::now();
  }
  for (int64_t pb = 0; pb < R.n_pix; pb += R.bp) {
    Batch B{pb, std::min(R.bp, R.n_pix - pb)};
    if ((rc = run_batch(s, R.P, B, (uint64_t*)s->pool->ws.accum.p, none, form, tm, tot))) return rc;
    HIPCHK(launch_resolve(R.P, B, (const uint64_t*)s->pool->ws.accum.p, d_rgb, d_var, f64, st));
    if ((rc = tm.mark(T_OTHER))) return rc;
    const int64_t done = pb + B.n_pixels;
    if (dumping && done < R.n_pix && dumper->due() &&
        (rc = dumper->dump(s, d_rgb, f64, (double)done / (double)R.n_pix)))
      return rc;
  }
  uint64_t c[CTR_COUNT];
  return finish_stats(s, R, tm, tot, stats, c);
}

int prt_render_device(prt_scene* s, const prt_render_opts* opts, float* d_rgb, float* d_var, prt_stats* stats) {
  if (!s || !d_rgb) return fail(PRT_E_INVALID, "bad arguments");
  return render_device(s, opts, d_rgb, d_var, stats);
}

int prt_render(prt_scene* s, const prt_render_opts* opts, float* out_rgb, float* out_var, prt_stats* stats) {
  if (!s || !out_rgb) return fail(PRT_E_INVALID, "bad arguments");
  HIPCHK(hipSetDevice(s->device));
  const size_t bytes = (size_t)s->P.W * s->P.H * 3 * sizeof(float);
  int rc;
  if ((rc = dev_alloc(s->out_rgb, bytes))) return rc;
  if (out_var && (rc = dev_alloc(s->out_var, bytes))) return rc;
  prt_render_opts o32{};
  if (opts) o32 = *opts;
  o32.image_f64 = 0;  // host outputs are float
  rc = render_device(s, &o32, (float*)s->out_rgb.p, out_var ? (float*)s->out_var.p : nullptr, stats);
  if (rc) return rc;
  HIPCHK(hipMemcpyAsync(out_rgb, s->out_rgb.p, bytes, hipMemcpyDeviceToHost, s->stream));
  if (out_var) HIPCHK(hipMemcpyAsync(out_var, s->out_var.p, bytes, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return PRT_OK;
}

int prt_render_dump(prt_scene* s, const prt_render_opts* opts, const prt_dump_opts* dump, float* out_rgb,
                    float* out_var, prt_stats* stats) {
  if (!s || !out_rgb) return fail(PRT_E_INVALID, "bad arguments");
  HIPCHK(hipSetDevice(s->device));
  const size_t bytes = (size_t)s->P.W * s->P.H * 3 * sizeof(float);
  int rc;
  if ((rc = dev_alloc(s->out_rgb, bytes))) return rc;
  if (out_var && (rc = dev_alloc(s->out_var, bytes))) return rc;
  prt_render_opts o32{};
  if (opts) o32 = *opts;
  o32.image_f64 = 0;  // host outputs are float
  ImageDumper dumper;
  dumper.d = dump;
  rc = render_device(s, &o32, (float*)s->out_rgb.p, out_var ? (float*)s->out_var.p : nullptr, stats, &dumper);
  if (rc) return rc;
  HIPCHK(hipMemcpyAsync(out_rgb, s->out_rgb.p, bytes, hipMemcpyDeviceToHost, s->stream));
  if (out_var) HIPCHK(hipMemcpyAsync(out_var, s->out_var.p, bytes, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return PRT_OK;
}

// ---------------------------------------------------------------- differentiable parameters
int prt_set_face_albedo_device(prt_scene* s, int entity, const float* d_albedo) {
  if (!s || !d_albedo || entity < 0 || entity >= (int)s->h_ents.size()) return fail(PRT_E_INVALID, "bad arguments");
  const DevEntity& e = s->h_ents[entity];
  if (e.type != PRT_ENTITY_POLYGON || !e.has_albedo)
    return fail(PRT_E_INVALID, "entity is not a POLYGON created with per-face albedo");
  HIPCHK(hipSetDevice(s->device));
  HIPCHK(launch_scatter_albedo((float*)s->tri_alb.p, (const uint32_t*)s->d_slot_of_tri.p, s->ent_first_tri[entity],
                               s->ent_n_tris[entity], d_albedo, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return PRT_OK;
}

static void sort_lights(prt_scene* s) {
  struct L { int32_t ent; double power; };
  std::vector<L> ls;
  for (int i = 0; i < (int)s->h_ents.size(); ++i) {
    const DevEntity& de = s->h_ents[i];
    if (!de.light || de.type == PRT_ENTITY_POLYGON) continue;
    ls.push_back(L{i, de.area * length(from(s->h_mats[de.material].emission))});
  }
  std::stable_sort(ls.begin(), ls.end(), [](const L& a, const L& b) { return a.power > b.power; });
  s->h_lights.clear();
  for (const L& l : ls) s->h_lights.push_back(l.ent);
}

int prt_hold_rr_albedo(prt_scene* s, int hold) {
  if (!s) return fail(PRT_E_INVALID, "null scene");
  HIPCHK(hipSetDevice(s->device));
  if (!hold) {
    s->P.tri_alb_rr = nullptr;
    return PRT_OK;
  }
  if (!s->tri_alb.p) return fail(PRT_E_INVALID, "scene has no per-face albedo");
  const size_t bytes = (size_t)s->n_tris * 3 * sizeof(float);
  int rc;
  if ((rc = dev_alloc(s->tri_alb_rr, bytes))) return rc;
  HIPCHK(hipMemcpyAsync(s->tri_alb_rr.p, s->tri_alb.p, bytes, hipMemcpyDeviceToDevice, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  s->P.tri_alb_rr = (const float*)s->tri_alb_rr.p;
  return PRT_OK;
}

int prt_set_emission(prt_scene* s, int entity, const double emission[3]) {
  if (!s || !emission || entity < 0 || entity >= (int)s->h_ents.size()) return fail(PRT_E_INVALID, "bad arguments");
  HIPCHK(hipSetDevice(s->device));
  DevEntity& e = s->h_ents[entity];
  DevMaterial& m = s->h_mats[e.material];
  std::memcpy(m.emission, emission, sizeof(m.emission));
  const int was_light = m.is_light;
  m.is_light = (m.type == PRT_REFLECTION_DIFFUSE && length(from(m.color)) < 0.001 && length(from(m.emission)) > 0.001);
  if (m.is_light != was_light) return fail(PRT_E_UNSUPPORTED, "changing whether an entity is a light");
  // the light list order follows power (light.h:99)
  sort_lights(s);
  int rc;
  if ((rc = dev_upload(s->mats, s->h_mats, s->stream))) return rc;
  if ((rc = dev_upload(s->lights, s->h_lights, s->stream))) return rc;
  HIPCHK(hipStreamSynchronize(s->stream));
  return PRT_OK;
}

// Adjoint, per batch: one pass renders the samples and records every vertex on
// the differentiated entity with its sample's radiance up to it; then each
// record's gradient is what the sample got after it.  Records are slots, 64 per
// chunk that a shade launch reads, also for lanes without a ray and vertices on
// other entities.  A batch that needs more than PRT_ADJOINT_RECORDS per sample and
// 64 * 64 (long paths, above all in batches below 2^19 samples: a slab writer has
// one chunk there, which counts in full until its last ray has ended), or for
// which the memory is not to be had, is replayed instead: the same paths again,
// each vertex's gradient from the radiance that the first pass found.  A record
// takes 32 bytes, up to 8.6 GB for a batch of 2^24 samples, kept in the device's
// pool.
// Measured with the forward render, box with 82k triangles: 256x256 x 32 spp 23.9
// ms replayed, 16.5 ms recorded; 64x48 x 16 spp 4.9 and 3.3 ms.  With 2 records per
// sample, so that every batch is replayed after all, 24.1 ms.
#ifndef PRT_ADJOINT_RECORDS
#define PRT_ADJOINT_RECORDS 16
#endif
// Records that the workspace holds (0: no memory), grown for a batch.
static uint32_t ensure_records(Workspace& w, uint64_t samples, int max_vertices) {
  const uint64_t want = std::min<uint64_t>(samples * (uint64_t)std::min(PRT_ADJOINT_RECORDS, max_vertices) + 64 * 64,
                                           0xFFFF0000ull);
  for (int k = 0; k < 5; ++k)
    if (dev_alloc(w.recs[k], (size_t)want * (k < 2 ? 4 : 8)) != PRT_OK) {
      (void)hipGetLastError();
      for (auto& b : w.recs) b.release();
      return 0u;
    }
  return (uint32_t)std::min<uint64_t>(w.recs[0].bytes / 4, 0xFFFF0000ull);
}
static AdjointRecs adjoint_records(Workspace& w, uint32_t cap) {
  AdjointRecs r{};
  r.id = (int32_t*)w.recs[0].p;
  r.slot = (uint32_t*)w.recs[1].p;
  for (int c = 0; c < 3; ++c) r.before[c] = (double*)w.recs[2 + c].p;
  r.cap = cap;
  return r;
}

int prt_adjoint_device(prt_scene* s, const prt_render_opts* o, const float* d_dimage, int entity,
                       float* d_albedo_grad, int light, double* emission_grad, prt_stats* stats) {
  if (!s || !d_dimage) return fail(PRT_E_INVALID, "bad arguments");
  std::lock_guard<std::recursive_mutex> pool_lock(s->pool->m);
  if (s->has_glass)
    return fail(PRT_E_UNSUPPORTED, "the adjoint needs one path per sample (no glass splits)");
  if (s->P.cutoff > 0.0f) return fail(PRT_E_UNSUPPORTED, "the adjoint needs luminance_cutoff <= 0");
  const bool want_alb = d_albedo_grad != nullptr;
  if (want_alb) {
    if (entity < 0 || entity >= (int)s->h_ents.size() || s->h_ents[entity].type != PRT_ENTITY_POLYGON ||
        !s->h_ents[entity].has_albedo)
      return fail(PRT_E_INVALID, "albedo gradient needs a POLYGON entity created with per-face albedo");
  }
  if (light >= (int)s->h_ents.size()) return fail(PRT_E_INVALID, "bad light entity");
  HIPCHK(hipSetDevice(s->device));
  RenderSetup R;
  int rc;
  if ((rc = setup_render(s, o, R))) return rc;
  if ((rc = ensure_workspace(s, R.bp * R.P.spp, true))) return rc;
  hipStream_t st = s->stream;
  const int64_t nf = want_alb ? s->ent_n_tris[entity] : 0;
  if ((rc = dev_alloc(s->grad_buf, (size_t)(3 * nf + 3) * sizeof(double)))) return rc;
  double* g_alb = (double*)s->grad_buf.p;
  double* g_e = g_alb + 3 * nf;
  HIPCHK(launch_fill_u64((uint64_t*)g_alb, 0ull, 3 * nf + 3, st));
  HIPCHK(launch_fill_u64((uint64_t*)s->pool->ws.ctr.p, 0ull, CTR_WORDS, st));
  Timer tm;
  if ((rc = tm.begin(o && o->timing != 0, st, &s->timer_events))) return rc;
  CallTotals tot;
  Adjoint A{};
  A.on = ADJ_REPLAY;
  A.entity = want_alb ? entity : -1;
  A.light = light;
  A.dimage = d_dimage;
  A.ltot = (const uint64_t*)s->pool->ws.accum2.p;
  A.grad_alb = g_alb;
  A.grad_e = g_e;
  A.scale = R.P.sensor_response * R.P.smp;
  const uint32_t cap = want_alb ? ensure_records(s->pool->ws, (uint64_t)R.bp * R.P.spp, R.P.max_vertices) : 0u;
  for (int64_t pb = 0; pb < R.n_pix; pb += R.bp) {
    Batch B{pb, std::min(R.bp, R.n_pix - pb)};
    Adjoint rec = A;
    rec.on = ADJ_RECORD;
    rec.recs = adjoint_records(s->pool->ws, cap);
    uint32_t n = 0;
    if ((rc = run_batch(s, R.P, B, (uint64_t*)s->pool->ws.accum2.p, rec, FORM_WAVEFRONT, tm, tot, &n))) return rc;
    if (!want_alb) continue;
    if (n <= cap) {
      HIPCHK(launch_adjoint_resolve(R.P, B, rec, n, st));
      continue;
    }
    // more vertices than records: the samples' radiance is known now, so a replay
    // can do without (the emission's gradient is complete)
    A.light = INT32_MIN;
    if ((rc = run_batch(s, R.P, B, (uint64_t*)s->pool->ws.accum.p, A, FORM_WAVEFRONT, tm, tot))) return rc;
    A.light = light;
    HIPCHK(launch_count_mismatch((const uint64_t*)s->pool->ws.accum.p, (const uint64_t*)s->pool->ws.accum2.p,
                                 3 * B.n_pixels * R.P.spp, (uint64_t*)s->pool->ws.ctr.p, st));
  }
  if (want_alb) HIPCHK(launch_grad_to_f32(g_alb, d_albedo_grad, 3 * nf, st));
  double ge[3] = {0, 0, 0};
  HIPCHK(hipMemcpyAsync(ge, g_e, sizeof(ge), hipMemcpyDeviceToHost, st));
  uint64_t c[CTR_COUNT];
  if ((rc = finish_stats(s, R, tm, tot, stats, c))) return rc;
  if (c[CTR_REPLAY_MISMATCH] != 0)
    return fail(PRT_E_INVALID, "adjoint replay diverged from the primal pass on " +
                                   std::to_string(c[CTR_REPLAY_MISMATCH]) + " sample channels");
  if (emission_grad) std::memcpy(emission_grad, ge, sizeof(ge));
  return PRT_OK;
}

}  // extern "C"
