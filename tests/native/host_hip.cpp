// host_hip.cpp — a stand-in for the HIP runtime, so that the library's host side
// (allocation, workspace sizes, engine choice, the order of launches on its two
// streams) runs without a GPU.
//
// Loaded before libprt.so with RTLD_GLOBAL it answers the HIP calls: device
// memory is host memory, copies happen at once, and a launch runs what this file
// knows of the kernel, which is only what the host reads back (counts of rays,
// counters, the tile queue's status).  It notes
//   - writes of fills outside live allocations, and accumulators, queues and
//     counters handed to a kernel that are not in one;
//   - launches that use the same traversal-stack area without an order between
//     them, found with a vector clock per stream and event.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "prt_device.h"
#include "prt_kernels.h"
#include "prt_stream.h"

namespace {

typedef std::vector<uint64_t> Clock;
void merge(Clock& a, const Clock& b) {
  if (a.size() < b.size()) a.resize(b.size());
  for (size_t i = 0; i < b.size(); ++i) a[i] = std::max(a[i], b[i]);
}
struct HostStream {
  size_t id;
  Clock clock;
};
struct HostEvent {
  Clock clock;
};
struct Use {  // a launch that used a stack area
  const void* area;
  size_t stream;
  uint64_t at;
  std::string name;
};

std::vector<HostStream*> g_streams;
Clock g_host;
std::map<uintptr_t, size_t> g_live;
std::map<const void*, std::string> g_names;
std::vector<std::string> g_faults, g_launched;
std::vector<Use> g_uses;
std::vector<uint32_t> g_script;  // children of the coming shade launches
size_t g_next = 0, g_limit = ~(size_t)0;
uint32_t g_lost = 0;
Persist g_path;  // of the last path kernel
uint32_t g_path_waves = 0;
float g_ms = 1000.0f;

HostStream* stream_of(hipStream_t s) { return reinterpret_cast<HostStream*>(s); }
HostEvent* event_of(hipEvent_t e) { return reinterpret_cast<HostEvent*>(e); }

uint64_t step(hipStream_t s) {
  HostStream* h = stream_of(s);
  merge(h->clock, g_host);
  if (h->clock.size() <= h->id) h->clock.resize(h->id + 1);
  return ++h->clock[h->id];
}

bool live(const void* p, size_t bytes) {
  auto it = g_live.upper_bound((uintptr_t)p);
  if (it == g_live.begin()) return false;
  --it;
  return (uintptr_t)p + bytes <= it->first + it->second;
}
bool need(const std::string& kernel, const char* what, const void* p, size_t bytes) {
  if (live(p, bytes)) return true;
  g_faults.push_back(kernel + ": " + what + " is no device memory");
  return false;
}

// A launch that traverses with the stack area at `area`.
void traverses(const std::string& name, hipStream_t s, const void* area) {
  HostStream* h = stream_of(s);
  for (const Use& u : g_uses)
    if (u.area == area && u.stream != h->id && (h->clock.size() <= u.stream || h->clock[u.stream] < u.at))
      g_faults.push_back(name + ": may run beside " + u.name + " on the same stack area");
  g_uses.push_back(Use{area, h->id, h->clock[h->id], name});
}
const void* region(const Params& P, int r) {
  return P.stack_ovf + (size_t)r * (size_t)P.ovf_threads * (size_t)P.ovf_words;
}

template <class T>
const T& arg(void** a, int k) {
  return *reinterpret_cast<const T*>(a[k]);
}
uint32_t entries(const ChunkList& cl) { return cl.n[4]; }  // counts: chunks at 0..3, entries at 4..7

void emulate(const std::string& n, void** a, hipStream_t s) {
  auto is = [&](const char* k) { return n.find(k) != std::string::npos; };
  if (is("k_fill_u32") || is("k_fill_u64") || is("k_fill_f32")) {
    const size_t size = is("k_fill_u64") ? 8 : 4;
    char* p = arg<char*>(a, 0);
    const int64_t count = arg<int64_t>(a, 2);
    if (!need(n, "the range", p, size * (size_t)count)) return;
    for (int64_t i = 0; i < count; ++i) std::memcpy(p + size * i, a[1], size);
  } else if (is("k_slab_index")) {
    const uint2* slabs = arg<const uint2*>(a, 0);
    uint64_t* ctr = arg<uint64_t*>(a, 6);
    uint32_t chunks = 0, total = 0;
    for (uint32_t i = 0; i < arg<uint32_t>(a, 1); ++i) {
      chunks += (slabs[i].y + 63u) / 64u;
      total += slabs[i].y;
    }
    *arg<uint32_t*>(a, 4) = chunks;
    *arg<uint32_t*>(a, 5) = total;
    if (arg<int>(a, 7) >= 0) ctr[arg<int>(a, 7)] += total;
  } else if (is("k_stream_extend")) {
    traverses(n, s, region(arg<Stream>(a, 0).scenes[0], 0));
  } else if (is("k_stream_shadow")) {
    traverses(n, s, region(arg<Stream>(a, 0).scenes[0], 1));
  } else if (is("k_stream_refill")) {
    arg<Stream>(a, 0).ctl->status = 1u;
  } else if (is("k_extend")) {
    traverses(n, s, region(arg<Params>(a, 0), 0));
    arg<uint64_t*>(a, 6)[CTR_TRACED] += entries(arg<ChunkList>(a, 2));
  } else if (is("k_shadow")) {
    traverses(n, s, region(arg<Params>(a, 0), 1));
    need(n, "accum", arg<uint64_t*>(a, 5), 24);
    arg<uint64_t*>(a, 7)[CTR_STRACED] += entries(arg<ChunkList>(a, 3));
  } else if (is("k_shade")) {
    uint2* slabs = arg<uint2*>(a, 9);
    need(n, "accum", arg<uint64_t*>(a, 10), 24);
    const uint32_t out = g_next < g_script.size() ? g_script[g_next++] : 0u;
    for (int i = 0; i < PRT_SLAB_WAVES; ++i) slabs[i] = make_uint2(0u, i ? 0u : out);
    arg<uint64_t*>(a, 12)[CTR_EXT] += out;
    if (is("k_shadeILi2E")) {  // a recording pass: 64 entries per input chunk
      const int64_t samples = arg<Batch>(a, 1).n_pixels * arg<Params>(a, 0).spp;
      const AdjointRecs& r = arg<Adjoint>(a, 11).recs;
      *r.next = *r.first + 64u * (arg<int>(a, 2) ? (uint32_t)((samples + 63) / 64) : *arg<ChunkList>(a, 4).n);
    }
  } else if (is("k_nee")) {
    uint2* slabs = arg<uint2*>(a, 5);
    const uint32_t out = 3u * entries(arg<ChunkList>(a, 3));
    for (int i = 0; i < PRT_SLAB_WAVES; ++i) slabs[i] = make_uint2(0u, i ? 0u : out);
    arg<uint64_t*>(a, 6)[CTR_SHADOW] += out;
  } else if (is("k_path")) {
    const Persist& p = arg<Persist>(a, 0);
    g_path = p;
    const bool batch = is("k_pathILi0E"), queue = is("k_pathILi2E"), chain = is("k_pathILi3E");
    traverses(n, s, region(batch ? p.scenes[0] : arg<Params>(a, 1), 0));
    if (queue) {
      p.ctr[CTR_TRACED] += entries(p.cl);
    } else {
      const uint64_t samples = batch ? p.sample_base[p.n_scenes]
                                     : (uint64_t)p.n_samples * (chain ? p.chain.it1 - p.chain.it0 : 1u);
      if (!chain) need(n, "accum", p.accum, 24 * (size_t)samples);
      p.ctr[CTR_QUEUED] += samples - g_lost;
      p.ctr[CTR_TRACED] += samples - g_lost;
    }
  }
}

struct CallConfig {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local CallConfig g_call;

}  // namespace

extern "C" {

// ---- what a test asks
void hh_fail_above(size_t bytes) { g_limit = bytes; }
void hh_script(const uint32_t* children, int n) {
  g_script.assign(children, children + n);
  g_next = 0;
}
void hh_lose(uint32_t samples) { g_lost = samples; }
// chunks, chunks per claim and waves of the last path kernel
void hh_path(uint32_t* out) {
  out[0] = g_path.n_chunks;
  out[1] = g_path.claim;
  out[2] = g_path_waves;
}
int hh_faults(char* out, int size) {
  std::string all;
  for (auto& f : g_faults) all += f + "\n";
  std::snprintf(out, (size_t)size, "%s", all.c_str());
  return (int)g_faults.size();
}
void hh_launched(char* out, int size) {
  std::string all;
  for (auto& f : g_launched) all += f + "\n";
  std::snprintf(out, (size_t)size, "%s", all.c_str());
  g_launched.clear();
}

// ---- the runtime
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, uint3*, uint3*, dim3*, dim3*, int*) {
  g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
  g_call = CallConfig{grid, block, shared, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
  *grid = g_call.grid;
  *block = g_call.block;
  *shared = g_call.shared;
  *s = g_call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s) {
  step(s);
  const std::string& name = g_names[f];
  if (name.find("k_path") != std::string::npos) g_path_waves = grid.x * 4u;
  g_launched.push_back(name);
  emulate(name, args, s);
  return hipSuccess;
}

hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->major = 9;
  p->minor = 5;
  return hipSuccess;
}
hipError_t hipDeviceTotalMem(size_t* bytes, hipDevice_t) {
  *bytes = (size_t)8 << 30;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }

hipError_t hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  if (bytes > g_limit) return hipErrorOutOfMemory;
  void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == MAP_FAILED) return hipErrorOutOfMemory;
  g_live[(uintptr_t)m] = bytes;
  *p = m;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  for (HostStream* s : g_streams) merge(g_host, s->clock);
  auto it = g_live.find((uintptr_t)p);
  if (it == g_live.end()) {
    g_faults.push_back("hipFree of no device memory");
    return hipErrorInvalidValue;
  }
  munmap(p, it->second);
  g_live.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s) {
  step(s);
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) {
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  g_streams.push_back(new HostStream{g_streams.size(), {}});
  *s = reinterpret_cast<hipStream_t>(g_streams.back());
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  merge(g_host, stream_of(s)->clock);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  step(s);
  merge(stream_of(s)->clock, event_of(e)->clock);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new HostEvent());
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete event_of(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  step(s);
  event_of(e)->clock = stream_of(s)->clock;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  merge(g_host, event_of(e)->clock);
  return hipSuccess;
}
// every measured span is a quarter of the one before it
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = g_ms;
  g_ms *= 0.25f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(&g_call);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *x = reinterpret_cast<hipGraphExec_t>(&g_call);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  step(s);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

}  // extern "C"
