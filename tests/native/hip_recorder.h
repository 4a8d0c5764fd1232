// A HIP runtime that runs nothing: it records which calls order which kernel
// launches, so that the library's host code can be checked on the CPU for
// launches that share memory without an order between them, for calls that an
// ongoing capture forbids, and for waits for other streams.
//
// Every stream has a vector clock (how far it has gone on itself and on each
// stream it has waited for), the host one of its own (what it has waited for;
// the threads of a check run one after the other).  hipStreamPerThread is
// another stream in every thread.  Launches on a capturing stream are recorded,
// not run.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdint>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "geometry.h"

namespace rec {
using Clock = std::map<int, unsigned>;
inline void merge(Clock& a, const Clock& b) {
  for (auto& kv : b) a[kv.first] = std::max(a[kv.first], kv.second);
}
struct Stream {
  int id = 0;
  Clock clock;
  unsigned seq = 0;
  bool capturing = false;
  hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
  std::thread::id by;  // the thread that captures
};
struct Event {
  Clock clock;
  bool captured = false;
};
struct Launch {
  std::string name;
  int stream;
  unsigned seq;
  Clock before;
  const char *in, *out, *H;
  long long hstride;
  int ntotal;
};
inline std::vector<Stream*> streams;
inline std::map<std::thread::id, Stream*> per_thread;
inline Clock host;
inline std::map<const char*, size_t> allocs;
inline size_t held = 0, alloc_limit = ~size_t(0);  // bytes of hipMalloc, and the most of them
inline std::vector<Launch> launches;
inline unsigned captured_launches = 0, device_waits = 0;
inline std::vector<std::string> faults;
inline std::map<std::string, std::string*> functions;
inline thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
inline thread_local hipError_t last = hipSuccess;

inline Stream* add_stream() {
  Stream* s = new Stream;
  s->id = (int)streams.size();
  streams.push_back(s);
  return s;
}
inline Stream* at(hipStream_t s) {
  if (streams.empty()) add_stream();  // 0: the null stream
  if (s == nullptr) return streams[0];
  if (s == hipStreamPerThread) {
    Stream*& t = per_thread[std::this_thread::get_id()];
    if (!t) t = add_stream();
    return t;
  }
  return reinterpret_cast<Stream*>(s);
}
inline hipStream_t new_stream() {
  at(nullptr);
  return reinterpret_cast<hipStream_t>(add_stream());
}
inline hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
// a call that a capture forbids (unless the calling thread has relaxed its mode)
inline bool forbidden(const char* what) {
  for (Stream* s : streams)
    if (s->capturing && mode != hipStreamCaptureModeRelaxed &&
        (s->by == std::this_thread::get_id() || (s->mode == hipStreamCaptureModeGlobal && mode == hipStreamCaptureModeGlobal))) {
      faults.push_back(std::string(what) + " during a capture");
      return true;
    }
  return false;
}
inline void wait_all() {
  ++device_waits;
  for (Stream* s : streams) merge(host, s->clock);
}
inline void begin_capture(hipStream_t s, hipStreamCaptureMode m = hipStreamCaptureModeGlobal) {
  at(s)->capturing = true;
  at(s)->mode = m;
  at(s)->by = std::this_thread::get_id();
}
inline void end_capture(hipStream_t s) { at(s)->capturing = false; }
inline char* alloc(size_t bytes) {
  static char* next = reinterpret_cast<char*>(uintptr_t(1) << 40);  // addresses only, never touched
  char* p = next;
  next += (bytes + 4095) / 4096 * 4096 + 4096;
  allocs[p] = bytes;
  return p;
}
// base address of the allocation p lies in
inline const char* base(const char* p) {
  auto it = allocs.upper_bound(p);
  if (it == allocs.begin()) return nullptr;
  --it;
  return p < it->first + it->second ? it->first : nullptr;
}
inline bool ordered(const Launch& a, const Launch& b) {
  auto it = b.before.find(a.stream);
  return it != b.before.end() && it->second >= a.seq;
}
// pairs of launches that meet in an allocation, one of them writing, without an order
inline unsigned races(bool print = true) {
  unsigned n = 0;
  for (size_t j = 0; j < launches.size(); ++j)
    for (size_t i = 0; i < j; ++i) {
      const Launch &a = launches[i], &b = launches[j];
      if (a.stream == b.stream || ordered(a, b)) continue;
      auto meet = [](const char* p, const char* q) { return p && q && base(p) && base(p) == base(q); };
      if (meet(a.out, b.out) || meet(a.out, b.in) || meet(a.in, b.out) || meet(a.out, b.H) || meet(a.H, b.out)) {
        if (print && n == 0)
          printf("unordered: %s on stream %d and %s on stream %d\n", a.name.c_str(), a.stream, b.name.c_str(), b.stream);
        ++n;
      }
    }
  return n;
}
}  // namespace rec

// ---- the runtime calls of the library ---------------------------------------
#define REC extern "C" __attribute__((visibility("default"))) hipError_t
REC hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
REC hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  memset(p, 0, sizeof *p);
  snprintf(p->name, sizeof p->name, "recorder");
  snprintf(p->gcnArchName, sizeof p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
REC hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 1, hipSuccess; }
REC hipSetDevice(int) { return hipSuccess; }
REC hipGetLastError() {
  const hipError_t e = rec::last;
  rec::last = hipSuccess;
  return e;
}
extern "C" const char* hipGetErrorString(hipError_t) { return "recorded error"; }
REC hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  if (rec::forbidden("hipMalloc")) return rec::ret(hipErrorStreamCaptureUnsupported);
  if (rec::held + bytes > rec::alloc_limit) return rec::ret(hipErrorOutOfMemory);
  rec::held += bytes;
  return *p = rec::alloc(bytes), hipSuccess;
}
REC hipFree(void* p) {
  if (!p) return hipSuccess;
  if (rec::forbidden("hipFree")) return rec::ret(hipErrorStreamCaptureUnsupported);
  rec::wait_all();
  auto it = rec::allocs.find((char*)p);
  if (it == rec::allocs.end()) return rec::faults.push_back("hipFree of what is not allocated"), hipSuccess;
  rec::held -= it->second;
  rec::allocs.erase(it);
  return hipSuccess;
}
REC hipHostMalloc(void** p, size_t bytes, unsigned) { return *p = malloc(bytes), hipSuccess; }
REC hipHostFree(void* p) { return free(p), hipSuccess; }
REC hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
REC hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return rec::wait_all(), hipSuccess; }
REC hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
REC hipMemset(void*, int, size_t) { return rec::wait_all(), hipSuccess; }
REC hipDeviceSynchronize() {
  for (rec::Stream* s : rec::streams)  // (in every mode)
    if (s->capturing) {
      rec::faults.push_back("hipDeviceSynchronize during a capture");
      return rec::ret(hipErrorStreamCaptureUnsupported);
    }
  return rec::wait_all(), hipSuccess;
}
REC hipStreamCreate(hipStream_t* s) { return *s = rec::new_stream(), hipSuccess; }
REC hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = rec::new_stream(), hipSuccess; }
REC hipStreamDestroy(hipStream_t s) { return rec::merge(rec::host, rec::at(s)->clock), hipSuccess; }
REC hipStreamSynchronize(hipStream_t s) {
  if (rec::at(s)->capturing) return rec::ret(hipErrorStreamCaptureUnsupported);
  return rec::merge(rec::host, rec::at(s)->clock), hipSuccess;
}
REC hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = rec::at(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
REC hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) { return std::swap(*m, rec::mode), hipSuccess; }
REC hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { return rec::begin_capture(s, m), hipSuccess; }
REC hipStreamEndCapture(hipStream_t s, hipGraph_t* g) { return rec::end_capture(s), *g = nullptr, hipSuccess; }
REC hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { return *e = nullptr, hipSuccess; }
REC hipGraphDestroy(hipGraph_t) { return hipSuccess; }
REC hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
REC hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
REC hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(new rec::Event), hipSuccess; }
REC hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
REC hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<rec::Event*>(e), hipSuccess; }
REC hipEventRecord(hipEvent_t e, hipStream_t s) {
  rec::Event* ev = reinterpret_cast<rec::Event*>(e);
  ev->captured = rec::at(s)->capturing;
  ev->clock = rec::at(s)->clock;
  return hipSuccess;
}
REC hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  rec::Event* ev = reinterpret_cast<rec::Event*>(e);
  if (ev->captured && !rec::at(s)->capturing) {
    rec::faults.push_back("a stream joined another one's capture");
    rec::at(s)->capturing = true;
  }
  return rec::merge(rec::at(s)->clock, ev->clock), hipSuccess;
}
REC hipEventSynchronize(hipEvent_t e) { return rec::merge(rec::host, reinterpret_cast<rec::Event*>(e)->clock), hipSuccess; }
REC hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
REC hipModuleLoad(hipModule_t* m, const char*) { return *m = reinterpret_cast<hipModule_t>(1), hipSuccess; }
REC hipModuleUnload(hipModule_t) { return hipSuccess; }
REC hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
  std::string*& s = rec::functions[name];
  if (!s) s = new std::string(name);
  return *f = reinterpret_cast<hipFunction_t>(s), hipSuccess;
}
REC hipModuleGetGlobal(hipDeviceptr_t* p, size_t* bytes, hipModule_t, const char*) {
  *bytes = (size_t)cfgeo::noalloc_scratch_bytes;
  return *p = rec::alloc(*bytes), hipSuccess;
}
REC hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, hipFunction_t, int, size_t) { return *n = 1, hipSuccess; }
REC hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                          hipStream_t s, void** args, void**) {
  const std::string& name = *reinterpret_cast<std::string*>(f);
  rec::Stream* st = rec::at(s);
  if (st->capturing) return ++rec::captured_launches, hipSuccess;
  rec::merge(st->clock, rec::host);
  rec::Launch l{name, st->id, ++st->seq, st->clock, nullptr, nullptr, nullptr, 0, 0};
  st->clock[st->id] = st->seq;
  for (const char* p : {"cf_row_", "cf_coly", "cf_colz", "cf_cube_", "cf_plane_", "cf_xy1_", "cf_mid", "cf_rows_", "cf_fft2_"})
    if (name.rfind(p, 0) == 0) {  // the argument list of the passes: in, out, H, tw, hstride, scale, ntotal
      l.in = *(const char**)args[0];
      l.out = *(const char**)args[1];
      l.H = *(const char**)args[2];
      l.hstride = *(long long*)args[4];
      l.ntotal = *(int*)args[6];
      rec::launches.push_back(l);
      break;
    }
  return hipSuccess;
}
