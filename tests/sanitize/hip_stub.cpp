// A stand-in for the HIP runtime, for runs of the library's host code on the
// CPU (tests/test_host_runtime.py): device memory is host memory, kernels do
// nothing, and a stream keeps its operations until something waits for them.
// An asynchronous copy reads a host source at the call, as the runtime does with
// pageable memory, and writes a host destination only when the stream is waited
// for.  It is stricter than a real runtime in one point: work counts as retired
// only by a wait for the stream that it was put on (an event wait runs it, but
// does not retire it).  What it objects to is counted in stub_faults() and
// printed.
#include "hip_stub.hpp"

#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

namespace {

struct Exec {
  int unretired = 0;  // launches whose stream has not been waited for
};
struct Event;
struct Stream {
  bool capturing = false, origin = false;
  bool unjoined = false;  // captured work that the origin does not wait for
  std::deque<std::function<void()>> todo;
  std::vector<Exec *> launched;
};
struct Event {
  Stream *on = nullptr;      // stream of the last record
  size_t left = 0;           // operations of `on` up to the record
  bool captured = false;
  double ms = 0.0;
};
struct Graph {
  int nodes = 0;
};

std::recursive_mutex mu;
int inside = 0;  // calls into this file
struct Guard {
  Guard() {
    mu.lock();
    ++inside;
  }
  ~Guard() {
    --inside;
    mu.unlock();
  }
};
Stream null_stream;
std::set<Stream *> streams{&null_stream};
std::set<void *> execs;
std::map<void *, size_t> device;
size_t cap = size_t(1) << 40, held = 0, peak = 0;
int faults = 0;
long launches = 0, graphs = 0, fail_in = 0;
double clock_ms = 0.0;
Graph *building = nullptr;
std::thread::id builder;       // the thread that captures (thread-local mode)
std::vector<Stream *> joined;  // streams that the capture reached
hipError_t last = hipSuccess;
dim3 cfg_grid, cfg_block;
size_t cfg_shared;
hipStream_t cfg_stream;

void fault(const char *what) {
  ++faults;
  std::fprintf(stderr, "hip_stub: %s\n", what);
  if (std::getenv("HIP_STUB_ABORT")) std::abort();
}
hipError_t fail(hipError_t e) { return last = e; }
Stream *of(hipStream_t s) {
  Stream *p = s ? reinterpret_cast<Stream *>(s) : &null_stream;
  if (!streams.count(p)) {
    fault("call on a stream that does not exist");
    return &null_stream;
  }
  return p;
}
void run(Stream *s, size_t n) {
  for (; n > 0 && !s->todo.empty(); --n) {
    auto f = std::move(s->todo.front());
    s->todo.pop_front();
    f();
  }
}
void retire(Stream *s) {
  run(s, s->todo.size());
  for (Exec *e : s->launched)
    if (execs.count(e)) --e->unretired;
  s->launched.clear();
}
void retire_all() {
  for (Stream *s : streams) retire(s);
}
// Whether p is inside an allocation.
bool on_device(const void *p) {
  auto it = device.upper_bound(const_cast<void *>(p));
  if (it == device.begin()) return false;
  --it;
  return (const char *)p < (const char *)it->first + it->second;
}
// An operation on a stream: a node while it is captured.
void put(Stream *s, std::function<void()> f) {
  if (s->capturing) {
    ++building->nodes;
    s->unjoined = !s->origin;
  } else {
    s->todo.push_back(std::move(f));
  }
}
std::map<const void *, std::string> &names() {  // filled before main
  static auto *m = new std::map<const void *, std::string>;
  return *m;
}
std::vector<std::string> launched;
void unsafe_in_capture(const char *what) {
  if (building && builder == std::this_thread::get_id()) fault(what);
}

}  // namespace

int stub_faults() { return faults; }
bool stub_inside() { return inside > 0; }
void stub_set_memory(size_t bytes) { cap = bytes; }
size_t stub_memory_held() { return held; }
size_t stub_memory_peak() { return peak; }
void stub_reset_peak() { peak = held; }
long stub_launches() { return launches; }
std::vector<std::string> stub_take_launches() {
  Guard l;
  return std::move(launched);
}
long stub_graphs() { return graphs; }
void stub_fail_launch(long n) { fail_in = n; }

extern "C" {

hipError_t hipMalloc(void **p, size_t n) {
  Guard l;
  unsafe_in_capture("hipMalloc during a capture");
  if (held + n > cap) return fail(hipErrorOutOfMemory);
  *p = std::calloc(1, n ? n : 1);
  device[*p] = n;
  held += n;
  peak = peak > held ? peak : held;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  Guard l;
  if (!p) return hipSuccess;
  unsafe_in_capture("hipFree during a capture");
  retire_all();
  auto it = device.find(p);
  if (it == device.end()) {
    fault("hipFree of memory that is not allocated");
    return fail(hipErrorInvalidValue);
  }
  held -= it->second;
  device.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return hipFree(p); }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  Guard l;
  *t = cap;
  *f = cap - held;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  Guard l;
  if (on_device(s)) {
    put(of(st), [=] { std::memcpy(d, s, n); });
  } else {
    std::vector<char> copy((const char *)s, (const char *)s + n);
    put(of(st), [d, copy] { std::memcpy(d, copy.data(), copy.size()); });
  }
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  Guard l;
  unsafe_in_capture("hipMemcpy during a capture");
  retire(&null_stream);
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind, hipStream_t st) {
  Guard l;
  put(of(st), [=] {
    for (size_t i = 0; i < h; ++i) std::memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
  });
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
  Guard l;
  if (of(st)->capturing) fault("hipMemsetAsync during a capture");
  put(of(st), [=] { std::memset(d, v, n); });
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  Guard l;
  retire(&null_stream);
  std::memset(d, v, n);
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  Guard l;
  Stream *p = new Stream;
  streams.insert(p);
  *s = reinterpret_cast<hipStream_t>(p);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  Guard l;
  Stream *p = of(s);
  if (p->capturing) fault("hipStreamDestroy during a capture");
  retire(p);
  if (p != &null_stream) {
    streams.erase(p);
    delete p;
  }
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  Guard l;
  Stream *p = of(s);
  if (p->capturing) fault("hipStreamSynchronize of a stream that is captured");
  retire(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  Guard l;
  *e = reinterpret_cast<hipEvent_t>(new Event);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<Event *>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t ev, hipStream_t s) {
  Guard l;
  Event *e = reinterpret_cast<Event *>(ev);
  e->on = of(s);
  e->captured = e->on->capturing;
  e->left = e->on->todo.size();
  e->ms = clock_ms += 1.0;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t ev) {
  Guard l;
  Event *e = reinterpret_cast<Event *>(ev);
  if (e->captured) fault("hipEventSynchronize of a captured event");
  if (e->on && streams.count(e->on)) run(e->on, e->left);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
  // times that differ from call to call, so that variants lose and win in turn
  static unsigned n = 0;
  *ms = (float)(reinterpret_cast<Event *>(b)->ms - reinterpret_cast<Event *>(a)->ms) +
        (float)((++n * 2654435761u) >> 24) / 64.f;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t ev, unsigned) {
  Guard l;
  Stream *p = of(s);
  Event *e = reinterpret_cast<Event *>(ev);
  if (e->captured && building) {
    if (!p->capturing) {
      p->capturing = p->unjoined = true;
      joined.push_back(p);
    }
    if (p->origin && e->on) e->on->unjoined = false;
    return hipSuccess;
  }
  if (p->capturing) fault("captured stream waits for an event from outside the capture");
  Stream *on = e->on;
  const size_t left = e->left;
  if (on && on != p) p->todo.push_back([on, left] { if (streams.count(on)) run(on, left); });
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  Guard l;
  Stream *p = of(s);
  if (building || s == nullptr) fault("capture begun inside another, or on the null stream");
  building = new Graph;
  ++graphs;
  builder = std::this_thread::get_id();
  p->capturing = p->origin = true;
  joined.clear();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
  Guard l;
  Stream *p = of(s);
  if (!p->capturing || !p->origin || !building) {
    fault("hipStreamEndCapture without a capture");
    return fail(hipErrorInvalidValue);
  }
  for (Stream *j : joined) {
    if (j->unjoined) fault("hipStreamEndCapture with a stream that was not joined");
    j->capturing = j->unjoined = false;
  }
  joined.clear();
  p->capturing = p->origin = false;
  *g = reinterpret_cast<hipGraph_t>(building);
  building = nullptr;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
  Guard l;
  *st = of(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  Guard l;
  if (fail_in > 0 && --fail_in == 0) return hipErrorInvalidValue;
  Exec *p = new Exec;
  execs.insert(p);
  *e = reinterpret_cast<hipGraphExec_t>(p);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  --graphs;
  delete reinterpret_cast<Graph *>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  Guard l;
  Exec *p = reinterpret_cast<Exec *>(e);
  if (!execs.count(p)) {
    fault("hipGraphExecDestroy of no executable");
    return fail(hipErrorInvalidValue);
  }
  if (p->unretired) fault("hipGraphExecDestroy before its stream was waited for");
  execs.erase(p);
  delete p;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  Guard l;
  Exec *p = reinterpret_cast<Exec *>(e);
  Stream *st = of(s);
  if (!execs.count(p)) fault("hipGraphLaunch of no executable");
  if (st->capturing) fault("hipGraphLaunch on a captured stream");
  ++p->unretired;
  st->launched.push_back(p);
  st->todo.push_back([p] { if (!execs.count(p)) fault("executable destroyed before it ran"); });
  return hipSuccess;
}

hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetSymbolAddress(void **p, const void *sym) {
  *p = const_cast<void *>(sym);
  return hipSuccess;
}

hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
  cfg_grid = g;
  cfg_block = b;
  cfg_shared = sh;
  cfg_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s) {
  *g = cfg_grid;
  *b = cfg_block;
  *sh = cfg_shared;
  *s = cfg_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t shared, hipStream_t s) {
  Guard l;
  if (!g.x || !g.y || !g.z || g.y > 65535 || g.z > 65535) fault("launch grid out of range");
  if (!b.x || b.x * b.y * b.z > 1024) fault("launch block out of range");
  if (shared > 160 * 1024) fault("launch with more LDS than a CU has");
  ++launches;
  auto it = names().find(f);
  launched.push_back(it == names().end() ? "?" : it->second);
  if (fail_in > 0 && --fail_in == 0) return fail(hipErrorInvalidValue);
  put(of(s), [] {});
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *,
                           void *, void *, int *) {
  names()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
int roctxRangePushA(const char *) { return 0; }
int roctxRangePop() { return 0; }

}  // extern "C"
