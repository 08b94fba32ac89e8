// The HIP host calls that libaslhip.so makes, on host memory: loaded before the
// library (tests/host_hip.py) they let its host side run without a GPU.
// Kernels do nothing but are logged; copies are copies and logged too; every
// launch takes a time that the test chooses, which events measure; a limit on
// the memory and the current device can be set.  Errors are HIP's: 2 out of memory, 400
// invalid handle (an event recorded on a stream of another device).
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace {
struct Dim {
  uint32_t x, y, z;
};
struct Launch {
  std::string name;
  uint32_t grid, block;
  void *stream;
};
struct Stream {
  int device;
  bool capturing = false;
  double captured = 0.;
};
struct Event {
  int device;
  double at = 0.;
};
struct Cost {
  std::string part;
  uint32_t block, below;  // workgroup size, number of workgroups below this (0: any)
  double ms;              // per workgroup
};

std::recursive_mutex mu;
std::map<const void *, std::string> names;
std::map<void *, size_t> allocated;
size_t used = 0, limit = 0;
int device = 0, last = 0, event_waits = 0;
double now = 0.;
bool no_new = false;
std::vector<Launch> launches;
struct Copy {
  char to, from;  // d device, p pinned, h other host memory
  size_t bytes;
};
std::vector<Copy> copies;
std::map<const void *, size_t> pinned;
std::vector<Cost> costs;
std::string text;
thread_local struct {
  Dim grid, block;
  size_t shared;
  void *stream;
} config;
int fail(int e) { return last = e; }
template <class M>
bool within(const M &m, const void *p) {
  auto it = m.upper_bound(const_cast<void *>(p));
  if (it == m.begin()) return false;
  --it;
  return static_cast<const char *>(p) < static_cast<const char *>(it->first) + it->second;
}
char kind(const void *p) { return within(allocated, p) ? 'd' : within(pinned, p) ? 'p' : 'h'; }
void copied(void *d, const void *s, size_t n) {
  if (copies.size() < copies.capacity() || !no_new) copies.push_back({kind(d), kind(s), n});
  std::memcpy(d, s, n);
}
}  // namespace

// the library's allocations on the host, which a test can make fail
void *operator new(size_t n) {
  void *p = no_new ? nullptr : std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

#define LOCK std::lock_guard<std::recursive_mutex> lock(mu)

extern "C" {

// what the tests call
void host_hip_device(int d) { device = d; }
void host_hip_limit(size_t n) { limit = n; }
size_t host_hip_used() { return used; }
int host_hip_event_waits() { return event_waits; }
void host_hip_no_new(int on) { no_new = on != 0; }
void host_hip_cost(const char *part, unsigned block, unsigned below, double ms) { costs.push_back({part, block, below, ms}); }
void host_hip_forget() {
  launches.clear();
  copies.clear();
}
const char *host_hip_copies() {  // "to from bytes" lines
  text.clear();
  for (const auto &c : copies) text += std::string(1, c.to) + " " + c.from + " " + std::to_string(c.bytes) + "\n";
  return text.c_str();
}
const char *host_hip_launches() {  // "kernel grid block" lines
  text.clear();
  for (const auto &l : launches) text += l.name + " " + std::to_string(l.grid) + " " + std::to_string(l.block) + "\n";
  return text.c_str();
}

// registration
void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  LOCK;
  names[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void *stream) {
  config = {grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *shared, void **stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return 0;
}

// devices and errors
int hipGetDevice(int *d) {
  *d = device;
  return 0;
}
int hipSetDevice(int d) {
  device = d;
  return 0;
}
int hipGetLastError() {
  const int e = last;
  last = 0;
  return e;
}
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : e == 400 ? "invalid resource handle" : "error"; }

// memory
int hipMalloc(void **p, size_t n) {
  LOCK;
  *p = nullptr;
  if (limit && used + n > limit) return fail(2);
  *p = std::malloc(n);
  if (!*p) return fail(2);
  allocated[*p] = n;
  used += n;
  return 0;
}
int hipFree(void *p) {
  LOCK;
  auto it = allocated.find(p);
  if (it == allocated.end()) return p ? fail(1) : 0;
  used -= it->second;
  allocated.erase(it);
  std::free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) {
  LOCK;
  if (!(*p = std::malloc(n))) return fail(2);
  pinned[*p] = n;
  return 0;
}
int hipHostFree(void *p) {
  LOCK;
  pinned.erase(p);
  std::free(p);
  return 0;
}
int hipPointerGetAttributes(int *type, const void *p) {  // the first member of hipPointerAttribute_t
  LOCK;
  *type = kind(p) == 'd' ? 2 : kind(p) == 'p' ? 1 : 0;
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  LOCK;
  copied(d, s, n);
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
  LOCK;
  copied(d, s, n);
  return 0;
}
int hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int) {
  for (size_t i = 0; i < h; ++i) std::memcpy(static_cast<char *>(d) + i * dp, static_cast<const char *>(s) + i * sp, w);
  return 0;
}
int hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return 0;
}
int hipGetSymbolAddress(void **p, const void *) {
  *p = nullptr;
  return fail(1);
}

// streams and events
int hipStreamCreate(void **s) {
  *s = new Stream{device};
  return 0;
}
int hipStreamDestroy(void *s) {
  delete static_cast<Stream *>(s);
  return 0;
}
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipStreamGetDevice(void *s, int *d) {
  *d = s ? static_cast<Stream *>(s)->device : device;
  return 0;
}
int hipEventCreateWithFlags(void **e, unsigned) {
  *e = new Event{device};
  return 0;
}
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) {
  delete static_cast<Event *>(e);
  return 0;
}
int hipEventRecord(void *e, void *s) {
  LOCK;
  if (s && static_cast<Stream *>(s)->device != static_cast<Event *>(e)->device) return fail(400);
  static_cast<Event *>(e)->at = now;
  return 0;
}
int hipEventSynchronize(void *) {
  LOCK;
  ++event_waits;
  return 0;
}
int hipEventElapsedTime(float *ms, void *a, void *b) {
  *ms = static_cast<float>(static_cast<Event *>(b)->at - static_cast<Event *>(a)->at);
  return 0;
}

// launches
int hipLaunchKernel(const void *f, Dim grid, Dim block, void **, size_t, void *stream) {
  LOCK;
  const std::string &name = names[f];
  launches.push_back({name, grid.x, block.x, stream});
  double ms = 0.;
  for (const auto &c : costs)  // later rules win
    if (name.find(c.part) != std::string::npos && (!c.block || c.block == block.x) && (!c.below || grid.x < c.below))
      ms = c.ms * grid.x;
  Stream *s = static_cast<Stream *>(stream);
  if (s && s->capturing)
    s->captured += ms;
  else
    now += ms;
  return 0;
}
int hipStreamBeginCapture(void *s, int) {
  static_cast<Stream *>(s)->capturing = true;
  static_cast<Stream *>(s)->captured = 0.;
  return 0;
}
int hipStreamEndCapture(void *s, void **g) {
  static_cast<Stream *>(s)->capturing = false;
  *g = new double(static_cast<Stream *>(s)->captured);
  return 0;
}
int hipGraphInstantiate(void **x, void *g, void *, char *, size_t) {
  *x = new double(*static_cast<double *>(g));
  return 0;
}
int hipGraphDestroy(void *g) {
  delete static_cast<double *>(g);
  return 0;
}
int hipGraphExecDestroy(void *x) {
  delete static_cast<double *>(x);
  return 0;
}
int hipGraphLaunch(void *x, void *) {
  LOCK;
  now += *static_cast<double *>(x);
  return 0;
}

}  // extern "C"
