// hip_stand_in.cpp -- the part of the HIP runtime that the library calls, on host memory:
// allocations come from malloc, copies are done in place, kernels and graphs are counted
// and not run.  Loaded before the library (RTLD_GLOBAL), it takes the runtime's place, so
// that the library's host code runs without a GPU and a test can make any call fail
// (stand_in_fail), look at what was asked for (stand_in_count, stand_in_bytes,
// stand_in_loaded_kernels) and have two devices.  Streams and events belong to the device that was current when they were
// made; a launch or a record with another device current fails, as in the runtime.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>

namespace {

constexpr int kInvalidValue = 1, kOutOfMemory = 2, kInvalidHandle = 400, kUnknown = 999;
constexpr size_t kMemory = size_t(288) << 30;

struct Handle {
  int device;
};
struct Block {
  size_t bytes;
  bool pinned;
};

std::mutex lock;
std::map<std::string, long long> calls;
std::map<std::string, std::pair<long long, int>> failures;  // call: fail from its n-th on, with this error
std::unordered_map<void*, Block> blocks;
size_t live[2] = {0, 0}, largest = 0;  // device, pinned
struct Module {
  int kernels = 0;
  bool loaded = false;
};
std::unordered_map<const void*, Module*> kernels;
long long loaded_kernels = 0;
thread_local int current = 0;
thread_local int last = 0;

int enter(const char* name) {
  std::lock_guard<std::mutex> g(lock);
  const long long n = ++calls[name];
  auto f = failures.find(name);
  last = f != failures.end() && n >= f->second.first ? f->second.second : last;
  return f != failures.end() && n >= f->second.first ? f->second.second : 0;
}
int done(int e) {
  if (e) last = e;
  return e;
}
int allocate(void** p, size_t bytes, bool pinned) {
  *p = std::malloc(bytes ? bytes : 1);
  if (!*p) return done(kOutOfMemory);
  std::lock_guard<std::mutex> g(lock);
  blocks[*p] = {bytes, pinned};
  live[pinned] += bytes;
  if (!pinned && bytes > largest) largest = bytes;
  return 0;
}
int release(void* p) {
  if (!p) return 0;
  {
    std::lock_guard<std::mutex> g(lock);
    auto b = blocks.find(p);
    if (b == blocks.end()) return done(kInvalidValue);
    live[b->second.pinned] -= b->second.bytes;
    blocks.erase(b);
  }
  std::free(p);
  return 0;
}
int make(void** h) {
  *h = new Handle{current};
  return 0;
}
int drop(void* h) {
  delete static_cast<Handle*>(h);
  return 0;
}
// a code object is loaded whole, at the first use of a kernel in it
void load(const void* kernel) {
  std::lock_guard<std::mutex> g(lock);
  auto k = kernels.find(kernel);
  if (k == kernels.end() || k->second->loaded) return;
  k->second->loaded = true;
  loaded_kernels += k->second->kernels;
}
int here(void* h) { return h && static_cast<Handle*>(h)->device != current ? done(kInvalidHandle) : 0; }

}  // namespace

#define ENTER(name)                   \
  do {                                \
    if (int e_ = enter(name)) return e_; \
  } while (0)

extern "C" {

// the test's side
void stand_in_fail(const char* call, long long from, int error) {
  std::lock_guard<std::mutex> g(lock);
  if (from > 0)
    failures[call] = {calls[call] + from, error};
  else
    failures.erase(call);
}
long long stand_in_count(const char* call) {
  std::lock_guard<std::mutex> g(lock);
  return calls[call];
}
long long stand_in_bytes(int what) {  // 0 device, 1 pinned, 2 the largest device allocation
  std::lock_guard<std::mutex> g(lock);
  return (long long)(what == 2 ? largest : live[what]);
}
int stand_in_device() { return current; }
long long stand_in_loaded_kernels() { return loaded_kernels; }

// the runtime's
int hipGetDevice(int* d) {
  ENTER("hipGetDevice");
  *d = current;
  return 0;
}
int hipSetDevice(int d) {
  ENTER("hipSetDevice");
  if (d < 0 || d > 1) return done(kInvalidValue);
  current = d;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
  ENTER("hipDeviceGetAttribute");
  *v = 160 * 1024;
  return 0;
}
int hipGetDevicePropertiesR0600(void*, int) { return kUnknown; }
int hipMemGetInfo(size_t* f, size_t* t) {
  ENTER("hipMemGetInfo");
  *f = *t = kMemory;
  return 0;
}
const char* hipGetErrorString(int e) {
  return e == 0 ? "no error" : e == kOutOfMemory ? "out of memory" : e == kInvalidHandle ? "invalid handle" : "stand-in error";
}
int hipGetLastError() {
  const int e = last;
  last = 0;
  return e;
}
int hipMalloc(void** p, size_t n) {
  ENTER("hipMalloc");
  return allocate(p, n, false);
}
int hipFree(void* p) {
  ENTER("hipFree");
  return release(p);
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  ENTER("hipHostMalloc");
  return allocate(p, n, true);
}
int hipHostFree(void* p) {
  ENTER("hipHostFree");
  return release(p);
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  ENTER("hipMemcpy");
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  ENTER("hipMemcpyAsync");
  std::memcpy(d, s, n);
  return 0;
}
int hipMemset(void* d, int v, size_t n) {
  ENTER("hipMemset");
  std::memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  ENTER("hipMemsetAsync");
  std::memset(d, v, n);
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) {
  ENTER("hipStreamCreateWithFlags");
  return make(s);
}
int hipStreamDestroy(void* s) {
  ENTER("hipStreamDestroy");
  return drop(s);
}
int hipStreamSynchronize(void*) {
  ENTER("hipStreamSynchronize");
  return 0;
}
int hipStreamWaitEvent(void*, void*, unsigned) {
  ENTER("hipStreamWaitEvent");
  return 0;
}
int hipGetStreamDeviceId(void* s) { return s ? static_cast<Handle*>(s)->device : current; }
int hipEventCreate(void** e) {
  ENTER("hipEventCreate");
  return make(e);
}
int hipEventCreateWithFlags(void** e, unsigned) {
  ENTER("hipEventCreateWithFlags");
  return make(e);
}
int hipEventDestroy(void* e) {
  ENTER("hipEventDestroy");
  return drop(e);
}
int hipEventRecord(void* e, void* s) {
  ENTER("hipEventRecord");
  if (s && static_cast<Handle*>(e)->device != static_cast<Handle*>(s)->device) return done(kInvalidHandle);
  return 0;
}
int hipEventSynchronize(void*) {
  ENTER("hipEventSynchronize");
  return 0;
}
int hipEventElapsedTime(float* ms, void*, void*) {
  ENTER("hipEventElapsedTime");
  *ms = 1.0f;
  return 0;
}
int hipStreamBeginCapture(void*, int) {
  ENTER("hipStreamBeginCapture");
  return 0;
}
int hipStreamEndCapture(void*, void** g) {
  ENTER("hipStreamEndCapture");
  return make(g);
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
  ENTER("hipGraphInstantiate");
  return make(x);
}
int hipGraphLaunch(void* x, void*) {
  ENTER("hipGraphLaunch");
  return x ? 0 : done(kInvalidValue);
}
int hipGraphExecDestroy(void* x) {
  ENTER("hipGraphExecDestroy");
  return drop(x);
}
int hipGraphDestroy(void* x) {
  ENTER("hipGraphDestroy");
  return drop(x);
}
int hipFuncSetAttribute(const void* f, int, int) {
  ENTER("hipFuncSetAttribute");
  load(f);
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int, size_t) {
  ENTER("hipOccupancyMaxActiveBlocksPerMultiprocessor");
  load(f);
  *n = 2;
  return 0;
}
struct Dim3 {
  unsigned x, y, z;
};
static thread_local struct {
  Dim3 grid, block;
  size_t lds;
  void* stream;
} pushed;
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void* s) {
  pushed = {g, b, lds, s};
  return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** s) {
  *g = pushed.grid;
  *b = pushed.block;
  *lds = pushed.lds;
  *s = pushed.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t, void* s) {
  ENTER("hipLaunchKernel");
  load(f);
  return here(s);
}
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(new Module); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void** m, const void* f, char*, const char*, unsigned, void*, void*, void*, void*, int*) {
  std::lock_guard<std::mutex> g(lock);
  kernels[f] = reinterpret_cast<Module*>(m);
  ++kernels[f]->kernels;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
