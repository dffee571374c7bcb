// A HIP runtime that launches nothing, for CPU tests of the library's host
// side: loaded before libimpactz_hip.so, it takes the calls the library makes
// and keeps account of them.
// - Device memory is host memory, up to a capacity the test sets; freeing a
//   block takes as long as the test says.
// - A kernel launch counts as work queued on its stream and is listed by its
//   kernel's name.  Synchronizing a stream completes its work and the work its
//   event waits made it follow; nothing else does, hipFree included (so a
//   library that relied on it shows work left over).
// - One launch can leave an error for the next hipGetLastError (the kernel is
//   queued all the same), as another user of the thread's last error would.
#include <chrono>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {
constexpr int kOk = 0, kInvalid = 1, kOutOfMemory = 2, kUnknown = 999;

using Clock = std::map<int, int64_t>;  // stream -> work up to this ticket

struct Stream {
  int id;
  Clock follows;  // other streams' work its queue waits for
};
struct Event {
  Clock seen;
};

struct State {
  std::mutex mu;
  std::map<const void *, std::string> kernels;
  std::vector<std::string> launched;
  std::map<void *, size_t> blocks;
  size_t held = 0, capacity = (size_t)1 << 40, peak = 0;
  int free_ms = 0;
  int next_stream = 1;
  Clock queued, done;
  std::string fail_kernel;
  size_t fail_bytes = 0;
  int last_error = kOk;
  // a value written into every copy from the device of this size
  size_t poke_bytes = 0, poke_at = 0;
  int64_t poke_value = 0;
};

State &st() {
  static State *s = new State;
  return *s;
}

void merge(Clock &to, const Clock &from) {
  for (const auto &p : from)
    if (to[p.first] < p.second) to[p.first] = p.second;
}

void enqueue(Stream *s) {
  if (s) st().queued[s->id]++;
}

struct Dim3 {
  unsigned x, y, z;
};
struct Config {
  Dim3 grid, block;
  size_t shared;
  Stream *stream;
};
thread_local Config config;
}  // namespace

extern "C" {

// ------------------------------------------------------- what tests ask
void fake_capacity(size_t bytes) { st().capacity = bytes; }
void fake_free_delay(int ms) { st().free_ms = ms; }
void fake_fail_kernel(const char *name) { st().fail_kernel = name; }
// allocations of this many bytes fail (0: none does)
void fake_fail_alloc(size_t bytes) { st().fail_bytes = bytes; }
void fake_poke(size_t bytes, size_t at, int64_t value) {
  st().poke_bytes = bytes;
  st().poke_at = at;
  st().poke_value = value;
}
size_t fake_held() {
  std::lock_guard<std::mutex> lock(st().mu);
  return st().held;
}
size_t fake_peak() {
  std::lock_guard<std::mutex> lock(st().mu);
  return st().peak;
}
int64_t fake_pending() {
  std::lock_guard<std::mutex> lock(st().mu);
  int64_t n = 0;
  for (const auto &p : st().queued) n += p.second - st().done[p.first];
  return n;
}
int64_t fake_launches(const char *name) {
  std::lock_guard<std::mutex> lock(st().mu);
  int64_t n = 0;
  for (const auto &k : st().launched) n += k.find(name) != std::string::npos;
  return n;
}
void fake_forget_launches() {
  std::lock_guard<std::mutex> lock(st().mu);
  st().launched.clear();
}

// ------------------------------------------------------------ registration
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  st().kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

// ------------------------------------------------------------------ device
int hipGetDeviceCount(int *n) {
  *n = 1;
  return kOk;
}
int hipGetDevice(int *d) {
  *d = 0;
  return kOk;
}
int hipSetDevice(int) { return kOk; }
int hipGetSymbolAddress(void **p, const void *) {
  static double words[1 << 17];
  *p = words;
  return kOk;
}
const char *hipGetErrorString(int) { return "injected"; }
int hipGetLastError() {
  const int e = st().last_error;
  st().last_error = kOk;
  return e;
}
int hipDeviceSynchronize() {
  std::lock_guard<std::mutex> lock(st().mu);
  st().done = st().queued;
  return kOk;
}

// ------------------------------------------------------------------ memory
int hipMalloc(void **p, size_t bytes) {
  std::lock_guard<std::mutex> lock(st().mu);
  *p = nullptr;
  if ((st().fail_bytes == bytes && bytes > 0) || st().held + bytes > st().capacity)
    return st().last_error = kOutOfMemory;
  *p = calloc(bytes ? bytes : 1, 1);
  st().blocks[*p] = bytes;
  st().held += bytes;
  if (st().held > st().peak) st().peak = st().held;
  return kOk;
}
int hipFree(void *p) {
  if (!p) return kOk;
  if (st().free_ms) std::this_thread::sleep_for(std::chrono::milliseconds(st().free_ms));
  std::lock_guard<std::mutex> lock(st().mu);
  const auto it = st().blocks.find(p);
  if (it == st().blocks.end()) return kInvalid;
  st().held -= it->second;
  st().blocks.erase(it);
  free(p);
  return kOk;
}
int hipHostMalloc(void **p, size_t bytes, unsigned) {
  *p = calloc(bytes, 1);
  return kOk;
}
int hipHostFree(void *p) {
  free(p);
  return kOk;
}
int hipMemset(void *p, int v, size_t n) {
  if (n <= (size_t)64 << 20) memset(p, v, n);
  return kOk;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  memcpy(d, s, n);
  return kOk;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, Stream *stream) {
  std::lock_guard<std::mutex> lock(st().mu);
  memcpy(d, s, n);
  if (kind == 2 && n == st().poke_bytes && n > 0)
    memcpy((char *)d + st().poke_at, &st().poke_value, sizeof(int64_t));
  enqueue(stream);
  return kOk;
}

// ------------------------------------------------------- streams and events
int hipStreamCreateWithFlags(Stream **s, unsigned) {
  std::lock_guard<std::mutex> lock(st().mu);
  *s = new Stream{st().next_stream++, {}};
  return kOk;
}
int hipStreamDestroy(Stream *s) {
  delete s;
  return kOk;
}
int hipStreamSynchronize(Stream *s) {
  std::lock_guard<std::mutex> lock(st().mu);
  if (!s) return kOk;
  merge(st().done, s->follows);
  st().done[s->id] = st().queued[s->id];
  return kOk;
}
int hipEventCreate(Event **e) {
  *e = new Event;
  return kOk;
}
int hipEventCreateWithFlags(Event **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(Event *e) {
  delete e;
  return kOk;
}
int hipEventRecord(Event *e, Stream *s) {
  std::lock_guard<std::mutex> lock(st().mu);
  e->seen.clear();
  if (!s) return kOk;
  e->seen = s->follows;
  e->seen[s->id] = st().queued[s->id];
  return kOk;
}
int hipStreamWaitEvent(Stream *s, Event *e, unsigned) {
  std::lock_guard<std::mutex> lock(st().mu);
  if (s) merge(s->follows, e->seen);
  return kOk;
}
int hipEventSynchronize(Event *e) {
  std::lock_guard<std::mutex> lock(st().mu);
  merge(st().done, e->seen);
  return kOk;
}
int hipEventQuery(Event *) { return kOk; }
int hipEventElapsedTime(float *ms, Event *, Event *) {
  *ms = 1.0f;
  return kOk;
}
int hipStreamIsCapturing(Stream *, int *status) {
  *status = 0;
  return kOk;
}
int hipStreamBeginCapture(Stream *, int) { return kInvalid; }
int hipStreamEndCapture(Stream *, void **) { return kInvalid; }
int hipGraphInstantiate(void **, void *, void *, char *, size_t) { return kInvalid; }
int hipGraphLaunch(void *, Stream *) { return kInvalid; }
int hipGraphDestroy(void *) { return kOk; }
int hipGraphExecDestroy(void *) { return kOk; }

// ---------------------------------------------------------------- launches
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, Stream *stream) {
  config = {grid, block, shared, stream};
  return kOk;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, Stream **stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return kOk;
}
int hipLaunchKernel(const void *kernel, Dim3, Dim3, void **, size_t, Stream *stream) {
  std::lock_guard<std::mutex> lock(st().mu);
  const std::string &name = st().kernels[kernel];
  st().launched.push_back(name);
  enqueue(stream);
  if (!st().fail_kernel.empty() && name.find(st().fail_kernel) != std::string::npos) {
    st().fail_kernel.clear();
    st().last_error = kUnknown;
  }
  return kOk;
}

}  // extern "C"
