// A HIP runtime on the host for tests of the library's host code without a
// GPU: memory is host memory, copies are done at once, kernels do nothing.
// It keeps the rule that an event is recorded on streams of its own device
// only, and can make pinned memory, threads and host memory run out.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>

namespace {
struct Stream {
  int device, id;
};
struct Event {
  int device;
  Stream *recorded;
};
thread_local int g_device = 0;
std::atomic<int> g_streams{0}, g_pinned{1 << 30}, g_threads{1 << 30};
std::atomic<long> g_new_max{-1}, g_device_max{-1};
std::mutex g_mu;
char g_log[1 << 20];
int g_log_len = 0;
// (the runtime's own objects come from malloc: its memory does not run out)
template <typename T>
T *make(T v) {
  return static_cast<T *>(memcpy(malloc(sizeof(T)), &v, sizeof(T)));
}
Stream *S(hipStream_t s) { return reinterpret_cast<Stream *>(s); }
Event *E(hipEvent_t e) { return reinterpret_cast<Event *>(e); }
void note(const char *what, hipStream_t s, int other = -1) {
  char b[64];
  if (other >= 0) snprintf(b, sizeof(b), "%s %d %d\n", what, s ? S(s)->id : 0, other);
  else snprintf(b, sizeof(b), "%s %d\n", what, s ? S(s)->id : 0);
  std::lock_guard<std::mutex> lk(g_mu);
  const int n = (int)strlen(b);
  if (g_log_len + n < (int)sizeof(g_log)) memcpy(g_log + g_log_len, b, n + 1), g_log_len += n;
}
bool take(std::atomic<int> &left) {
  if (left.load() <= 0) return false;
  left--;
  return true;
}
}  // namespace

extern "C" {
// test controls: how many more pinned allocations and threads succeed, the
// largest operator new that does (-1: any), the calls so far (then cleared)
void stub_limits(int pinned, int threads, long new_max) {
  g_pinned = pinned;
  g_threads = threads;
  g_new_max = new_max;
}
// the largest device allocation that succeeds (-1: any)
void stub_device_max(long bytes) { g_device_max = bytes; }
int stub_log(char *out, int n) {
  std::lock_guard<std::mutex> lk(g_mu);
  const int len = g_log_len;
  snprintf(out, n, "%s", g_log);
  g_log_len = 0;
  g_log[0] = 0;
  return len;
}
int stub_device() { return g_device; }

hipError_t hipGetDeviceCount(int *n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = g_device, hipSuccess; }
hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return hipErrorInvalidDevice;
  return g_device = d, hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipMalloc(void **p, size_t n) {
  const long max = g_device_max.load();
  if (max >= 0 && n > (size_t)max) return *p = nullptr, hipErrorOutOfMemory;
  return *p = calloc(n ? n : 1, 1), hipSuccess;
}
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (!take(g_pinned)) return hipErrorOutOfMemory;
  return *p = malloc(n), hipSuccess;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  if (k == hipMemcpyDeviceToHost) note("read", st);
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemcpyToSymbol(const void *, const void *, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  return *s = reinterpret_cast<hipStream_t>(make(Stream{g_device, ++g_streams})), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return free(S(s)), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { return *d = s ? S(s)->device : g_device, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  note("wait", s, E(e)->recorded ? E(e)->recorded->id : 0);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  return *e = reinterpret_cast<hipEvent_t>(make(Event{g_device, nullptr})), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return free(E(e)), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (E(e)->device != (s ? S(s)->device : g_device)) return hipErrorInvalidHandle;
  return E(e)->recorded = S(s), hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s) {
  note("launch", s);
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t);
}

// launches carry their stream through the call configuration
namespace {
thread_local struct {
  dim3 grid, block;
  size_t shared;
  hipStream_t st;
} g_call;
}
extern "C" hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
  g_call = {g, b, sh, st};
  return hipSuccess;
}
extern "C" hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
  *g = g_call.grid, *b = g_call.block, *sh = g_call.shared, *st = g_call.st;
  return hipSuccess;
}

// std::thread and operator new as the library sees them
void std::thread::_M_start_thread(std::unique_ptr<_State> s, void (*)()) {
  if (!take(g_threads)) throw std::system_error(EAGAIN, std::generic_category());
  pthread_t id;
  auto run = [](void *p) -> void * {
    std::unique_ptr<_State> st(static_cast<_State *>(p));
    st->_M_run();
    return nullptr;
  };
  if (pthread_create(&id, nullptr, run, s.get())) throw std::system_error(EAGAIN, std::generic_category());
  s.release();
  _M_id = std::thread::id(id);
}
void *operator new(size_t n) {
  const long max = g_new_max.load();
  if (max >= 0 && n > (size_t)max) throw std::bad_alloc();
  void *p = malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
