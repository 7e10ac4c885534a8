// A HIP runtime for host-side tests: device memory is host memory, kernels are
// not run, and every call of interest is recorded.  The test program defines
// these symbols itself and exports them (-rdynamic), so a library it dlopens
// binds to them instead of the installed runtime, and the library's host code
// runs on a machine without a GPU.
#pragma once

#include <hip/hip_runtime_api.h>

#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

namespace rec
{
struct Call
{
  std::string what;     // "launch", "copy", "malloc", "free", "stream_wait", "event_record", "wait_event", ...
  std::string kernel;   // launches: the kernel's mangled name
  void* stream = nullptr;
  void* event = nullptr;
  size_t bytes = 0;     // copies, allocations
  unsigned grid = 0, block = 0;
};

inline std::recursive_mutex g_m;
inline std::vector<Call> g_calls;
inline std::map<const void*, std::string> g_kernels;
inline std::map<void*, size_t> g_live;  // device blocks
inline int g_fail_malloc = 0, g_fail_copy = 0;  // > 0: the n-th one from now fails
inline bool g_capturing = false;
inline int g_not_ready = 0;  // > 0: so many stream queries answer "not ready", as an error that stays
inline hipError_t g_last = hipSuccess;
// Called at a launch (stands in for what the kernel would leave in pinned
// memory) and at a host wait, outside the lock.
inline std::function<void(const std::string&, void**)> on_launch;
inline std::function<void(const char*)> on_wait;

inline void note(Call c)
{
  std::lock_guard<std::recursive_mutex> g(g_m);
  g_calls.push_back(std::move(c));
}
inline hipError_t fail(hipError_t e)
{
  g_last = e;
  return e;
}
inline size_t count(const std::string& what, const std::string& kernel = "")
{
  std::lock_guard<std::recursive_mutex> g(g_m);
  size_t n = 0;
  for (const Call& c : g_calls) n += c.what == what && c.kernel.find(kernel) != std::string::npos;
  return n;
}
inline void clear()
{
  std::lock_guard<std::recursive_mutex> g(g_m);
  g_calls.clear();
}
inline size_t live_blocks()
{
  std::lock_guard<std::recursive_mutex> g(g_m);
  return g_live.size();
}
inline void waited(const char* how)
{
  if (on_wait) on_wait(how);
}

struct Config
{
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
};
inline thread_local std::vector<Config> t_config;
}  // namespace rec

extern "C" {

void** __hipRegisterFatBinary(const void*)
{
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*,
                           int*)
{
  std::lock_guard<std::recursive_mutex> g(rec::g_m);
  rec::g_kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s)
{
  rec::t_config.push_back({grid, block, shmem, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s)
{
  const rec::Config c = rec::t_config.back();
  rec::t_config.pop_back();
  *grid = c.grid;
  *block = c.block;
  *shmem = c.shmem;
  *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t s)
{
  rec::Call c;
  c.what = "launch";
  {
    std::lock_guard<std::recursive_mutex> g(rec::g_m);
    c.kernel = rec::g_kernels[f];
  }
  c.stream = (void*)s;
  c.grid = grid.x;
  c.block = block.x;
  rec::note(c);
  if (rec::on_launch) rec::on_launch(c.kernel, args);
  return hipSuccess;
}

hipError_t hipGetDevice(int* d)
{
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipRuntimeGetVersion(int* v)
{
  *v = 1;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "planted error"; }
hipError_t hipGetLastError(void)
{
  const hipError_t e = rec::g_last;
  rec::g_last = hipSuccess;
  return e;
}

hipError_t hipMalloc(void** p, size_t bytes)
{
  std::lock_guard<std::recursive_mutex> g(rec::g_m);
  if (rec::g_fail_malloc > 0 && --rec::g_fail_malloc == 0)
  {
    *p = nullptr;
    return rec::fail(hipErrorOutOfMemory);
  }
  *p = calloc(1, bytes ? bytes : 1);
  rec::g_live[*p] = bytes;
  rec::Call c;
  c.what = "malloc";
  c.bytes = bytes;
  rec::g_calls.push_back(c);
  return hipSuccess;
}
hipError_t hipFree(void* p)
{
  std::lock_guard<std::recursive_mutex> g(rec::g_m);
  rec::Call c;
  c.what = "free";
  rec::g_calls.push_back(c);
  if (p && rec::g_live.erase(p) == 0) abort();
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned)
{
  *p = calloc(1, bytes ? bytes : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
  free(p);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t bytes)
{
  memset(p, v, bytes);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t bytes, hipMemcpyKind)
{
  std::lock_guard<std::recursive_mutex> g(rec::g_m);
  if (rec::g_fail_copy > 0 && --rec::g_fail_copy == 0) return rec::fail(hipErrorStreamCaptureUnsupported);
  memcpy(d, s, bytes);
  rec::Call c;
  c.what = "copy";
  c.bytes = bytes;
  rec::g_calls.push_back(c);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t st)
{
  rec::Call c;
  c.what = "copy_async";
  c.stream = (void*)st;
  c.bytes = bytes;
  memcpy(d, s, bytes);
  rec::note(c);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
  static char room[1 << 22];
  *p = room;
  return hipSuccess;
}
hipError_t hipMemcpyFromSymbol(void* d, const void*, size_t bytes, size_t, hipMemcpyKind)
{
  memset(d, 0, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
  *s = (hipStream_t)malloc(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
  free((void*)s);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st)
{
  *st = rec::g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t)
{
  rec::waited("stream_query");
  return rec::g_not_ready > 0 && rec::g_not_ready-- > 0 ? rec::fail(hipErrorNotReady) : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
  rec::Call c;
  c.what = "stream_wait";
  c.stream = (void*)s;
  rec::note(c);
  rec::waited("stream");
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void)
{
  rec::waited("device");
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
  rec::Call c;
  c.what = "wait_event";
  c.stream = (void*)s;
  c.event = (void*)e;
  rec::note(c);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e)
{
  *e = (hipEvent_t)malloc(1);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
  free((void*)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
  rec::Call c;
  c.what = "event_record";
  c.stream = (void*)s;
  c.event = (void*)e;
  rec::note(c);
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t)
{
  rec::waited("event");
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
  *ms = 1.0f;
  return hipSuccess;
}

}  // extern "C"
