// A stand-in for the HIP runtime calls libsemtex_amd.so makes, preloaded into
// a CPU process by tests/test_alloc_failures.py: device memory is host memory,
// kernel launches are counted by name and do nothing, and allocations can be
// made to fail.  Only host code (allocation, bookkeeping, what is launched)
// runs on it.
#include <hip/hip_runtime.h>

#include "../include/semtex_amd.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex mu;
std::map<void*, size_t> live;               // device and pinned allocations
std::map<const void*, std::string> names;   // kernel stub -> device name
std::map<std::string, long> launched;
long allocs = 0, fail_at = -1, fail_to = -1, device = 0, bad = 0, freed = 0;
bool sync_fails = false, bad_pivots = false;
size_t limit = 0;                           // bytes on the "device" (0: no limit)
hipError_t last = hipSuccess;

hipError_t ret (hipError_t e) { if (e != hipSuccess) last = e; return e; }

hipError_t allocate (void** p, size_t bytes)
{
  std::lock_guard<std::mutex> lock (mu);
  const long i = allocs++;
  size_t used = 0;
  if (limit) for (auto& a : live) used += a.second;
  if ((fail_at >= 0 && i >= fail_at && i < fail_to) || (limit && used + bytes > limit)) {
    *p = nullptr;
    return ret (hipErrorOutOfMemory);
  }
  *p = std::malloc (bytes + !bytes);
  std::memset (*p, 0xA5, bytes);
  live[*p] = bytes;
  return hipSuccess;
}
hipError_t release (void* p)
{
  std::lock_guard<std::mutex> lock (mu);
  if (!p) return hipSuccess;
  if (!live.erase (p)) { std::abort (); }   // not an allocation, or freed twice
  freed++;
  std::free (p);
  return hipSuccess;
}
}  // namespace

// control, called from the test
extern "C" {
// allocations from now on: the ones numbered [first, first + count) fail
void stub_fail (long first, long count) { allocs = 0; fail_at = first; fail_to = first + count; }
void stub_limit (size_t bytes) { limit = bytes; }
void stub_device (long d) { device = d; }
void stub_bad_pivots (int on) { bad_pivots = on != 0; }
void stub_sync_fails (int on) { sync_fails = on != 0; }
long stub_allocs () { return allocs; }
long stub_freed () { return freed; }
long stub_live () { return (long) live.size (); }
size_t stub_bytes () { size_t n = 0; for (auto& a : live) n += a.second; return n; }
long stub_launches (const char* part)
{
  long n = 0;
  for (auto& l : launched) if (l.first.find (part) != std::string::npos) n += l.second;
  return n;
}

hipError_t hipMalloc (void** p, size_t bytes) { return allocate (p, bytes); }
hipError_t hipFree (void* p) { return release (p); }
hipError_t hipHostMalloc (void** p, size_t bytes, unsigned) { return allocate (p, bytes); }
hipError_t hipHostFree (void* p) { return release (p); }
hipError_t hipMemcpy (void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy (d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync (void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy (d, s, n); return hipSuccess; }
hipError_t hipMemset (void* d, int v, size_t n) { std::memset (d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync (void* d, int v, size_t n, hipStream_t) { std::memset (d, v, n); return hipSuccess; }
hipError_t hipGetDevice (int* d) { *d = (int) device; return hipSuccess; }
hipError_t hipSetDevice (int d) { device = d; return hipSuccess; }
hipError_t hipGetDeviceCount (int* n) { *n = 2; return hipSuccess; }
hipError_t hipDeviceSynchronize () { return sync_fails ? ret (hipErrorStreamCaptureUnsupported) : hipSuccess; }
hipError_t hipDeviceGetAttribute (int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600 (hipDeviceProp_tR0600* p, int)
{
  std::memset (p, 0, sizeof *p);
  std::strcpy (p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString (hipError_t) { return "stub error"; }
hipError_t hipGetLastError () { hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipFuncSetAttribute (const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes (hipFuncAttributes* a, const void*) { std::memset (a, 0, sizeof *a); return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor (int* n, const void*, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipGetSymbolAddress (void** p, const void*)   // (the library has one device array)
{
  static void* a = std::calloc (SX_NOALLOC_DOUBLES, 8);
  *p = a;
  return hipSuccess;
}

hipError_t hipStreamCreate (hipStream_t* s) { *s = (hipStream_t) std::malloc (1); return hipSuccess; }
hipError_t hipStreamDestroy (hipStream_t s) { std::free ((void*) s); return hipSuccess; }
hipError_t hipStreamSynchronize (hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent (hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture (hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture (hipStream_t, hipGraph_t* g) { *g = (hipGraph_t) std::malloc (1); return hipSuccess; }
hipError_t hipStreamIsCapturing (hipStream_t, hipStreamCaptureStatus* c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGraphInstantiate (hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = (hipGraphExec_t) std::malloc (1); return hipSuccess; }
hipError_t hipGraphLaunch (hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy (hipGraph_t g) { std::free ((void*) g); return hipSuccess; }
hipError_t hipGraphExecDestroy (hipGraphExec_t e) { std::free ((void*) e); return hipSuccess; }
hipError_t hipEventCreate (hipEvent_t* e) { *e = (hipEvent_t) std::malloc (1); return hipSuccess; }
hipError_t hipEventCreateWithFlags (hipEvent_t* e, unsigned) { return hipEventCreate (e); }
hipError_t hipEventDestroy (hipEvent_t e) { std::free ((void*) e); return hipSuccess; }
hipError_t hipEventRecord (hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize (hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime (float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

// Pointer arguments (by position) of the kernels the tests here reach that
// must lie in a live allocation
static const struct { const char* name; int at[4]; } pointers[] = {
    {"k_tree_assemble", {0, 2, 3, 9}}, {"k_tree_panel", {0, 2, 4, 7}},
    {"k_tree_update", {0, 2, 4, 0}},   {"k_tree_operators", {0, 2, 4, 0}},
    {"k_tree_residual", {3, 4, 5, 6}}, {"k_tree_entries", {1, 2, 3, 4}},
    {"k_band_assemble", {1, 2, 3, 7}}, {"k_band_factor", {0, 4, 0, 0}},
};
long stub_bad_pointers () { return bad; }

hipError_t hipLaunchKernel (const void* f, dim3, dim3, void** args, size_t, hipStream_t)
{
  std::lock_guard<std::mutex> lock (mu);
  const std::string& name = names[f];
  launched[name]++;
  if (bad_pivots && name.find ("k_tree_panel") != std::string::npos) **(int**) args[7] = 1;
  for (auto& k : pointers)
    if (name.find (k.name) != std::string::npos)
      for (int i : k.at) {
        char* p = *(char**) args[i];
        auto a = live.upper_bound (p);
        if (a == live.begin () || p >= (char*) (--a)->first + a->second) bad++;
      }
  return hipSuccess;
}
void** __hipRegisterFatBinary (const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary (void**) {}
void __hipRegisterFunction (void**, const void* host, char*, const char* name, unsigned, void*, void*,
                            void*, void*, int*)
{
  std::lock_guard<std::mutex> lock (mu);
  names[host] = name;
}
void __hipRegisterVar (void**, void*, char*, char*, int, size_t, int, int) {}

static thread_local struct { dim3 g, b; size_t l; hipStream_t s; } call;
hipError_t __hipPushCallConfiguration (dim3 g, dim3 b, size_t l, hipStream_t s)
{
  call = {g, b, l, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration (dim3* g, dim3* b, size_t* l, hipStream_t* s)
{
  *g = call.g; *b = call.b; *l = call.l; *s = call.s;
  return hipSuccess;
}
}
