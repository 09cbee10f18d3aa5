// A HIP runtime of host memory, for CPU tests of the library's host code: device
// memory is the heap, copies are memcpy, and a launch only writes a line to a log
// (kernel name, workgroups, threads, cooperative or not; the id-order readback also
// does its work).  Loaded with global
// symbols before libsplashtank_hip.so, whose HIP calls then come here.  Built by the
// package build into tests/c/libhost_hip.so and used through tests/host_hip.py.
// host_hip_set makes calls fail, and lets the one-per-tile solves mark their work
// as done as the kernels would.
#include <hip/hip_runtime.h>
#include <malloc.h>
#include <stdint.h>
#include <stdio.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "flip_device.h"
#include "flip_kernels.h"

static std::string g_log;
static std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> m;
  return m;
}
static int64_t g_live = 0;
static int g_refuse = 0;      // cooperative launches of this many threads are refused
static int g_solves = 0;      // the one-per-tile solves do their work
static int g_failCapture = 0; // the next capture ends with an error
static int g_failLaunch = 0;  // the next look for a launch's error finds one
static int g_failMalloc = 0;  // the next allocation fails
static char g_any[64];        // what handles point at

static hipError_t logf(const char* what, const void* f, dim3 g, dim3 b, hipStream_t st) {
  auto k = kernels().find(f);
  g_log += std::string(what) + " " + (k == kernels().end() ? "?" : k->second) + " " + std::to_string(g.x) + " " + std::to_string(b.x) + "\n";
  return hipSuccess;
}

extern "C" {
const char* host_hip_log() { return g_log.c_str(); }
void host_hip_clear() { g_log.clear(); }
int64_t host_hip_live() { return g_live; }
void host_hip_set(const char* what, int v) {
  if (!strcmp(what, "refuse")) g_refuse = v;
  if (!strcmp(what, "solves")) g_solves = v;
  if (!strcmp(what, "failCapture")) g_failCapture = v;
  if (!strcmp(what, "failLaunch")) g_failLaunch = v;
  if (!strcmp(what, "failMalloc")) g_failMalloc = v;
}

void** __hipRegisterFatBinary(const void*) { return (void**)g_any; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned int, void*, void*, dim3*, dim3*, int*) { kernels()[f] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static dim3 g_grid, g_block;
static size_t g_shared;
static hipStream_t g_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
  g_grid = g, g_block = b, g_shared = s, g_stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = g_grid, *b = g_block, *s = g_shared, *st = g_stream;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int threads, size_t) {
  *n = threads >= 1024 ? 1 : 7;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_failLaunch ? hipErrorLaunchFailure : hipSuccess;
  g_failLaunch = 0;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "host"; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = g_any; return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) {
  if (g_failMalloc) {
    g_failMalloc = 0;
    return hipErrorOutOfMemory;
  }
  *p = calloc(1, n ? n : 1);
  if (!*p) return hipErrorOutOfMemory;
  g_live += int64_t(malloc_usable_size(*p));
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (p) g_live -= int64_t(malloc_usable_size(p));
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { *p = calloc(1, n ? n : 1); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  g_log += "copy null\n";
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
  memset(p, v, n);
  g_log += "memset stream\n";
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) { *s = (hipStream_t)g_any; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { g_log += "sync\n"; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)g_any;
  if (!g_failCapture) return hipSuccess;
  g_failCapture = 0;
  return hipErrorStreamCaptureInvalidated;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = (hipGraphExec_t)g_any; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { g_log += "graph\n"; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)g_any; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 1.0f; return hipSuccess; }

hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t, hipStream_t st) {
  if (kernels()[f].find("8k_unsortP") != std::string::npos) {  // the id-order readback: (src, ids, out, n)
    const float4* src = *(const float4**)args[0];
    const uint32_t* id = *(const uint32_t**)args[1];
    for (uint32_t i = 0; i < *(uint32_t*)args[3]; i++) (*(float4**)args[2])[id[i]] = src[i];
  }
  return logf("launch", f, g, b, st);
}
hipError_t hipLaunchCooperativeKernel(const void* f, dim3 g, dim3 b, void** args, unsigned int, hipStream_t st) {
  if (g_refuse && b.x == unsigned(g_refuse)) {
    logf("refused", f, g, b, st);
    return hipErrorCooperativeLaunchTooLarge;
  }
  if (g_solves) {
    const std::string& n = kernels()[f];
    if (n.find("kb_sor_tiles") != std::string::npos) {  // (tanks, table, nt, plan, safe)
      (*(uint32_t**)args[3])[3u * *(uint32_t*)args[2] + 1u] = 1u;
    } else if (n.find("k_sor_tiles") != std::string::npos) {  // (P, G, iters, tag, seq, safe)
      ((DGrid*)args[1])->sorBar[COOP_MAX_WG + 4] = *(uint32_t*)args[4];
    }
  }
  return logf("coop", f, g, b, st);
}
}
