// Stands before the HIP runtime's cooperative launch, for GPU tests of what follows a
// one-per-tile pressure solve that gives up, or a resident one that is refused.
// Loaded with global symbols before libsplashtank_hip.so (tests/test_coop_fallbacks.py).
// Mode 1: the one-per-tile launches find their arrival word marked late, as the first
// workgroup that waited too long would leave it, and check it however few they are;
// every workgroup then ends at once.  Mode 2: launches of 1024 threads are refused.
#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include "flip_device.h"
#include "flip_kernels.h"

static int g_mode = 0, g_hits = 0;
static const uint32_t kLate = 0x80000000u;

extern "C" {
void coop_shim_set(int mode) { g_mode = mode, g_hits = 0; }
int coop_shim_hits() { return g_hits; }

// batch launches have five arguments, a tank's six: the caller says which it makes
static int g_batch = 0;
void coop_shim_batch(int b) { g_batch = b; }

hipError_t hipLaunchCooperativeKernel(const void* f, dim3 grid, dim3 block, void** args, unsigned int shared, hipStream_t st) {
  typedef hipError_t (*Launch)(const void*, dim3, dim3, void**, unsigned int, hipStream_t);
  static const Launch next = (Launch)dlsym(RTLD_NEXT, "hipLaunchCooperativeKernel");
  if (!next) return hipErrorNotFound;
  if (g_mode == 2 && block.x == COOP_WG) {
    g_hits++;
    return hipErrorCooperativeLaunchTooLarge;
  }
  if (g_mode == 1 && block.x != COOP_WG) {
    uint32_t* here;
    if (g_batch) {  // (tanks, table, nt, plan, safe)
      here = *(uint32_t**)args[3] + batch_here(*(uint32_t*)args[2]);
      *(uint32_t*)args[4] = 0u;
    } else {  // (P, G, iters, tag, seq, safe)
      here = ((DGrid*)args[1])->sorBar + SOR_HERE;
      *(uint32_t*)args[5] = 0u;
    }
    const hipError_t e = hipMemcpyAsync(here, &kLate, 4, hipMemcpyHostToDevice, st);
    if (e != hipSuccess) return e;
    g_hits++;
  }
  return next(f, grid, block, args, shared, st);
}
}
