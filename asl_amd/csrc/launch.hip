// launch.hip — the launchers by template: each picks the kernels of d3q15,
// d3q19 or d3q27 (one object of kernels.hip per template), and the staging
// array of aslhip_read_f_noalloc.
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/aslhip.h"
#include "kernels.hpp"

namespace aslhip {

namespace {
const KernelTable *table(int q) {
  switch (q) {
    case 15: return &kernels_q15();
    case 19: return &kernels_q19();
    case 27: return &kernels_q27();
    default: return nullptr;
  }
}
}  // namespace

// Staging memory of aslhip_read_f_noalloc: a file-scope device array, so the
// entry point needs no allocation.  In host code `scratch` only names the
// symbol; its device address on each GPU comes from hipGetSymbolAddress (the
// array's name is never passed to a kernel or a copy).
static __device__ __align__(256) unsigned char scratch[ASLHIP_NOALLOC_SCRATCH_BYTES];
namespace {
constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex scratch_mu;
void *scratch_ptr[SCRATCH_MAX_DEVICES] = {};  // its address on each device (null: not looked up yet)
}  // namespace

hipError_t noalloc_scratch(void **ptr) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    scratch_ptr[dev] = p;
  }
  *ptr = scratch_ptr[dev];
  return hipSuccess;
}

int reduce_blocks(int len) {
  constexpr int RED_MAX_BLOCKS = 1024;
  const int nb = (len + 255) / 256;  // one cell per lane of k_reduce's workgroups
  return nb < RED_MAX_BLOCKS ? (nb < 1 ? 1 : nb) : RED_MAX_BLOCKS;
}

hipError_t launch_step(int q, int dtype, bool odd, bool periodic, bool wide, const StepLaunch &a, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->step(dtype, odd, periodic, wide, a, s) : hipErrorInvalidValue;
}
hipError_t launch_step_batch(int q, int dtype, bool odd, bool periodic, bool wide, const BatchLaunch &b,
                             hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->batch(dtype, odd, periodic, wide, b, s) : hipErrorInvalidValue;
}
hipError_t launch_vlinks(int q, int dtype, const VLinkArgs &a, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->vlinks(dtype, a, s) : hipErrorInvalidValue;
}
hipError_t launch_init(int q, int dtype, const InitArgs &a, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->init(dtype, a, s) : hipErrorInvalidValue;
}
hipError_t launch_write_f(int q, int dtype, const WriteFArgs &a, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->write_f(dtype, a, s) : hipErrorInvalidValue;
}
hipError_t launch_surface(int q, int dtype, const SurfaceArgs &a, const StepHot &g, const StepArgs *args,
                          hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->surface(dtype, a, g, args, s) : hipErrorInvalidValue;
}
hipError_t launch_vis(int q, int dtype, const VisArgs &a, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->vis(dtype, a, s) : hipErrorInvalidValue;
}
hipError_t launch_unpermute(int q, int dtype, const UnpermuteArgs &a, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->unpermute(dtype, a, s) : hipErrorInvalidValue;
}
hipError_t launch_reduce(int q, int dtype, const ReduceArgs &a, double *out, hipStream_t s) {
  const KernelTable *t = table(q);
  return t ? t->reduce(dtype, a, out, s) : hipErrorInvalidValue;
}

}  // namespace aslhip
