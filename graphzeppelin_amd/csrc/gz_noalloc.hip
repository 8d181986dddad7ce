// gz_noalloc.hip -- Sketch::update over a batch (src/sketch.cpp:69-83) for callers that cannot
// allocate device memory: code under HIP graph capture, tight serving loops, harnesses that forbid
// hipMalloc.  It runs the same kernel as gz_sketch_update_batch on the indices where the caller keeps
// them in device memory (nothing is staged).
#include <hip/hip_runtime.h>

#include "../../include/gz_hip.h"
#include "gz_runtime.hpp"

namespace gz {
namespace {

constexpr size_t kNoAllocMax = size_t(1) << 26;  // indices per call

// Makes `dev` current for the call and restores the caller's device afterwards.
struct DeviceScope {
  int prev = -1;
  explicit DeviceScope(int dev) {
    GZ_HIP(hipGetDevice(&prev));
    if (prev != dev) GZ_HIP(hipSetDevice(dev));
    else prev = -1;
  }
  ~DeviceScope() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

}  // namespace
}  // namespace gz

extern "C" int gz_sketch_update_batch_device_noalloc(gz_sketch* s, const uint64_t* idx_device, size_t count) {
  try {
    if (!s || (!idx_device && count)) throw gz::GzError(GZ_ERR_INVALID_ARG, "null argument");
    if (count > gz::kNoAllocMax)
      throw gz::GzError(GZ_ERR_INVALID_ARG, "count above the no-allocation limit of 2^26 indices per call");
    if (count) {
      gz::GzSketch& S = *s->s;
      gz::DeviceScope scope(S.dev);
      gz::launch_sketch_update(S.gb, idx_device, count, S.slab.p, S.geo, S.col_bf.p, S.st);
      GZ_HIP(hipGetLastError());
      GZ_HIP(hipStreamSynchronize(S.st));
    }
    gz::clear_last_error();
    return GZ_OK;
  } catch (const std::exception& e) {
    return gz::status_of(e);
  }
}
