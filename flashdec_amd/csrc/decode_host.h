// Host-side helpers shared by the decode entry points.
#pragma once

#include <hip/hip_ext.h>

#include "decode_unit.h"

namespace fd {

// Compute units of the current device.
int device_cus();

// The MFMA row kernel's and the even-share kernel's shape, stride and
// alignment requirements (defined beside the row kernel's launch).
bool fast_path_ok(const fd_paged_decode_args& a, int64_t group);

// Validates the launch arguments shared by the decode entry points and fills
// the kernel parameters; fn names the entry point in error messages.
int fill_decode_params(const fd_paged_decode_args* args, const char* fn, DecodeParams& p);

// One dispatch; events given are recorded at its start / end (profiling hook).
template <typename F, typename... Args>
void dispatch(F kernel, dim3 grid, dim3 block, hipStream_t stream, void* start, void* stop, Args... args) {
  if (launch_record_on()) record_launch(reinterpret_cast<const void*>(kernel), stream);
  if (start || stop)
    hipExtLaunchKernelGGL(kernel, grid, block, 0, stream, static_cast<hipEvent_t>(start),
                          static_cast<hipEvent_t>(stop), 0, args...);
  else
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, args...);
}

}  // namespace fd
