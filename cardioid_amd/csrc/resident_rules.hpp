// resident_rules.hpp -- the rules of the resident form that need no device:
// plain functions, the same on the host and in the kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace cdh {

// Whether a cooperative launch that ended with `e` was turned down for what it
// asks of the device, so that step kernels take the run; any other error is
// the caller's.
inline bool resident_refused(hipError_t e)
{
   return e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported;
}

}  // namespace cdh
