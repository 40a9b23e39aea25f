// hhost.h -- host-side helpers shared by the library's .hip translation units.
#pragma once
#include <hip/hip_runtime.h>
#include "harmstep.h"

namespace hh {

harm_status set_error(harm_status st, const char* fmt, ...);
harm_status check_hip(hipError_t e, const char* what);
harm_status check_launch(const char* kernel);

}  // namespace hh

#define HH_TRY(expr)                          \
  do {                                        \
    harm_status _st = (expr);                 \
    if (_st != HARM_OK) return _st;           \
  } while (0)

#define HH_HIP(expr) HH_TRY(hh::check_hip((expr), #expr))
