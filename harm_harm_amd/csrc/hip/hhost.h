// hhost.h -- host-side helpers shared by the library's .hip translation units.
#pragma once
#include <hip/hip_runtime.h>
#include "harmstep.h"

namespace hh {

harm_status set_error(harm_status st, const char* fmt, ...);
harm_status check_hip(hipError_t e, const char* what);
harm_status check_launch(const char* kernel);

// Rounds of 256 zones a block of the batched inversions takes, for nr runs of
// 256 zones on a chip that holds `resident` blocks: whole passes of that many
// blocks with at most 16 rounds each.  Up to `resident` runs every run is a
// block of its own and its solves run through (their length is the call's
// latency).
inline int inversion_rounds(long nr, long resident)
{
  const long passes = (nr + resident * 16 - 1) / (resident * 16);
  return (int)((nr + resident * passes - 1) / (resident * passes));
}

}  // namespace hh

#define HH_TRY(expr)                          \
  do {                                        \
    harm_status _st = (expr);                 \
    if (_st != HARM_OK) return _st;           \
  } while (0)

#define HH_HIP(expr) HH_TRY(hh::check_hip((expr), #expr))
