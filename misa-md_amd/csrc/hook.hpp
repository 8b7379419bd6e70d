// Hook-mode launcher.
#pragma once
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "host_setup.hpp"
#include "inter_common.hpp"
#include "site_common.hpp"

namespace misa {

// which: 0 rho, 1 df, 2 force.  full: the handle's full lists on the device;
// rec, sp: scratch for a record and a byte per slot.
void launchHook(int which, const Box& b, double rc, const FullPlaneOffsets* full, const Tables<double>& tb, site::Rec64 rec,
                uint8_t* sp, AtomElement* a, hipStream_t st);

}  // namespace misa
