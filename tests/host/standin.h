// Host stand-in of the HIP runtime and of the kernel launchers, so that the
// engine's host code runs on the CPU: device memory is host memory counted
// against a limit, copies are immediate, launches do nothing but can be looked at
// or made to fail.
#pragma once
#include <stddef.h>

#include <functional>

#include "../../seismic_amd/csrc/xc_kernels.h"
#include "../../seismic_amd/csrc/xc_lag.h"

namespace standin {
extern size_t limit;                // bytes of device memory
size_t used();                      // now
size_t size_of(const void* block);  // of the device block that holds this address (0: none)
// called with a launch's arguments; a non-zero return is the launch's error
extern std::function<int(int R, const sxc::ForwardArgs&)> on_forward;
extern std::function<int(int R, bool full, const sxc::PairArgs&)> on_pairs;
extern std::function<int(int R, const sxc::ResolveArgs&)> on_resolve;
extern std::function<int(const sxc::LagPrepArgs&)> on_lag_prep;
extern std::function<int(bool bf16x3, const sxc::LagPairArgs&)> on_lag_pairs;
}  // namespace standin
