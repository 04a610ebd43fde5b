// Small 2-D and 3-D fields in one kernel, f64.
#include <hip/hip_runtime.h>

#include "fft_field.hpp"

namespace vkfx {
// radices up to 10 in 120 to 148 registers, larger ones (214) apart
KernelFn pick_field_f64(int dir, bool large) {
    if (large) return dir < 0 ? k_field<double, -1, 16> : k_field<double, 1, 16>;
    return dir < 0 ? k_field<double, -1, 10> : k_field<double, 1, 10>;
}
}  // namespace vkfx
