// Small 2-D and 3-D fields in one kernel, f32.
#include <hip/hip_runtime.h>

#include "fft_field.hpp"

namespace vkfx {
KernelFn pick_field_f32(int dir, bool) { return dir < 0 ? k_field<float, -1, 16> : k_field<float, 1, 16>; }
}  // namespace vkfx
