// The update kernel's variants for head_dim padded to 32.
#include "sa_update_kernel.h"

namespace sa {

hipError_t launch_update_d32(const UpdateParams& p, int mode, const LaunchShape& shape, int dtype, hipStream_t stream) {
  if (mode == kInt8)
    return shape.rows == 128 ? launch_variant<32, 1, kInt8>(p, shape, dtype, stream)
                       : launch_variant<32, 2, kInt8>(p, shape, dtype, stream);
  return shape.rows == 128 ? launch_variant<32, 1, kRows>(p, shape, dtype, stream)
                     : launch_variant<32, 2, kRows>(p, shape, dtype, stream);
}

}  // namespace sa
