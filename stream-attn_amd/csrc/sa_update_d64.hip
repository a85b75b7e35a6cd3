// The update kernel's variants for head_dim padded to 64.
#include "sa_update_kernel.h"

namespace sa {

hipError_t launch_update_d64(const UpdateParams& p, int mode, int rows, int dtype, hipStream_t stream) {
  if (mode == kInt8)
    return rows == 128 ? launch_variant<64, 1, kInt8>(p, dtype, stream)
                       : launch_variant<64, 2, kInt8>(p, dtype, stream);
  return rows == 128 ? launch_variant<64, 1, kRows>(p, dtype, stream)
                     : launch_variant<64, 2, kRows>(p, dtype, stream);
}

}  // namespace sa
