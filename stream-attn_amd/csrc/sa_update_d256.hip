// The update kernel's variants for head_dim padded to 256.  INT8 K/V covers
// head_dim <= 128: with head_dim 256 the 16-bit stages and the raw staging
// would not fit in LDS together.
#include "sa_update_kernel.h"

namespace sa {

hipError_t launch_update_d256(const UpdateParams& p, int mode, const LaunchShape& shape, int dtype, hipStream_t stream) {
  (void)mode;
  return shape.rows == 128 ? launch_variant<256, 1, kRows>(p, shape, dtype, stream)
                     : launch_variant<256, 2, kRows>(p, shape, dtype, stream);
}

}  // namespace sa
