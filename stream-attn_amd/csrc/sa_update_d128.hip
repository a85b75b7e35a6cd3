// The update kernel's variants for head_dim padded to 128.
#include "sa_update_kernel.h"

namespace sa {
namespace {

template <int MODE>
hipError_t launch_mode(const UpdateParams& p, const LaunchShape& shape, int dtype, hipStream_t stream) {
  switch (shape.rows) {
    case 128: return launch_variant<128, 1, MODE>(p, shape, dtype, stream);
    case 256: return launch_variant<128, 2, MODE>(p, shape, dtype, stream);
    default: return launch_variant<128, 3, MODE>(p, shape, dtype, stream);
  }
}

}  // namespace

hipError_t launch_update_d128(const UpdateParams& p, int mode, const LaunchShape& shape, int dtype, hipStream_t stream) {
  switch (mode) {
    case kInt8: return launch_mode<kInt8>(p, shape, dtype, stream);
    case kTransposedV: return launch_mode<kTransposedV>(p, shape, dtype, stream);
    default: return launch_mode<kRows>(p, shape, dtype, stream);
  }
}

}  // namespace sa
