// Instantiations of the general matrix-core kernels for 2-bit codes (xgemm.h).
#include "xgemm.h"

namespace affon {
namespace xgemm {
hipError_t launch_b2(const Args& args, Shape shape, bool g32, int x_dtype, int p_dtype, hipStream_t stream) {
  return launch<2>(args, shape, g32, x_dtype, p_dtype, stream);
}
}  // namespace xgemm
}  // namespace affon
