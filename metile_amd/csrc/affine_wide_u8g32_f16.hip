// Instances of the wide affine GEMM kernel: 8-bit codes, groups of 32, f16.
#include "affine_wide_kernel.h"

namespace mt {

hipError_t launch_affine_wide_u8g32_f16(const WideParams& p, int nproj, hipStream_t stream) {
  return launch_proj<8, kF16, true>(p, nproj, stream);
}

}  // namespace mt
