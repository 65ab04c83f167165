// Instances of the wide affine GEMM kernel: 8-bit codes, groups of 64 or more, f16.
#include "affine_wide_kernel.h"

namespace mt {

hipError_t launch_affine_wide_u8_f16(const WideParams& p, int nproj, hipStream_t stream) {
  return launch_proj<8, kF16, false>(p, nproj, stream);
}

}  // namespace mt
