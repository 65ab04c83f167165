// Dispatch of the wide affine GEMM kernel to its instances (one source per code width, group class
// and activation type, so that they compile side by side).
#include "affine_wide.h"
#include "common.h"

namespace mt {

#define MT_WIDE_INSTANCES(name) \
  hipError_t launch_affine_wide_##name(const WideParams& p, int nproj, hipStream_t stream);
MT_WIDE_INSTANCES(u4_bf16)
MT_WIDE_INSTANCES(u4_f16)
MT_WIDE_INSTANCES(u8_bf16)
MT_WIDE_INSTANCES(u8_f16)
MT_WIDE_INSTANCES(u8g32_bf16)
MT_WIDE_INSTANCES(u8g32_f16)
#undef MT_WIDE_INSTANCES

hipError_t launch_affine_wide(const WideParams& p, int bits, int dtype, int nproj,
                              hipStream_t stream) {
  const bool bf = dtype == kBF16;
  if (bits == 4)
    return p.group_shift < 6 ? hipErrorInvalidValue
           : bf              ? launch_affine_wide_u4_bf16(p, nproj, stream)
                             : launch_affine_wide_u4_f16(p, nproj, stream);
  if (p.group_shift < 6)
    return bf ? launch_affine_wide_u8g32_bf16(p, nproj, stream)
              : launch_affine_wide_u8g32_f16(p, nproj, stream);
  return bf ? launch_affine_wide_u8_bf16(p, nproj, stream)
            : launch_affine_wide_u8_f16(p, nproj, stream);
}

}  // namespace mt
