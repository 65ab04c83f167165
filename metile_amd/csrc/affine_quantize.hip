// Affine group quantization of dense 16-bit weights into MLX's packed format, for gfx950.
//
// Restates the published algorithm of MLX's affine quantize (mlx.core.quantize with
// mode="affine", mlx 0.32; the call sites are metile/backends/mlx_compressed_down.py:41-48 and
// the tests of metile/backends): per group of G consecutive elements of a row, with
// n = 2^bits - 1 and all arithmetic in fp32,
//   scale = max((max - min) / n, 1e-7), negated unless |min| > |max|;
//   edge  = min if |min| > |max| else max  (the extreme of larger magnitude);
//   q0    = rint(edge / scale); if q0 != 0: scale = edge / q0, bias = edge; else bias = 0,
// so the edge value maps to a code exactly. Scale and bias are rounded to the weights' 16-bit
// type; codes are rint((w - bias) / scale) with those rounded values, clamped to [0, n], and
// packed low bits first (code k of a row in word k / (32 / bits)).
#include "common.h"
#include "affine_quantize.h"

namespace mt {

namespace {

// A lane takes 8 consecutive weights, a group the G / 8 lanes beside each other (K is a multiple
// of G, so groups tile the flat array and never cross a wave). Extremes meet by lane exchanges in
// registers, so the weights are read once, 16 bytes a lane, and a lane's codes leave as one or two
// words beside its neighbours'. Bound by HBM (2 bytes in, bits / 8 out per weight): a bf16
// 14336 x 4096 weight to 4 bits in 32 us, 4.7 TB/s (one thread per group, reading two bytes at a
// time: 1098 us), to 8 bits 33 us (1318 us).
// VEC: w is 16-byte aligned and w_q 8-byte aligned; otherwise the same lanes move single elements.
template <int BITS, int DT, int LPG, bool VEC>
__global__ __launch_bounds__(256) void affine_quantize_kernel(const uint16_t* __restrict__ w,
                                                              uint32_t* __restrict__ w_q,
                                                              uint16_t* __restrict__ scales,
                                                              uint16_t* __restrict__ biases,
                                                              uint32_t chunks) {
  constexpr float kBins = (float)((1 << BITS) - 1);
  for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < chunks; t += gridDim.x * 256u) {
    float v[8];
    if constexpr (VEC) {
      const u32x4 raw = reinterpret_cast<const u32x4*>(w)[t];
      const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = lo16<DT>(words[i]);
        v[2 * i + 1] = hi16<DT>(words[i]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = act_to_f32<DT>(w[(size_t)t * 8 + e]);
    }
    float w_max = v[0], w_min = v[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) {
      w_max = fmaxf(w_max, v[e]);
      w_min = fminf(w_min, v[e]);
    }
    // Within LPG = 4, 8 or 16 lanes: quads, then halves of a row of 16, then the row. The loop's
    // bound is a multiple of LPG, so a group's lanes are in or out of it together.
    w_max = fmaxf(w_max, dpp_read<kDppXor1>(w_max));
    w_min = fminf(w_min, dpp_read<kDppXor1>(w_min));
    w_max = fmaxf(w_max, dpp_read<kDppXor2>(w_max));
    w_min = fminf(w_min, dpp_read<kDppXor2>(w_min));
    if constexpr (LPG >= 8) {
      w_max = fmaxf(w_max, dpp_read<kDppHalfMirror>(w_max));
      w_min = fminf(w_min, dpp_read<kDppHalfMirror>(w_min));
    }
    if constexpr (LPG >= 16) {
      w_max = fmaxf(w_max, dpp_read<kDppRowRor8>(w_max));
      w_min = fminf(w_min, dpp_read<kDppRowRor8>(w_min));
    }
    const bool low_edge = fabsf(w_min) > fabsf(w_max);
    float scale = fmaxf((w_max - w_min) / kBins, 1e-7f);
    if (!low_edge) scale = -scale;
    const float edge = low_edge ? w_min : w_max;
    const float q0 = rintf(edge / scale);
    float bias = 0.0f;
    if (q0 != 0.0f) {
      scale = edge / q0;
      bias = edge;
    }
    const uint16_t s16 = f32_to_act<DT>(scale);
    const uint16_t b16 = f32_to_act<DT>(bias);
    if (t % LPG == 0) {
      scales[t / LPG] = s16;
      biases[t / LPG] = b16;
    }
    const float s = act_to_f32<DT>(s16);
    const float b = act_to_f32<DT>(b16);
    // (w - b) / s correctly rounded, in three operations a weight: a first quotient from the
    // hardware reciprocal (a few ulp off), its residual (exact: s has at most 11 significant bits)
    // and one correction, which leaves an error of about 2^-21 ulp before its rounding; a quotient
    // by such an s is never that close to a rounding midpoint (at least 2^-12 ulp from one, or on
    // it only if exact). |s| is at least 5e-8. (The division itself: a
    // 14336 x 4096 weight in 47.8 us, this 32.2 us.)
    const float r = __builtin_amdgcn_rcpf(s);
    uint32_t word[2] = {0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = v[e] - b;
      const float first = a * r;
      const float quot = __builtin_fmaf(__builtin_fmaf(-s, first, a), r, first);
      const float q = fminf(fmaxf(rintf(quot), 0.0f), kBins);
      word[e * BITS / 32] |= (uint32_t)q << (e * BITS % 32);
    }
    if constexpr (BITS == 4) {
      w_q[t] = word[0];
    } else if constexpr (VEC) {
      reinterpret_cast<u32x2*>(w_q)[t] = (u32x2){word[0], word[1]};
    } else {
      w_q[(size_t)t * 2] = word[0];
      w_q[(size_t)t * 2 + 1] = word[1];
    }
  }
}

template <int BITS, int DT, bool VEC>
void launch(const uint16_t* w, uint32_t* w_q, uint16_t* scales, uint16_t* biases,
            uint32_t chunks, int G, int blocks, hipStream_t stream) {
  if (G == 32)
    affine_quantize_kernel<BITS, DT, 4, VEC><<<blocks, 256, 0, stream>>>(w, w_q, scales, biases,
                                                                         chunks);
  else if (G == 64)
    affine_quantize_kernel<BITS, DT, 8, VEC><<<blocks, 256, 0, stream>>>(w, w_q, scales, biases,
                                                                         chunks);
  else
    affine_quantize_kernel<BITS, DT, 16, VEC><<<blocks, 256, 0, stream>>>(w, w_q, scales, biases,
                                                                          chunks);
}

}  // namespace

hipError_t launch_affine_quantize(const uint16_t* w, uint32_t* w_q, uint16_t* scales,
                                  uint16_t* biases, int N, int K, int G, int bits, int dtype,
                                  hipStream_t stream) {
  const uint32_t chunks = (uint32_t)((size_t)N * K / 8);  // below 2^27: the tensor is under 2 GiB
  const uint32_t want = (chunks + 255) / 256;
  const int blocks = (int)(want < 16384 ? want : 16384);
  if (blocks == 0) return hipSuccess;
  const bool vec = (reinterpret_cast<uintptr_t>(w) & 15u) == 0 &&
                   (reinterpret_cast<uintptr_t>(w_q) & 7u) == 0;
  auto go = bits == 4 ? (dtype == kBF16 ? (vec ? launch<4, kBF16, true> : launch<4, kBF16, false>)
                                        : (vec ? launch<4, kF16, true> : launch<4, kF16, false>))
                      : (dtype == kBF16 ? (vec ? launch<8, kBF16, true> : launch<8, kBF16, false>)
                                        : (vec ? launch<8, kF16, true> : launch<8, kF16, false>));
  go(w, w_q, scales, biases, chunks, G, blocks, stream);
  return hipGetLastError();
}

}  // namespace mt
