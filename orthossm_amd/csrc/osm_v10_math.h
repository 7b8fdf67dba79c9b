// Per-token arithmetic that the full path and the fixed-coefficient forward
// share: the megakernel's softsign and the layout of its table in LDS.
#pragma once

#include "osm_device.h"

namespace osm {

constexpr float kLog2e = 1.4426950408889634f;
// Floats per LUT row in LDS: the 8 values of T_k padded to 12, so that the
// 16-byte reads of random rows by the lanes of a wave spread over more LDS
// banks than with 8 (rows i and i' collide when 12 (i - i') = 0 mod the
// bank count).  Measured on the full path at B=4 S=16384 D=512 on MI355X: 221
// against 227 us.
constexpr int kLutStride = 12;

// The megakernel's softsign: |u| and sign(u); NaN reads as 0.
__device__ __forceinline__ void v10_softsign(float xb, float& absu, float& sgn) {
  const float xs = xb == xb ? xb : 0.0f;
  const float ax = __builtin_fmaxf(__builtin_fabsf(xs), 1e-7f);
  absu = 1.0f - __builtin_amdgcn_rcpf(1.0f + ax);
  sgn = xs >= 0.0f ? 1.0f : -1.0f;
}

}  // namespace osm
