// Decode-layer launches of the token step that have no C entry point of their own.
#pragma once

#include <stdint.h>

#include "grout_attn_hip.h"

namespace grout {

// residual_out = residual + x; out = weight [m, k] @ RMSNorm(residual + x), or
// with `silu` SiLU(gate) * up of the [2m, k] gate_up weight: add_rms_norm_decode
// and the GEMV behind it (src/model.rs:3151-3176, :3513-3565) in one launch.
// residual_out must not be residual or x: every workgroup reads both.  For k up
// to the limit of add_norm_gemv_fits.
bool add_norm_gemv_fits(int32_t k);
int32_t add_norm_gemv(const uint16_t* residual, const uint16_t* x, const uint16_t* norm_weight,
                      uint16_t* residual_out, float eps, const uint16_t* weight, uint16_t* out, int32_t m,
                      int32_t k, bool silu, grout_stream_t stream);

}  // namespace grout
