// One head row of any dim up to 64 in any storage dtype: element access and the
// LayerNorm that the head-dim-generic kernels share.
#pragma once

#include "prime_common.h"

namespace prime {

// round to storage dtype dt (to nearest even), as a module's tensor of that dtype holds it
__device__ __forceinline__ float round_dt(float x, int dt) {
    if (dt == PRIME_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(x));
    if (dt == PRIME_F16) return h16_bits_to_f32(f32_to_h16_bits(x));
    return x;
}

// One head row of D values in place: LayerNorm over D (biased variance;
// weight w / bias bb, or none when w is null), rounded to the storage dtype
// dt as the module's LayerNorm returns it, then the scale (rounded again).
// The prefill's QK-norm on load and prime_head_layernorm share it, so both
// give the same bits.
__device__ __forceinline__ void generic_ln_row(float *row, int D, const void *w, const void *bb, int dt_norm,
                                               float ln_eps, float scale, int dt) {
    if (w) {
        float m = 0.f;
        for (int i = 0; i < D; ++i) m += row[i];
        m /= static_cast<float>(D);
        float var = 0.f;
        for (int i = 0; i < D; ++i) var += (row[i] - m) * (row[i] - m);
        const float rs = rsqrtf(var / static_cast<float>(D) + ln_eps);
        for (int i = 0; i < D; ++i) row[i] = round_dt((row[i] - m) * rs * load_elem(w, i, dt_norm) + load_elem(bb, i, dt_norm), dt);
    }
    if (scale != 1.0f)
        for (int i = 0; i < D; ++i) row[i] = round_dt(row[i] * scale, dt);
}

}  // namespace prime
