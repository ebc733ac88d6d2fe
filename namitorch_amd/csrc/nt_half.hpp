// nt_half.hpp — the float16 pass's arithmetic between its hardware
// instructions, and the rule for the launches that use it (lean_slice_f16).
//
// Plain code on plain floats, so the same lines also compile with a host
// compiler: the host unit test (tests/host/half_test.cpp) runs every pair of
// float16 significands through them.
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>

#include "../../include/namitorch_amd.h"

#if defined(__HIPCC__)
#define NT_HALF_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define NT_HALF_FN inline
#endif

namespace nt {

// a / b before its rounding to float16, for finite nonzero float16 values a
// and b; `inv` is 1 / b to within an fp32 ulp.
NT_HALF_FN float quotient_step(float a, float b, float inv) {
    const float q = a * inv;
    return __builtin_fmaf(__builtin_fmaf(-q, b, a), inv, q);
}

// sqrt(x) before its rounding to float16, for a positive finite float16
// value; `y` is 1 / sqrt(x) to within an fp32 ulp.
NT_HALF_FN float root_step(float x, float y) {
    const float s = x * y;
    return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
}

// Whether `x` is a finite float16 value.
inline bool half_value(float x) {
    const float a = fabsf(x);
    if (!(a <= 65504.0f)) return false;
    uint32_t bits;
    memcpy(&bits, &a, sizeof(bits));
    if (a >= 0x1p-14f) return (bits & 0x1fffu) == 0u;            // normal: 11 significand bits
    return a * 0x1p24f == floorf(a * 0x1p24f);                   // a multiple of the smallest
}

// Whether coefficient slots [0, n) all allow lean_slice_f16: AdamW without
// maximize, parameters updated, and coefficients that are float16 values (the
// options rounded to float16, but for a caller of the C ABI that passes others)
// with bias corrections it can divide by through their inverse.
inline bool half_lean_slots(const nt_adamw_coefs *slots, uint32_t n) {
    for (uint32_t i = 0; i < n; ++i) {
        const nt_adamw_coefs &c = slots[i];
        if (c.maximize || c.coupled_weight_decay || !c.update_parameter) return false;
        for (float x : {c.lr, c.beta1, c.beta2, c.complement1, c.complement2, c.eps, c.weight_decay, c.decay_factor,
                        c.correction1, c.correction2})
            if (!half_value(x)) return false;
        if (!(c.correction1 > 0.0f && c.correction2 > 0.0f)) return false;
    }
    return true;
}

}  // namespace nt
