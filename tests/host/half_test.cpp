// Host unit test of the float16 pass's arithmetic and of the rule that selects
// it (namitorch_amd/csrc/nt_half.hpp).  Built by tests/test_host_tables.py with
// g++ and AddressSanitizer/UBSan; no GPU.
//
// The device computes a quotient or root of float16 values with
// quotient_step/root_step from the hardware's reciprocal or reciprocal root
// (within one fp32 ulp) and rounds it to float16; NumPy rounds the IEEE fp32
// result.  A float16 value is an 11-bit significand times a power of two, and
// no step leaves fp32's normal range, so the steps of a pair depend on its
// significands alone and its rounding on the quotient's exponent as well: all
// 1024 x 1024 normalized significands at every exponent a quotient can have
// are all pairs.  Signs mirror; v_div_fixup_f32 gives zeros, infinities and NaN.
#include <cmath>
#include <cstdio>
#include <initializer_list>

#include "../../namitorch_amd/csrc/nt_half.hpp"

using namespace nt;

static int failures = 0;
#define CHECK(cond)                                                              \
    do {                                                                         \
        if (!(cond)) {                                                           \
            if (failures < 20) std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
            ++failures;                                                          \
        }                                                                        \
    } while (0)

// A nonnegative fp32 value rounded to float16 (nearest even), as a double.
static double to_half(float x) {
    const double a = x;
    if (!(a < 65520.0)) return a >= 65520.0 ? (double)INFINITY : a;
    const double quantum = a < 0x1p-14 ? 0x1p-24 : std::ldexp(1.0, std::ilogb(a) - 10);
    return std::nearbyint(a / quantum) * quantum;
}

// `x` and its two neighbours: what an instruction exact to one ulp may return.
static float off_by(float x, int ulps) { return ulps == 0 ? x : nextafterf(x, ulps < 0 ? 0.0f : INFINITY); }

static void test_every_quotient() {
    long differing = 0;
    for (int mb = 1024; mb < 2048; ++mb) {
        const float b = (float)mb * 0x1p-10f;             // [1, 2)
        for (int ulps = -1; ulps <= 1; ++ulps) {
            const float inv = off_by((float)(1.0 / (double)b), ulps);
            for (int ma = 1024; ma < 2048; ++ma) {
                const float a = (float)ma * 0x1p-10f;
                const float exact = a / b, got = quotient_step(a, b, inv);
                if (exact == got) continue;               // equal bits round alike at every exponent
                ++differing;
                // 2**-24 / 65504 to 65504 / 2**-24
                for (int e = -41; e <= 41; ++e) CHECK(to_half(ldexpf(exact, e)) == to_half(ldexpf(got, e)));
            }
        }
    }
    std::printf("%ld of %d quotients differ from the fp32 one\n", differing, 3 * 1024 * 1024);
    // The exponent itself, at the ends of what the operands allow.
    for (float a : {0x1p-24f, 0x1.8p-23f, 1.0f, 1.5f, 65504.0f})
        for (float b : {0x1p-24f, 0x1.8p-23f, 1.0f, 1.5f, 65504.0f})
            for (int ulps = -1; ulps <= 1; ++ulps)
                CHECK(to_half(quotient_step(a, b, off_by((float)(1.0 / (double)b), ulps))) == to_half(a / b));
}

static void test_every_root() {
    for (int bits = 1; bits < 0x7c00; ++bits) {           // every positive finite float16 value
        const int e = bits >> 10, m = bits & 1023;
        const float x = e == 0 ? ldexpf((float)m, -24) : ldexpf((float)(1024 + m), e - 25);
        for (int ulps = -1; ulps <= 1; ++ulps) {
            const float y = off_by((float)(1.0 / std::sqrt((double)x)), ulps);
            CHECK(to_half(root_step(x, y)) == to_half(sqrtf(x)));
        }
    }
}

static float half(double x) { return (float)to_half((float)x); }

// An optimizer's coefficients for float16 parameters.
static nt_adamw_coefs adamw() {
    nt_adamw_coefs c{};
    c.lr = half(0.001), c.beta1 = half(0.9), c.beta2 = half(0.999), c.complement1 = half(0.1);
    c.complement2 = half(0.001), c.eps = half(1e-4), c.weight_decay = half(0.1), c.decay_factor = half(1 - 1e-4);
    c.correction1 = half(0.41), c.correction2 = half(0.005), c.update_parameter = 1;
    return c;
}

static void test_which_launches_are_lean() {
    CHECK(half_value(0.0f) && half_value(-65504.0f) && half_value(0x1p-24f) && half_value(0x1.ffcp0f));
    CHECK(!half_value(65520.0f) && !half_value(0x1p-25f) && !half_value(0x1.8p-24f) && !half_value(0x1.ffep0f));
    CHECK(!half_value(INFINITY) && !half_value(NAN));
    nt_adamw_coefs slots[2] = {adamw(), adamw()};
    CHECK(half_lean_slots(slots, 1) && half_lean_slots(slots, 2));
    slots[0].weight_decay = 0.0f;
    CHECK(half_lean_slots(slots, 2));
    auto refused = [](auto change) {
        nt_adamw_coefs one[2] = {adamw(), adamw()};
        change(one[1]);
        return half_lean_slots(one, 1) && !half_lean_slots(one, 2);   // the second slot alone
    };
    CHECK(refused([](nt_adamw_coefs &c) { c.lr = 0.0003f; }));
    CHECK(refused([](nt_adamw_coefs &c) { c.eps = 1e-8f; }));
    CHECK(refused([](nt_adamw_coefs &c) { c.correction1 = 0.0f; }));
    CHECK(refused([](nt_adamw_coefs &c) { c.correction2 = 0.0f; }));
    CHECK(refused([](nt_adamw_coefs &c) { c.maximize = 1; }));
    CHECK(refused([](nt_adamw_coefs &c) { c.coupled_weight_decay = 1; }));
    CHECK(refused([](nt_adamw_coefs &c) { c.update_parameter = 0; }));
}

int main() {
    test_every_quotient();
    test_every_root();
    test_which_launches_are_lean();
    if (failures != 0) {
        std::printf("%d checks failed\n", failures);
        return 1;
    }
    std::printf("all checks passed\n");
    return 0;
}
