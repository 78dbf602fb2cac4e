// CPU check of the one-multiply-one-FMA forms of birp_cpp_amd/csrc/exact_math.h.
//   scale        birp_scale_fma2 == birp_scale_chain for every significand, at several exponents
//   div <b>      birp_div_fma2(a, RN(1/b), RN(1/b - RN(1/b))) == a / b for every significand of a
//   lerp <seed>  birp_lerp_unit == std::lerp for pairs without a sign change and t in [0, 1 - 2^-24]
// Prints "mismatches N checked M" and exits 0 when N == 0.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include "../../birp_cpp_amd/csrc/exact_math.h"

static float f_of(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }

int main(int argc, char** argv) {
    unsigned long long bad = 0, checked = 0;
    if (argc == 2 && !strcmp(argv[1], "scale")) {
        const int exps[] = {-100, -37, 0, 41, 109};
        for (int e : exps)
            for (uint32_t m = 0; m < (1u << 23); m++, checked++) {
                const float v = f_of((uint32_t)(127 + e) << 23 | m);
                bad += birp_scale_fma2(v) != birp_scale_chain(v);
            }
    } else if (argc == 3 && !strcmp(argv[1], "div")) {
        const float b = strtof(argv[2], 0);
        volatile float one = 1.0f;
        const float rh = one / b, rl = (float)(std::fma(-(double)rh, (double)b, 1.0) / (double)b);
        for (uint32_t m = 0; m < (1u << 23); m++, checked++) {
            const float a = f_of(127u << 23 | m);
            volatile float q = a / b;
            bad += birp_div_fma2(a, rh, rl) != q;
        }
    } else if (argc == 3 && !strcmp(argv[1], "lerp")) {
        std::mt19937 g((unsigned)atoi(argv[2]));
        for (int i = 0; i < 20000000; i++, checked++) {
            const uint32_t x = g(), y = g(), z = g();
            // neighbours within 2^15 ulps, pairs of any ratio, subnormals, zero first corners
            const uint32_t ua = (z & 8) ? x >> 1 & 0x00FFFFFFu : (100u + (x >> 27)) << 23 | (x & 0x7FFFFFu);
            uint32_t ub = (z & 1) ? (100u + (y >> 27)) << 23 | (y & 0x7FFFFFu) : ua + (y & 0xFFFFu);
            const float t = (z & 2) ? 1.0f - std::ldexp((float)(1 + (z >> 28)), -24) : (float)(z >> 8) * 0x1p-24f;
            float a = (z & 4 && (z & 0xF0) == 0) ? 0.0f : f_of(ua), b = f_of(ub ? ub : 1u);
            if (z & 16 && a > 0) { const float s = a; a = b; b = s; }
            if (z & 32 && a > 0) { a = -a; b = -b; }
            const float r = std::lerp(a, b, t), u = birp_lerp_unit(a, b, t);
            bad += r != u;
        }
    } else return 2;
    printf("mismatches %llu checked %llu\n", bad, checked);
    return bad == 0 ? 0 : 1;
}
