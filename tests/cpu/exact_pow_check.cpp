// CPU check of the square root and the power of birp_cpp_amd/csrc/exact_math.h.
//   sqrt <e>     birp_sqrt_rn(a, y) == sqrt(a) for every significand of a in [2^e, 2^(e + 2)), y = 1 / sqrt(a)
//                off by -8 .. 8 ulps
//   pow <seed>   birp_powf(b, e) within 0.5 + 2^-9 float ulps of the long double power, over b in the model's
//                range and in all that birp_powf_takes accepts, and inf, 0 and subnormals past the float range
// Prints "mismatches N checked M" and exits 0 when N == 0.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include "../../birp_cpp_amd/csrc/exact_math.h"

int main(int argc, char** argv) {
    unsigned long long bad = 0, checked = 0;
    if (argc != 3) return 2;
    if (!strcmp(argv[1], "sqrt")) {
        const int e = atoi(argv[2]);
        for (uint32_t m = 0; m < (1u << 24); m++, checked++) {
            const float a = birp_f32_of(((uint32_t)(127 + e) << 23) + m), y = (float)(1.0 / std::sqrt((double)a));
            const int off = (int)(m * 2654435761u >> 16) % 17 - 8;
            bad += birp_sqrt_rn(a, birp_f32_of(birp_f32_bits(y) + (uint32_t)off)) != std::sqrt(a);
        }
    } else if (!strcmp(argv[1], "pow")) {
        std::mt19937 g((unsigned)atoi(argv[2]));
        double worst = 0;
        for (int i = 0; i < 8000000; i++) {
            const float u = (float)(g() >> 8) * 0x1p-24f, w = (float)(g() >> 8) * 0x1p-24f;
            float b, e;
            if (i & 1) b = 0.05f + 12.0f * u, e = -14.0f + 28.0f * w;               // distances / 10, exponents
            else if (i & 2) b = 1.0f + 0x1p-10f * (u - 0.5f), e = -4096.0f + 8192.0f * w;  // near 1
            else b = birp_f32_of(0x0F800000u + g() % 0x60000000u), e = -2.0f + 4.0f * w;
            if (!birp_powf_takes(b, e)) { bad++; continue; }
            const long double want = powl((long double)b, (long double)e);
            const float got = birp_powf(b, e);
            checked++;
            if (want >= 0x1p128L || want < 0x1p-126L) {  // overflow; subnormals and 0: absolute
                const float f = (float)want;
                bad += std::isinf(f) ? !std::isinf(got) && got < 0x1.fffffep127f : std::fabs((double)got - (double)f) > 0x1p-149;
                continue;
            }
            const long double ulp = std::ldexp(1.0L, std::ilogb(want) - 23), err = std::fabs((long double)got - want) / ulp;
            if (err > worst) worst = (double)err;
            bad += err > 0.5L + 0x1p-9L && !(std::isinf(got) && want > 0x1.fffffep127L);
        }
        const struct { float b, e, r; } exact[] = {{1, 0, 1}, {3, 0, 1}, {1, 5, 1}, {2, 3, 8}, {4, -0.5f, 0.5f}, {9, 0.5f, 3}};
        for (auto& x : exact) bad += birp_powf(x.b, x.e) != x.r;
        bad += birp_powf_takes(0.0f, 1) || birp_powf_takes(-1.0f, 1) || birp_powf_takes(INFINITY, 1) || birp_powf_takes(NAN, 1) ||
               birp_powf_takes(0x1p-97f, 1) || birp_powf_takes(0x1p96f, 1) || birp_powf_takes(2, INFINITY) || birp_powf_takes(2, NAN) ||
               birp_powf_takes(2, -0x1p20f);
        printf("worst %.5f ulp ", worst);
    } else return 2;
    printf("mismatches %llu checked %llu\n", bad, checked);
    return bad == 0 ? 0 : 1;
}
