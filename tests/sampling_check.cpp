// Compares the splat's sampling transform (gps_rng.h corrected_box_muller_v,
// gps_detmath.h det_neg2_logf_normal and det_sincosf_u32, the source the GPU
// splat compiles) with the general functions it stands for, bit for bit:
//   logs:   every float in [2^-8, 1], every 61st below down to 1e-37
//   angles: every uint32 rounded to float (all 2^23 mantissas of the eight
//           binades up to 2^32, every integer below 2^24)
//   points: `n` random (u1, u2, alpha), with the extremes of each
// Prints the number of mismatches of each.  Zeros count as equal whatever
// their sign.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "gps_rng.h"

using namespace gps;

static bool same(float a, float b) { return f2u_bits(a) == f2u_bits(b) || (a == 0.0f && b == 0.0f); }

static bool same_angle(uint32_t k) {
    const float v = (float)k;
    float s0, c0, s1, c1;
    det_sincosf_inrange(GPS_TWO_PI_F * (v * 0x1.0p-32f), &s0, &c0);
    det_sincosf_u32(v, &s1, &c1);
    return same(s0, s1) && same(c0, c1);
}

static f32x2 general(float u1, float u2, float alpha) {
    const float q = det_div_li2max((1.0f - u1) * dilog(alpha));
    const float a = glm_clamp(corrected_inv_alpha(alpha) * inv_dilog_poly(1.0f < q ? 1.0f : q), 1.e-37f, 1.0f);
    const float R = det_sqrt(det_fmax(-2.0f * det_logf(a), 0.0f));
    float s, c;
    det_sincosf(GPS_TWO_PI_F * u2, &s, &c);
    return f32x2{R * c, R * s};
}

int main(int argc, char** argv) {
    const uint32_t n = argc > 1 ? (uint32_t)atoi(argv[1]) : 4000000u;
    uint64_t logs = 0, angles = 0, points = 0;
    for (uint32_t ix = f2u_bits(1.0f); ix >= f2u_bits(1.e-37f); ix -= ix > f2u_bits(0x1.0p-8f) ? 1u : 61u) {
        const float a = u2f_bits(ix);
        const float ref = -2.0f * det_logf_normal(a);
        logs += !(same(ref, det_neg2_logf_normal(a)) && ref >= 0.0f);
    }
    for (uint32_t k = 0; k < (1u << 24); ++k) angles += !same_angle(k);
    for (int b = 24; b < 32; ++b)
        for (uint32_t m = 0; m < (1u << 23); ++m) angles += !same_angle((uint32_t)((1ull << b) + ((uint64_t)m << (b - 23))));
    angles += !same_angle(0xFFFFFFFFu);
    const uint32_t edge[6] = {0u, 1u, 0x7FFFFFFFu, 0x80000000u, 0xFFFFFF00u, 0xFFFFFFFFu};
    const float alpha_edge[6] = {1.0f, 0.99999994f, 1.0f / 255.0f, 1e-6f, 1e-30f, 1e-38f};
    for (uint32_t i = 0; i < n; ++i) {
        u32x2 st = make_seed(i, 7u);
        float alpha = (float)hash32(i ^ 0x51u) * 0x1.0p-32f;
        if (i < 36u * 6u) {
            st.x = edge[i % 6u];
            st.y = edge[i / 6u % 6u];
            alpha = alpha_edge[i / 36u];
        }
        const f32x2 r = general((float)st.x * 0x1.0p-32f, (float)st.y * 0x1.0p-32f, alpha);
        const f32x2 g = corrected_box_muller_v((float)st.x, (float)st.y, corrected_inv_alpha(alpha), dilog(alpha));
        points += !(same(r.x, g.x) && same(r.y, g.y));
    }
    printf("%llu %llu %llu\n", (unsigned long long)logs, (unsigned long long)angles, (unsigned long long)points);
    return 0;
}
