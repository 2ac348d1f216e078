// The demultiplied channel of a PNG pixel: the rule in f64, and the f32 form that the rows'
// kernel evaluates with factors chosen so that it gives the rule's value.  Host and device
// share the f32 expression, so what the host checks is what the kernel runs.
#pragma once
#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#define RVK_HOST_DEVICE __host__ __device__ inline
#else
#define RVK_HOST_DEVICE inline
#endif

namespace rvk_png {

constexpr int kSpecial = 6;

// per alpha the factor r, at least 1, or k / 8 where table row k holds the values
struct Demul {
    float r[256];
    uint8_t special[kSpecial][256];
};

// The f64 rule for channel c at alpha a.
inline uint32_t demul_rule(uint32_t c, uint32_t a) {
    if (a == 255u) return c;
    const double d = (double)c / ((double)a / 255.0) + 0.5;
    return d != d ? 0u : d >= 255.0 ? 255u : d <= 0.0 ? 0u : (uint32_t)d;
}

// floor(c r + 0.5) with one rounding, at most 255.  The factors are at most 1024 (at alpha 0,
// where every channel but 0 gives 255), so the sum is well within an integer's range, out of
// which the conversion would be undefined.
RVK_HOST_DEVICE uint32_t straight_channel(uint32_t c, float r) {
    const uint32_t v = (uint32_t)fmaf((float)c, r, 0.5f);
    return v < 255u ? v : 255u;
}
RVK_HOST_DEVICE bool by_table(float r) { return r < 1.0f; }
RVK_HOST_DEVICE int table_row(float r) { return (int)(8.0f * r); }

inline bool make_demul(Demul &t) {
    int nspecial = 0;
    for (uint32_t a = 0; a < 256; a++) {
        const float r0 = a ? 255.0f / (float)a : 1024.0f;
        const float tries[3] = {r0, std::nextafter(r0, 0.0f), std::nextafter(r0, 1e38f)};
        bool found = false;
        for (int k = 0; k < 3 && !found; k++) {
            found = true;
            for (uint32_t c = 0; c < 256 && found; c++) found = straight_channel(c, tries[k]) == demul_rule(c, a);
            t.r[a] = tries[k];
        }
        if (found && !by_table(t.r[a])) continue;
        if (nspecial == kSpecial) return false;
        for (uint32_t c = 0; c < 256; c++) t.special[nspecial][c] = (uint8_t)demul_rule(c, a);
        t.r[a] = (float)nspecial++ / 8.0f;
    }
    return true;
}

}  // namespace rvk_png
