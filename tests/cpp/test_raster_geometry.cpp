// rvs_math.h's quotients that share a divisor, the rejection by approximate
// barycentrics and the near box, against plain division and a scan of every
// pixel.  The reciprocal is within an ulp, as the device's instruction; for the
// largest mantissa it is the rounded one (the steps, which are those of the
// device's own division, need it there).
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

static uint32_t g_rng = 12345u;
static inline float near_rcp(float x) {
    const float r = 1.0f / x;
    uint32_t xb;
    std::memcpy(&xb, &x, 4);
    if (!std::isfinite(r) || r == 0.f || (xb & 0x7fffffu) == 0x7fffffu) return r;
    g_rng = g_rng * 1664525u + 1013904223u;
    uint32_t u;
    std::memcpy(&u, &r, 4);
    u += (g_rng >> 16) % 3u - 1u;
    float o;
    std::memcpy(&o, &u, 4);
    // 1/x rounded, one float up or down, can be 1.5 ulp away: only what is within one
    const double exact = 1.0 / (double)x, ulp = std::ldexp(1.0, std::ilogb(exact) - 23);
    return std::fabs((double)o - exact) <= ulp ? o : r;
}
#define RVS_MATH_TEST_RCP near_rcp
#include "../../rvs-cuda_amd/csrc/rvs_math.h"
using namespace rvs_math;

static std::mt19937_64 rng(7);
static float uni(float a, float b) { return std::uniform_real_distribution<float>(a, b)(rng); }
static float bits(int elo, int ehi) {   // random mantissa (often all ones or nearly), exponent in [elo, ehi]
    uint32_t m = (uint32_t)rng() & 0x7fffffu;
    const int kind = (int)(rng() % 8);
    if (kind == 0) m = 0x7fffffu - (m & 7u);
    if (kind == 1) m &= 7u;
    return u2f(((uint32_t)(elo + 127 + (int)(rng() % (uint64_t)(ehi - elo + 1))) << 23) | m);
}

static long quotients(long n) {
    long bad = 0;
    for (long k = 0; k < n; ++k) {
        const float d = k % 16 == 0 ? (k % 32 ? 9.313225746e-10f : 1.099511628e12f) : bits(-30, 39);
        float a = bits(-50, 59) * (rng() & 1 ? -1.f : 1.f);
        if (k % 3 == 0) a = d * bits(-20, 0) * (rng() & 1 ? -1.f : 1.f);   // the barycentrics' range
        if (!quot_den(d) || !quot_num(a)) continue;
        const float q = quot(a, d, recip(d)), e = a / d;
        if (std::fabs(e) < 2e-38f) continue;
        bad += f2u(q) != f2u(e);
    }
    return bad;
}

static float coord(int kind) {
    switch (kind) {
    case 0: return uni(-3.f, 45.f);
    case 1: return uni(-300.f, 400.f);
    case 2: return uni(10.f, 14.f);
    case 3: return (float)(int)uni(-2.f, 40.f) * 0.5f;
    case 4: return uni(-1e6f, 1e6f);
    default: {
        const float s[] = {INFINITY, -INFINITY, NAN, 3e9f, -3e9f, 1e20f, -1e20f, 2147483648.f, 0.f};
        return s[rng() % 9];
    }
    }
}

int main() {
    const long bad_q = quotients(20000000);
    long boxed = 0, outside = 0, missed = 0, wrong = 0, rejected = 0, covered = 0;
    const int W = 41, H = 33;
    for (long k = 0; k < 400000; ++k) {
        const int kind = (int)(k % 6);
        float c[6];
        for (float& x : c) x = coord(kind == 5 && rng() % 3 ? 0 : kind);
        if (kind == 2) for (int m = 2; m < 6; ++m) c[m] = c[m % 2] + uni(-2.5f, 2.5f);
        const float A0 = c[0], A1 = c[1], B0 = c[2], B1 = c[3], C0 = c[4], C1 = c[5];
        const float den = (B1 - C1) * (A0 - C0) + (C0 - B0) * (A1 - C1);
        if (den <= 0.f) continue;
        const float xs[3] = {A0, B0, C0}, ys[3] = {A1, B1, C1};
        // colorize_triangle's box
        const int xmin = imax(0, cvt_i32(std::floor(smin(smin(xs[0], xs[1]), xs[2]))));
        const int ymin = imax(0, cvt_i32(std::floor(smin(smin(ys[0], ys[1]), ys[2]))));
        const int xmax = imin(W - 1, cvt_i32(std::ceil(smax(smax(xs[0], xs[1]), xs[2]))));
        const int ymax = imin(H - 1, cvt_i32(std::ceil(smax(smax(ys[0], ys[1]), ys[2]))));
        int xa = 0, xb = W - 1, ya = 0, yb = H - 1;
        const bool box = tri_near_box(A0, A1, B0, B1, C0, C1, den, 0, W - 1, 0, H - 1, xa, xb, ya, yb);
        boxed += box;
        const bool fast = cover_den(den);
        const float r = fast ? recip(den) : 0.f;
        for (int y = ymin; y <= ymax; ++y)
            for (int x = xmin; x <= xmax; ++x) {
                const float px = (float)x + 0.5f, py = (float)y + 0.5f;
                const float n1 = (B1 - C1) * (px - C0) + (C0 - B0) * (py - C1);
                const float n2 = (C1 - A1) * (px - C0) + (A0 - C0) * (py - C1);
                const float l1 = n1 / den, l2 = n2 / den, l3 = 1.f - l1 - l2;
                const bool in = l1 >= -1e-6f && l2 >= -1e-6f && l3 >= -1e-6f;
                covered += in;
                if (box && in && (x < xa || x > xb || y < ya || y > yb)) ++outside;
                const float a1 = n1 * r, a2 = n2 * r;
                const bool rej = min3f(a1, a2, 1.f - a1 - a2) < -2e-6f;
                rejected += rej;
                if (rej && in) ++missed;
                if (!fast) continue;
                const float q1 = quot(n1, den, r), q2 = quot(n2, den, r), q3 = 1.f - q1 - q2;
                const bool qin = q1 >= -1e-6f && q2 >= -1e-6f && q3 >= -1e-6f;
                if (qin != in) ++wrong;
                if (in && quot_den(den) && quot_num(n1) && quot_num(n2) && (f2u(q1) != f2u(l1) || f2u(q2) != f2u(l2))) ++wrong;
            }
    }
    std::printf("quotients %ld wrong; boxes %ld, covered %ld, outside %ld; rejected %ld, missed %ld; coverage %ld wrong\n",
                bad_q, boxed, covered, outside, rejected, missed, wrong);
    return bad_q || outside || missed || wrong || boxed < 10000 || covered < 100000 || rejected < 100000;
}
