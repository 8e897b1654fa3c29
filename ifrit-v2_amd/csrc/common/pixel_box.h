// A proven pixel box of a triangle, so that the raster looks at the pixels a
// small triangle can cover instead of walking its tiles' blocks.
//
// Coverage tests every edge at a sample as fma(ey, y, ex * x) < -ez in FP32.
// The box returned here holds every pixel any of whose samples can pass all
// three tests.  The triangle's own extent would not do: the edge constants
// carry a bias of 1e-8 W H and the rounding of sums far larger than the
// triangle, which move the edges of pixel-sized triangles by tenths of a pixel
// and those of thinner ones by whole pixels.
//
// Bound.  A sample P that passes edge k satisfies s_k(P) = ex x + ey y + ez <
// d_k with d_k = 2.01 u (|ex| W + |ey| H), the rounding of the test (u = 2^-24).
// For any point V, s_k(P) = n_k . (P - V) + s_k(V), so n_k . (P - V) < a_k with
// a_k = d_k - s_k(V).  With D_ij = n_i x n_j of one sign and away from 0 for all
// three pairs the half-planes bound a triangle whose corners are V_ij + q with
// n_i . q = a_i, n_j . q = a_j.  V_ij are the projected vertices as computed
// here.  a_k is evaluated as -s_k(V), off by less than r = 8 u max(|ex| W +
// |ey| H + |ez|) in all; that moves a corner by at most 2 r M / |D| per axis (M
// the largest |ex|, |ey|), and the rounding of D (under 8 u M^2) by its share of
// |q|.
#pragma once
#include "x86_fp.h"

namespace ifx {

// x0 | y0 << 16 and x1 | y1 << 16, inclusive; x0 > x1 where no pixel is covered.  The
// low end is clamped to 0, the high end only to 16 bits: whether a pixel's 2x2
// quad is covered, which selects its depth expression, does not stop at the
// target's right and lower edge.
struct PixelBox {
    uint32_t lo, hi;
};
IFX_HD PixelBox whole_target() { return PixelBox{0u, 0xffffffffu}; }

IFX_HD float fabs1(float a) { return u2f(f2u(a) & 0x7fffffffu); }
#if defined(__HIP_DEVICE_COMPILE__)
IFX_HD float fma1(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
IFX_HD float max1(float a, float b) { return __builtin_fmaxf(a, b); }
IFX_HD float min1(float a, float b) { return __builtin_fminf(a, b); }
IFX_HD float rcp1(float a) { return __builtin_amdgcn_rcpf(a); }  // 1 ulp
#else
IFX_HD float fma1(float a, float b, float c) { return fmaf(a, b, c); }
IFX_HD float max1(float a, float b) { return fmaxf(a, b); }
IFX_HD float min1(float a, float b) { return fminf(a, b); }
IFX_HD float rcp1(float a) { return 1.0f / a; }
#endif

// Vertices (x, y) in NDC, with edge k between vertices k and k + 1 (mod 3), whose
// coefficients are e[k] = (ex, ey, ez); the target's size and whether samples
// lie inside the pixels (msaa) or on their corners.  whole_target() where the
// bound does not apply (a vertex far outside, a degenerate triangle).
IFX_HD PixelBox pixel_box(const float* x, const float* y, const float e[3][3], int width, int height, bool msaa) {
    constexpr float u = 5.9604645e-8f;  // 2^-24
    const float hw = 0.5f * (float)width, hh = 0.5f * (float)height;
    const float W = (float)width + 64.0f, H = (float)height + 64.0f;
    float X[3], Y[3], D[3];
    float M = 0.0f, A = 0.0f;
    for (int k = 0; k < 3; k++) {
        const int j = k == 0 ? 2 : k - 1;
        X[k] = fma1(x[k], hw, hw);
        Y[k] = fma1(y[k], hh, hh);
        const float ax = fabs1(e[k][0]), ay = fabs1(e[k][1]);
        M = max1(M, max1(ax, ay));
        A = max1(A, fma1(ax, W, fma1(ay, H, fabs1(e[k][2]))));
        D[k] = fma1(e[k][0], e[j][1], neg(e[k][1] * e[j][0]));  // vertex k meets edges k and k - 1
    }
    const float dlo = min1(D[0], min1(D[1], D[2])), dhi = max1(D[0], max1(D[1], D[2]));
    const float e8 = 8.0f * u * (M * M);
    const float Dm = max1(dlo, neg(dhi)) - e8;  // below every |D|, and positive only if they share a sign
    float q = 0.0f, x0 = 0.0f, x1 = 0.0f, y0 = 0.0f, y1 = 0.0f, far = 0.0f;
    for (int k = 0; k < 3; k++) {
        const int j = k == 0 ? 2 : k - 1;
        const float ai = neg(fma1(e[k][0], X[k], fma1(e[k][1], Y[k], e[k][2])));
        const float aj = neg(fma1(e[j][0], X[k], fma1(e[j][1], Y[k], e[j][2])));
        const float rd = rcp1(D[k]);
        const float qx = fma1(ai, e[j][1], neg(aj * e[k][1])) * rd, qy = fma1(aj, e[k][0], neg(ai * e[j][0])) * rd;
        q = max1(q, max1(fabs1(qx), fabs1(qy)));
        far = max1(far, max1(max1(-64.0f - X[k], X[k] - W), max1(-64.0f - Y[k], Y[k] - H)));
        const float cx = X[k] + qx, cy = Y[k] + qy;
        x0 = k ? min1(x0, cx) : cx;
        x1 = k ? max1(x1, cx) : cx;
        y0 = k ? min1(y0, cy) : cy;
        y1 = k ? max1(y1, cy) : cy;
    }
    // margin = 2 r M / |D| for a_k, the share of D's rounding in q (and of the products' in q, within
    // the same bound), 2^-8 for the rounding of coordinates below 2^15
    const float num = fma1(2.1f * 8.0f * u * A, M, 3.0f * e8 * q);
    if (!(Dm > 1e-25f && M < 1e15f && A < 1e30f && far <= 0.0f && num <= 64.0f * Dm && q < 64.0f)) return whole_target();
    const float m = fma1(num, rcp1(Dm), 0.00390625f);
    x0 -= m;
    y0 -= m;
    // a pixel's samples lie in [px, px + 1), or at px on its corner
    const int bx0 = (int)(msaa ? __builtin_floorf(x0) : __builtin_ceilf(x0));
    const int by0 = (int)(msaa ? __builtin_floorf(y0) : __builtin_ceilf(y0));
    const int bx1 = (int)__builtin_floorf(x1 + m), by1 = (int)__builtin_floorf(y1 + m);
    const int lx = bx0 < 0 ? 0 : bx0, ly = by0 < 0 ? 0 : by0;
    if (bx1 < lx || by1 < ly) return PixelBox{1u, 0u};
    return PixelBox{(uint32_t)lx | ((uint32_t)ly << 16), (uint32_t)bx1 | ((uint32_t)by1 << 16)};
}

}  // namespace ifx
