// FP32-shifted moments and collisions with every rounding written out.
//
// d2q9_f32.h leaves it to the compiler which multiplications and additions
// it fuses, and that depends on the code around them: the same source rounds
// differently in two kernels.  The kernels that must agree bit for bit (the
// bulk stream-collide of a single case and of the serving engine, the tiled
// step) take their arithmetic from here: uncontracted, with the fused
// operations as explicit fused multiply-adds.
//
// SITE selects between the two roundings in use: false, the bulk
// stream-collide's, which rounds some products before they are added; true,
// the support sites', fused throughout.  Both are the same expressions; `mad`
// marks where they differ.  Which products those are has no numerical reason: it
// is how the two kernels were contracted when their results became the ones to
// keep, bit for bit.  FORCE false: the site's force is zero, whose
// terms (a zero each) are left out.
#pragma once

#include "d2q9_f32.h"

namespace life {

#pragma clang fp contract(off)

LIFE_DF float fmaf_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// a * b + c with one rounding (SITE) or two.
template <bool SITE>
LIFE_DF float mad(float a, float b, float c) {
    return SITE ? __builtin_fmaf(a, b, c) : a * b + c;
}

// x * w_v with w_v = k / 36 (see wmul): k = 16, 4 or 1, kx = k * x exactly.
LIFE_DF float w36(float kx) { return fmaf_(kx, kW36hi, kx * kW36lo); }

// Moments of one site.  nx, ny: momentum + F/2; inv: 1 / rho.
struct Moments32 {
    float drho, nx, ny, inv, ux, uy;
};
LIFE_DF Moments32 moments32_rn(const float g[kNV], float Fx, float Fy) {
    Moments32 m;
    const float dr = ((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7])) + g[8];
    const float jx = (g[1] - g[2]) + (g[5] - g[6]) + (g[7] - g[8]);
    const float jy = (g[3] - g[4]) + (g[5] - g[6]) + (g[8] - g[7]);
    // 1 / (1 + dr) with the rounding error of the sum put back (moments32)
    const float r = 1.0f + dr;
    const float e = dr - (r - 1.0f);
    const float inv0 = 1.0f / r;
    m.inv = fmaf_(-inv0, e * inv0, inv0);
    m.drho = dr;
    m.nx = fmaf_(0.5f, Fx, jx);
    m.ny = fmaf_(0.5f, Fy, jy);
    m.ux = m.nx * m.inv;
    m.uy = m.ny * m.inv;
    return m;
}

// BGK + Guo (collide_bgk32) of one site, in place.
template <bool SITE, bool FORCE>
LIFE_DF void collide_bgk32_rn(float omega, float g[kNV], const Moments32& m, float Fx, float Fy) {
    const float ux = m.ux, uy = m.uy, dr = m.drho;
    const float usq = fmaf_(ux, ux, uy * uy);  // times 1.5 below
    const float cF = fmaf_(-0.5f, omega, 1.0f);
#pragma unroll
    for (int v = 0; v < kNV; v++) {
        const int cx = kCX[v], cy = kCY[v];
        const float k = v == 0 ? 16.0f : (v < 5 ? 4.0f : 1.0f);
        float cu;
        if (cx == 0 && cy == 0) cu = 0.0f;
        else if (cy == 0) cu = (float)cx * ux;
        else if (cx == 0) cu = (float)cy * uy;
        // c.u on a diagonal, the second product fused where SITE
        else if (v == 5) cu = mad<SITE>(m.ny, m.inv, ux);
        else if (v == 6) cu = mad<SITE>(-m.nx, m.inv, -uy);
        else if (v == 7) cu = mad<SITE>(-m.ny, m.inv, ux);
        else cu = mad<SITE>(m.ny, m.inv, -ux);
        const float cu3 = 3.0f * cu;
        const float q = fmaf_(cu, 4.5f * cu, cu3);
        const float P = mad<SITE>(-1.5f, usq, q);
        const float eq = w36(k * fmaf_(dr, P, dr + P));
        const float go = fmaf_(eq - g[v], omega, g[v]);
        if (!FORCE) {
            g[v] = go;
            continue;
        }
        // (c - u).F + 3 (c.u) (c.F)
        const float dx = fmaf_(-m.nx, m.inv, (float)cx);
        const float dy = mad<SITE>(-m.ny, m.inv, (float)cy);
        const float A = cx == 0 && cy == 0 ? 0.0f : (cy == 0 ? (float)cx * Fx : (cx == 0 ? (float)cy * Fy
                                                                                        : (float)cx * Fx + (float)cy * Fy));
        float B;
        if (SITE) B = fmaf_(Fx, dx, Fy * dy);
        else if (cx != 0 && cy != 0) B = dy * Fy + Fx * dx;
        else B = fmaf_(dy, Fy, Fx * dx);
        const float fv = w36(k * (3.0f * fmaf_(A, cu3, B)));
        g[v] = fmaf_(fv, cF, go);
    }
}

// Central moments (collide_cm32) of one site, in place.
template <bool SITE, bool FORCE>
LIFE_DF void collide_cm32_rn(float omega, float cs2, float g[kNV], const Moments32& m, float Fx, float Fy) {
    const float X = m.ux, Y = m.uy, dr = m.drho;
    const float XX = X * X, YY = Y * Y, XY = X * Y;
    const float XXY = Y * XX, XYY = X * YY;
    // c - u for c = 0, 1, -1
    const float dx0 = -X, dxp = fmaf_(-m.nx, m.inv, 1.0f), dxm = fmaf_(-m.nx, m.inv, -1.0f);
    const float dy0 = -Y, dyp = fmaf_(-m.ny, m.inv, 1.0f), dym = fmaf_(-m.ny, m.inv, -1.0f);
    float k4p = SITE ? fmaf_(X, X, -YY) : fmaf_(-Y, Y, XX);
    float k5p = XY;
    const float dx0q = dx0 * dx0;
#pragma unroll
    for (int v = 0; v < kNV; v++) {
        const float dx = kCX[v] == 0 ? dx0 : (kCX[v] > 0 ? dxp : dxm);
        const float dy = kCY[v] == 0 ? dy0 : (kCY[v] > 0 ? dyp : dym);
        // dx^2 - dy^2: the product of the moving direction is the exact one
        const float d = kCX[v] == 0 ? fmaf_(-dy, dy, dx0q) : fmaf_(dx, dx, -(dy * dy));
        k4p = fmaf_(d, g[v], k4p);
        k5p = fmaf_(dy, dx * g[v], k5p);
    }
    const float k1 = 0.5f * Fx, k2 = 0.5f * Fy;
    const float k4 = (1.0f - omega) * k4p, k5 = (1.0f - omega) * k5p;
    const float k6 = cs2 * k2, k7 = cs2 * k1;
    // 9 c^2 u^2 + 6 c u - 3 u^2 along x and y, c = 0, 1, -1
    const float X6 = 6.0f * X, Y6 = 6.0f * Y, YY9 = 9.0f * YY;
    const float bx0 = -3.0f * XX, bxp = fmaf_(-3.0f, XX, fmaf_(9.0f, XX, X6)), bxm = fmaf_(-3.0f, XX, fmaf_(9.0f, XX, -X6));
    const float by0 = -3.0f * YY;
    const float byp = SITE ? fmaf_(-3.0f, YY, fmaf_(9.0f, YY, Y6)) : fmaf_(6.0f, Y, YY9) - 3.0f * YY;
    const float bym = SITE ? fmaf_(-3.0f, YY, fmaf_(9.0f, YY, -Y6)) : (YY9 - Y6) - 3.0f * YY;
    // columns of M^-1 (De Rosis 2019 basis); products by powers of two are exact
    const float x4 = 0.25f * X, y4 = 0.25f * Y, xx4 = 0.25f * XX, yy4 = 0.25f * YY;
    const float x8 = 0.125f * X, y8 = 0.125f * Y, xx8 = 0.125f * XX, yy8 = 0.125f * YY;
    const float xy2 = 0.5f * XY, xxy2 = 0.5f * XXY, xyy2 = 0.5f * XYY;
    const float hx = 0.5f * X, hy = 0.5f * Y;
    const float uX = mad<SITE>(-X, YY, X);   // X (1 - YY)
    const float uY = mad<SITE>(-Y, XX, Y);   // Y (1 - XX)
    const float xy = XY + XY;
    const float m1[kNV] = {2.0f * XYY - (X + X),
                           0.5f + (uX - 0.5f * YY),
                           -0.5f + (uX + 0.5f * YY),
                           mad<SITE>(-X, Y, -XYY),
                           mad<SITE>(-X, YY, XY),
                           (xyy2 + (xy2 + y4)) + yy4,
                           ((y4 - xy2) + xyy2) - yy4,
                           ((xyy2 - xy2) - y4) + yy4,
                           ((xy2 - y4) + xyy2) - yy4};
    const float m2[kNV] = {2.0f * XXY - (Y + Y),
                           mad<SITE>(-X, Y, -XXY),
                           mad<SITE>(-Y, XX, XY),
                           (uY - 0.5f * XX) + 0.5f,
                           (uY + 0.5f * XX) - 0.5f,
                           (xxy2 + (xy2 + x4)) + xx4,
                           ((x4 - xy2) + xxy2) - xx4,
                           ((xy2 - x4) + xxy2) - xx4,
                           ((xxy2 - xy2) - x4) + xx4};
    const float m4[kNV] = {0.5f * YY - 0.5f * XX,
                           ((x4 + xx4) - yy4) + 0.25f,
                           ((xx4 - x4) - yy4) + 0.25f,
                           ((xx4 - yy4) - y4) - 0.25f,
                           ((xx4 - yy4) + y4) - 0.25f,
                           ((-x8 - xx8) + yy8) + y8,
                           ((x8 - xx8) + yy8) - y8,
                           ((-x8 - xx8) + yy8) - y8,
                           ((x8 - xx8) + yy8) + y8};
    const float m5[kNV] = {4.0f * XY,
                           -xy - Y,
                           Y - xy,
                           -xy - X,
                           X - xy,
                           mad<SITE>(X, Y, hx + hy) + 0.25f,
                           ((XY - hy) - hx) + 0.25f,
                           mad<SITE>(X, Y, hy - hx) - 0.25f,
                           mad<SITE>(X, Y, hx - hy) - 0.25f};
    const float m6[kNV] = {Y + Y, -Y, -Y,
                           mad<SITE>(-m.ny, m.inv, -0.5f), mad<SITE>(-m.ny, m.inv, 0.5f),
                           hy + 0.25f, hy - 0.25f, hy - 0.25f, hy + 0.25f};
    const float m7[kNV] = {X + X,
                           mad<SITE>(-m.nx, m.inv, -0.5f), mad<SITE>(-m.nx, m.inv, 0.5f),
                           -X, -X, hx + 0.25f, hx - 0.25f, hx + 0.25f, hx - 0.25f};
#pragma unroll
    for (int v = 0; v < kNV; v++) {
        const float k = v == 0 ? 16.0f : (v < 5 ? 4.0f : 1.0f);
        const float bx = kCX[v] == 0 ? bx0 : (kCX[v] > 0 ? bxp : bxm);
        const float by = kCY[v] == 0 ? by0 : (kCY[v] > 0 ? byp : bym);
        const float dev = w36(k * fmaf_(by, 0.25f * bx, 0.5f * (by + bx)));  // feqCM(1,u) - w
        float s = fmaf_(dr, dev, w36(dr * k) + dev);
        if (FORCE) {
            s = fmaf_(m1[v], k1, s);
            s = fmaf_(m2[v], k2, s);
        }
        s = fmaf_(m4[v], k4, s);
        s = fmaf_(m5[v], k5, s);
        if (!FORCE) {
            g[v] = s;
            continue;
        }
        // the bulk rounds these products on four of the populations
        s = v == 7 ? mad<SITE>(m6[v], k6, s) : (v == 8 ? mad<SITE>(m6[v], k6, s) : fmaf_(m6[v], k6, s));
        s = v == 4 || v == 6 || v == 7 ? mad<SITE>(m7[v], k7, s) : fmaf_(m7[v], k7, s);
        g[v] = s;
    }
}

// One site, in place: Fxm, Fym the force of the previous step (moments),
// Fx, Fy of this one.
template <bool CM, bool SITE, bool FORCE = true>
LIFE_DF void step_site32(const GridScalars& gs, float g[kNV], float Fxm, float Fym, float Fx, float Fy) {
    const Moments32 m = moments32_rn(g, Fxm, Fym);
    if (CM) collide_cm32_rn<SITE, FORCE>((float)gs.omega, (float)gs.cs2, g, m, Fx, Fy);
    else collide_bgk32_rn<SITE, FORCE>((float)gs.omega, g, m, Fx, Fy);
}

// Support site of the last spread: moments and forcing with force_xy +
// force_ibm (IBMNode.cpp:97-136).
template <bool CM>
LIFE_DF void support_push32_site(const float* __restrict__ src, float* __restrict__ dst, const GridScalars& g,
                                 const double* __restrict__ fibm, long long id) {
    const long long S = g.S;
    float gs[kNV];
#pragma unroll
    for (int v = 0; v < kNV; v++) gs[v] = src[v * S + id];
    // moments as stored at the end of the previous step (its force_xy),
    // forcing of this step
    const float Fxm = (float)(g.Fxm + fibm[id]), Fym = (float)(g.Fym + fibm[S + id]);
    const float Fx = (float)(g.Fx + fibm[id]), Fy = (float)(g.Fy + fibm[S + id]);
    step_site32<CM, true>(g, gs, Fxm, Fym, Fx, Fy);
    push_site32(dst, g, id, gs);
}

}  // namespace life
