// Boundary-site arithmetic (GridClass::applyBCs, regularisedBC,
// convectiveBC, Grid.cpp:302-474) shared by the boundary kernels: FP64 with
// the reference's operation order, for both storages.
//
// Nine lanes work on one site, lane v on population v: a site's arithmetic
// is several times a bulk collision's and there are only O(Nx + Ny) sites,
// so with one lane per site the whole time is one long dependent chain on a
// few wavefronts.  Split over the populations, a lane evaluates two
// equilibria instead of eighteen and the chain is about a third as long.
// Sums over the populations are formed by every lane, in v order from zero,
// so each value is the one a single lane would compute.
#pragma once

#include "d2q9_f64.h"

namespace life {

constexpr int kBCLanes = kNV;            // lanes per boundary site
constexpr int kBCPerWave = 64 / kBCLanes;  // sites per wavefront (one lane left over)

// Lattice velocity and opposite of population v, at run time.
LIFE_DI int cx_rt(int v) { return v == 1 || v == 5 || v == 7 ? 1 : (v == 2 || v == 6 || v == 8 ? -1 : 0); }
LIFE_DI int cy_rt(int v) { return v == 3 || v == 5 || v == 8 ? 1 : (v == 4 || v == 6 || v == 7 ? -1 : 0); }
LIFE_DI int opp_rt(int v) { return v == 0 ? 0 : ((v - 1) ^ 1) + 1; }

// feq64 with a run-time lattice velocity.
template <bool CM>
LIFE_DI double feq64_rt(double rho, double ux, double uy, int cx, int cy, double w) {
    if (CM) {
        double ax = 9.0 * (cx * cx) * (ux * ux) + 6.0 * cx * ux - 3.0 * (ux * ux) + 2.0;
        double ay = 9.0 * (cy * cy) * (uy * uy) + 6.0 * cy * uy - 3.0 * (uy * uy) + 2.0;
        return 0.25 * rho * w * ax * ay;
    } else {
        double cu = cx * ux + cy * uy;
        double q = ux * ux * (cx * cx - 1.0 / 3.0) + uy * uy * (cy * cy - 1.0 / 3.0);
        return rho * w * (1.0 + 3.0 * cu + 4.5 * q + 9.0 * cx * cy * ux * uy);
    }
}

// Populations that regularisedBC rebuilds (those that entered from outside
// the domain).
LIFE_DI bool bc_unknown(int nx, int ny, int nd, int cx, int cy) {
    return nx != 0 && ny != 0 ? (cx == nx || cy == ny) : (nd == 0 ? cx == nx : cy == ny);
}

// The site reads its two inward neighbours: the zero gradient of free-slip
// and pressure sites, the density extrapolation of corners.
LIFE_DI bool bc_reads_neighbours(int type, int nx, int ny) {
    return type == 3 || type == 4 || (nx != 0 && ny != 0);
}

// Orders LDS writes of some lanes before later reads by other lanes of the
// same wavefront.
LIFE_DI void bc_lane_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Density and the velocity along the side (momentum + F/2 over density,
// moments64) of a neighbour's populations.
LIFE_DI void bc_neighbour(const double f[kNV], int nd, double F, double& r, double& ut) {
    double s = 0.0, m = 0.0;
#pragma unroll
    for (int v = 0; v < kNV; v++) {
        s += f[v];
        m += (nd != 0 ? kCX[v] : kCY[v]) * f[v];
    }
    r = s;
    ut = (m + 0.5 * F) / s;
}

// applyBCs + regularisedBC of one wall, velocity, free-slip or pressure site:
// the value of population v, on lane v of the site.  fs: the site's
// post-stream populations (unknown ones not used); f1, f2: the inward
// neighbours' (used only where bc_reads_neighbours); uwx, uwy: u_in times
// the ramp; rho_in; rn, uxn, uyn: the site's previous moments (used only at
// a pressure corner: everywhere else all three are overwritten); F1, F2:
// force_xy at the neighbours along the side; share: kNV entries of LDS of
// the site's own.  All lanes of the site call it together.
template <bool CM>
LIFE_DI double bc_value(const GridScalars& g, int v, int type, int nx, int ny, int nd, const double fs[kNV],
                        const double f1[kNV], const double f2[kNV], double uwx, double uwy, double rho_in, double rn,
                        double uxn, double uyn, double F1, double F2, double* share) {
    const bool corner = nx != 0 && ny != 0;
    const bool velocity_like = type == 1 || type == 2 || type == 3;  // wall, velocity, free-slip
    if (type == 1) {
        uxn = 0.0;
        uyn = 0.0;
    } else if (type == 2) {
        uxn = uwx;
        uyn = uwy;
    }
    if (bc_reads_neighbours(type, nx, ny)) {
        double r1, r2, u1, u2;
        bc_neighbour(f1, nd, F1, r1, u1);
        bc_neighbour(f2, nd, F2, r2, u2);
        if (type == 3 || type == 4) {
            if (type == 3) {
                if (nd == 0) uxn = 0.0;
                else uyn = 0.0;
            } else {
                rn = rho_in;
            }
            // Utils::zeroGradient order 2 on the current velocity (Utils.h:200-210)
            const double ut = (4.0 / 3.0) * u1 - (1.0 / 3.0) * u2;
            if (nd != 0) uxn = ut;
            else uyn = ut;
        }
        if (corner && velocity_like) rn = 2.0 * r1 - r2;  // Utils.h:150-162
    }
    if (!corner) {
        const int nn = nd == 0 ? nx : ny;
        double fplus = 0.0, fzero = 0.0;
#pragma unroll
        for (int q = 0; q < kNV; q++) {
            const int cn = nd == 0 ? kCX[q] : kCY[q];
            fplus = cn == -nn ? fplus + fs[q] : fplus;
            fzero = cn == 0 ? fzero + fs[q] : fzero;
        }
        const double s = 2.0 * fplus + fzero;
        if (velocity_like) {
            rn = s / (1.0 - nn * (nd == 0 ? uxn : uyn));
        } else if (type == 4) {
            const double un = nn * (1.0 - s / rn);
            if (nd == 0) uxn = un;
            else uyn = un;
        }
    }
    const int cx = cx_rt(v), cy = cy_rt(v);
    const double w = w64(v);
    double f = 0.0, fopp = 0.0;
    const int vo = opp_rt(v);
#pragma unroll
    for (int q = 0; q < kNV; q++) {
        f = q == v ? fs[q] : f;
        fopp = q == vo ? fs[q] : fopp;
    }
    const double feq = feq64_rt<CM>(rn, uxn, uyn, cx, cy, w);
    const double feqo = feq64_rt<CM>(rn, uxn, uyn, -cx, -cy, w);
    if (bc_unknown(nx, ny, nd, cx, cy)) f = corner && nx * cx + ny * cy == 0 ? feq : feq + (fopp - feqo);
    share[v] = f - feq;
    bc_lane_fence();
    double Sxx = 0.0, Syy = 0.0, Sxy = 0.0;
#pragma unroll
    for (int q = 0; q < kNV; q++) {
        const double fneq = share[q];
        Sxx += kCX[q] * kCX[q] * fneq;
        Syy += kCY[q] * kCY[q] * fneq;
        Sxy += kCX[q] * kCY[q] * fneq;
    }
    bc_lane_fence();  // share may be rewritten after the call
    return feq + (w / (2.0 * g.cs4)) * (((cx * cx - g.cs2) * Sxx) + ((cy * cy - g.cs2) * Syy) + (2.0 * cx * cy * Sxy));
}

// convectiveBC (Grid.cpp:468-474): the value of population v = 2, 6 or 8 at
// an outlet site from its value fn before the step.
LIFE_DI double bc_convective(int v, double fn, double dux, double duy) {
    return fn + 3.0 * w64(v) * (dux * cx_rt(v) + duy * cy_rt(v));
}

}  // namespace life
