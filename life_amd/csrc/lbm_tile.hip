// Tiled lattice step: stream-collide and boundaries of several time steps in
// one launch, for a lattice without immersed bodies, convective outlet or
// pressure corner, or of one step of any lattice.
//
// The plain step is a bulk push kernel and a boundary kernel that wait for
// each other: two launches of 4-5 us on a small lattice, and one trip of the
// whole lattice through memory per step on a large one.  Here a workgroup
// owns a tile plus a rim of `steps` sites around it, keeps the nine
// populations of each site on the CU and runs whole steps on them: collide
// in registers, push through LDS, boundary sites from LDS.  The rim is
// recomputed by every tile that needs it and shrinks by one site per step,
// so after `steps` steps exactly the tile is valid and is stored: one launch
// and one trip through memory for `steps` steps.
//
// Every site update is the plain kernels' arithmetic (collide64,
// step_site32, bc_value), so the values are the same bit for bit.  Bound by
// the arithmetic of tile and rim and by one step's chain (collide, two
// barriers, the boundary sites); the tile sizes and their measured times
// stand at the rule that picks them (tile_shape in runtime.cpp).
#include <hip/hip_runtime.h>

#include "d2q9_f32_rn.h"
// (uncontracted from here on, see d2q9_f64.h)
#include "bc_site.h"
#include "dev_util.h"
#include "launch.h"
#include "lds_limit.h"

namespace life {

namespace {

// Site arithmetic by storage type: moments and collision of one site.
// Fm: force_xy of the previous step (moments), F: of this step, both with
// force_ibm where the lattice has immersed bodies.
// FORCE false: no uniform force.  site: the same with the force of a support
// site, rounded as the support-site kernels round.
template <typename T, bool CM, bool FORCE>
struct TileOps;

template <bool CM, bool FORCE>
struct TileOps<double, CM, FORCE> {
    static __device__ __forceinline__ void step(const GridScalars& g, double f[kNV], double Fxm, double Fym, double Fx,
                                                double Fy) {
        double rho, ux, uy, fo[kNV];
        moments64(f, Fxm, Fym, rho, ux, uy);
        collide64<CM, FORCE>(g, f, rho, ux, uy, Fx, Fy, fo);
#pragma unroll
        for (int v = 0; v < kNV; v++) f[v] = fo[v];
    }
    static __device__ __forceinline__ void site(const GridScalars& g, double f[kNV], double Fxm, double Fym, double Fx,
                                                double Fy) {
        TileOps<double, CM, true>::step(g, f, Fxm, Fym, Fx, Fy);
    }
};

template <bool CM, bool FORCE>
struct TileOps<float, CM, FORCE> {
    static __device__ __forceinline__ void step(const GridScalars& g, float f[kNV], double Fxm, double Fym, double Fx,
                                                double Fy) {
        step_site32<CM, false, FORCE>(g, f, (float)Fxm, (float)Fym, (float)Fx, (float)Fy);
    }
    static __device__ __forceinline__ void site(const GridScalars& g, float f[kNV], double Fxm, double Fym, double Fx,
                                                double Fy) {
        step_site32<CM, true>(g, f, (float)Fxm, (float)Fym, (float)Fx, (float)Fy);
    }
};

// A boundary site of the tile: where it lies in the tile, its type and
// normal (BCSite's, resolved from the walls alone) and what its condition
// reads from memory.
struct TileBC {
    int t;              // tile-local index a * EJ + b
    signed char type, nx, ny, nd;
    double ux, uy;      // inlet velocity without the ramp
    double rho_in;
    // one step per launch only:
    double old[3];      // convective: populations 2, 6, 8 before the step; [0] at a pressure corner: its previous u_y
};

// Site type and normal of (i, j), as site_type and normal_vector of the
// runtime (Grid.cpp:498-545, 931-957).
__device__ __forceinline__ int tile_site_type(const TileArgs& a, int Nx, int Ny, int i, int j) {
    int t = 0;
    if (i == 0) t = a.wall[0];
    else if (i == Nx - 1) t = a.wall[1];
    if (j == 0) t = a.wall[2];
    else if (j == Ny - 1) t = a.wall[3];
    return t;
}

__device__ __forceinline__ bool tile_bc(const TileArgs& a, int Nx, int Ny, int i, int j, TileBC& b) {
    if (i != 0 && i != Nx - 1 && j != 0 && j != Ny - 1) return false;
    const int type = tile_site_type(a, Nx, Ny, i, j);
    if (type == 0) return false;
    int nx = i == 0 ? 1 : (i == Nx - 1 ? -1 : 0), ny = j == 0 ? 1 : (j == Ny - 1 ? -1 : 0);
    int nd = ny != 0 ? 1 : 0;
    if (nx != 0 && ny != 0) {
        if (tile_site_type(a, Nx, Ny, i + nx, j) == 0) {
            nd = 0;
            ny = 0;
        } else if (tile_site_type(a, Nx, Ny, i, j + ny) == 0) {
            nd = 1;
            nx = 0;
        }
    }
    b.type = (signed char)type;
    b.nx = (signed char)nx;
    b.ny = (signed char)ny;
    b.nd = (signed char)nd;
    return true;
}

// Population v as the FP64 value (Pops<T>::get of a register).
__device__ __forceinline__ double to64(double f, int) { return f; }
__device__ __forceinline__ double to64(float f, int v) { return (double)f + w64(v); }

// GridClass::convectiveSpeed's mean (Grid.cpp:477-487) over the outlet
// velocities col[0..Ny) in LDS, by the whole workgroup: serial in row order
// for FP64 populations, else the tree of convective_finish (its threads'
// sums of rows tid, tid + kConvThreads, ..., combined in halves), which
// leaves the sum in red[0].  The caller synchronises before reading it.
template <typename T>
__device__ __forceinline__ void tile_outlet_sum(const double* col, int Ny, double* red) {
    const int t = threadIdx.x, nt = blockDim.x;
    if (sizeof(T) == 8) {
        if (t == 0) red[0] = serial_sum(0.0, col, Ny);
        return;
    }
    for (int q = t; q < kConvThreads; q += nt) {
        double part = 0.0;
        for (int j = q; j < Ny; j += kConvThreads) part += col[j];
        red[q] = part;
    }
    __syncthreads();
    tree_sum(red);
}

// Two intervals of sites have one in common.
__device__ __forceinline__ bool meet(int a0, int a1, int b0, int b1) { return a0 < b1 && b0 < a1; }

// Interpolation, direct forcing and ordered spread (IBMNode.cpp:26-83) of the
// markers whose support blocks reach the tile or its rim, rows [li, hi) and
// columns [lj, hj), from the populations before the step: the sum at the
// lane's site (i, j) and whether it is a support site.  Every tile forms the
// forces that it needs itself, in the order of the markers, so a case of few
// rigid markers has one launch a step.  lds: 24 bytes per lane, free until the
// tile's populations are pushed.  All lanes of the workgroup.  The launch that it
// replaces took 6.1 us of a step and its start: 441 x 83 FP64 14.3 -> 12.2 us a
// step, 1024 x 256 FP32 22.0 -> 18.0; tiles without markers only compare them.
template <typename T>
__device__ __forceinline__ bool tile_forces(const T* __restrict__ src, const GridScalars& g, const TileArgs& a, int li,
                                            int hi, int lj, int hj, bool act, int i, int j, int lanes, double* lds,
                                            double& Bx, double& By) {
    __shared__ unsigned short near[kTileMarkers];
    __shared__ int found[kTileMaxSites / 64];
    const int t = threadIdx.x, nt = blockDim.x, lane = t % 64, wave = t / 64;
    const int Nx = g.Nx, Ny = g.Ny;
    const int4* box = reinterpret_cast<const int4*>(a.supp_box);
    int count = 0;
    for (int m0 = 0; m0 < a.markers; m0 += nt) {
        const int m = m0 + t;
        bool in = false;
        if (m < a.markers) {
            const int4 b = box[m];
            // a periodic lattice's rim lies on the other side
            const bool mi = meet(b.x, b.x + b.z, li, hi) ||
                            (a.per_i && (meet(b.x, b.x + b.z, li + Nx, hi + Nx) || meet(b.x, b.x + b.z, li - Nx, hi - Nx)));
            const bool mj = meet(b.y, b.y + b.w, lj, hj) ||
                            (a.per_j && (meet(b.y, b.y + b.w, lj + Ny, hj + Ny) || meet(b.y, b.y + b.w, lj - Ny, hj - Ny)));
            in = mi && mj;
        }
        const unsigned long long mask = __ballot(in);
        if (lane == 0) found[wave] = __popcll(mask);
        __syncthreads();
        int at = count + __popcll(mask & ((1ull << lane) - 1));
        for (int w = 0; w < nt / 64; w++) {
            if (w < wave) at += found[w];
            count += found[w];
        }
        if (in) near[at] = (unsigned short)m;
        __syncthreads();
    }
    Bx = By = 0.0;
    bool site = false;
    const int group = lanes / kSupp;  // markers at a time, nine lanes each
    double *ta = lds, *tb = lds + lanes, *tc = lds + 2 * lanes;
    for (int c0 = 0; c0 < count; c0 += group) {
        const int q = t / kSupp, s = t - q * kSupp, qn = min(group, count - c0);
        const bool on = q < qn;
        const int m = near[on ? c0 + q : 0], p = m * kSupp + s;
        const int4 b = box[m];
        const bool term = on && s < b.z * b.w;
        const double d = a.supp_delta[p];
        const double e = a.eps[m], ds = a.ds[m], vx = a.vel[2 * m], vy = a.vel[2 * m + 1];
        if (term) interpolate_terms(src, g.S, (long long)a.supp_site[p], a.F[0][0], a.F[0][1], d, ta[t], tb[t], tc[t]);
        __syncthreads();
        double cx = 0.0, cy = 0.0;
        if (on) {
            double iR = 0.0, mx = 0.0, my = 0.0;
            const int first = q * kSupp;
            for (int r = 0; r < b.z * b.w; r++) {
                iR += ta[first + r];
                mx += tb[first + r];
                my += tc[first + r];
            }
            cx = 2.0 * (g.velScale * iR * vx - mx) * e * ds * 1.0 * d;
            cy = 2.0 * (g.velScale * iR * vy - my) * e * ds * 1.0 * d;
        }
        __syncthreads();
        int4* mbox = reinterpret_cast<int4*>(tc);
        if (term) {
            ta[t] = cx;
            tb[t] = cy;
        }
        if (on && s == 0) mbox[q] = b;
        __syncthreads();
        if (act)
            for (int r = 0; r < qn; r++) {
                const int4 n = mbox[r];
                const int di = i - n.x, dj = j - n.y;
                if (di >= 0 && di < n.z && dj >= 0 && dj < n.w) {
                    Bx += ta[r * kSupp + di * n.w + dj];
                    By += tb[r * kSupp + di * n.w + dj];
                    site = true;
                }
            }
        __syncthreads();
    }
    return site;
}

// One tile of CI x CJ sites (at most) and its rim, one site per lane.  FORCE
// false: no uniform force in these steps.  ONE: one step per launch, with
// what depends on the step before: force_ibm at the support sites of the last
// spread (a.fibm; it is zero elsewhere), a convective outlet, a pressure
// corner.  MARK: with the force at the support sites formed here (the sites of
// the outlet column are not among them).
template <typename T, bool CM, bool FORCE, bool ONE, bool MARK>
__global__ __launch_bounds__(kTileMaxSites) void k_tile_step(const T* __restrict__ src, T* __restrict__ dst,
                                                             GridScalars g, TileArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];
    __shared__ int s_nbc;
    const int n = a.steps;
    const int Nx = g.Nx, Ny = g.Ny;
    const long long S = g.S;
    // the tile: rows [i0, i1) and columns [j0, j1), dealt out evenly
    const unsigned tile = xcd_block(blockIdx.x, gridDim.x);
    const int ti = (int)(tile / (unsigned)a.nj), tj = (int)(tile - (unsigned)ti * (unsigned)a.nj);
    const int i0 = ti * a.qi + min(ti, a.ri), i1 = i0 + a.qi + (ti < a.ri ? 1 : 0);
    const int j0 = tj * a.qj + min(tj, a.rj), j1 = j0 + a.qj + (tj < a.rj ? 1 : 0);
    // with its rim; a side of the lattice with boundary conditions ends it
    const int li = a.per_i ? i0 - n : (i0 - n > 0 ? i0 - n : 0), hi = a.per_i ? i1 + n : (i1 + n < Nx ? i1 + n : Nx);
    const int lj = a.per_j ? j0 - n : (j0 - n > 0 ? j0 - n : 0), hj = a.per_j ? j1 + n : (j1 + n < Ny ? j1 + n : Ny);
    const int EJ = a.EJ;  // row stride of the tile, at least hj - lj
    const int PS = a.PS;  // plane stride: EI * EJ and EJ + 1 spare entries at each end
    T* P = reinterpret_cast<T*>(tile_lds) + (EJ + 1);
    TileBC* bcs = reinterpret_cast<TileBC*>(tile_lds + a.bc_off);
    const int t = threadIdx.x;
    const int ra = t / EJ, rb = t - ra * EJ;
    const bool act = li + ra < hi && lj + rb < hj;
    // lattice coordinates, wrapped where the lattice is periodic
    int i = li + ra, j = lj + rb;
    if (a.per_i) i = ((i % Nx) + Nx) % Nx;
    if (a.per_j) j = ((j % Ny) + Ny) % Ny;
    const long long id = act ? (long long)i * Ny + j : 0;
    const int tl = act ? t : 0;
    T f[kNV];
#pragma unroll
    for (int v = 0; v < kNV; v++) f[v] = src[v * S + id];
    double Bx = 0.0, By = 0.0;
    bool site = false;  // a support site of the last spread
    if constexpr (MARK) {
        site = tile_forces(src, g, a, li, hi, lj, hj, act, i, j, min((int)blockDim.x, PS),
                           reinterpret_cast<double*>(tile_lds), Bx, By);
    } else if (ONE && a.fibm) {
        Bx = a.fibm[id];
        By = a.fibm[S + id];
        site = Bx != 0.0 || By != 0.0;
        if (sizeof(T) == 4 && !site) {
            // FP32 rounds a support site its own way also where the force is
            // exactly zero: look it up in the spread's site list
            const int u = a.site_uid[id];
            site = (unsigned)u < (unsigned)*a.uniq_n && a.uniq[u] == id;
        }
    }
    // outlet: every tile on that side forms the mean velocity of the last
    // column itself (launches of their own, with their own waits, cost more)
    const bool outlet = ONE && a.wall[1] == 5 && hi == Nx;
    double* u3 = reinterpret_cast<double*>(tile_lds + a.out_off);  // 3 columns x EJ rows x 2
    double* red = u3 + 6 * EJ;
    double* col = red + (sizeof(T) == 8 ? 1 : kConvThreads);
    if (outlet) {
        for (int q = t; q < Ny; q += (int)blockDim.x) {
            const long long cid = (long long)(Nx - 1) * Ny + q;
            double fc[kNV], r, ux, uy;
            load_site(src, S, cid, fc);
            moments64(fc, a.F[0][0] + (a.fibm ? a.fibm[cid] : 0.0), a.F[0][1] + (a.fibm ? a.fibm[S + cid] : 0.0), r, ux,
                      uy);
            col[q] = ux;
        }
        if (act && i >= Nx - 3) {
            double fc[kNV], r, ux, uy;
#pragma unroll
            for (int v = 0; v < kNV; v++) fc[v] = to64(f[v], v);
            moments64(fc, a.F[0][0] + Bx, a.F[0][1] + By, r, ux, uy);
            u3[((Nx - 1 - i) * EJ + rb) * 2] = ux;
            u3[((Nx - 1 - i) * EJ + rb) * 2 + 1] = uy;
        }
    }
    if (t == 0) s_nbc = 0;
    __syncthreads();
    {
        // The boundary sites are gathered: in place, each wavefront of a
        // tile along a wall would run the boundary arithmetic for its few
        // sites.
        TileBC b;
        if (act && tile_bc(a, Nx, Ny, i, j, b)) {
            b.t = t;
            b.ux = a.u_in[2 * j];
            b.uy = a.u_in[2 * j + 1];
            b.rho_in = a.rho_in[j];
            if (ONE && b.type == 5) {
                b.old[0] = to64(f[2], 2);
                b.old[1] = to64(f[6], 6);
                b.old[2] = to64(f[8], 8);
            } else if (ONE && b.type == 4 && b.nx != 0 && b.ny != 0) {
                double fp[kNV], rn, uxn;
#pragma unroll
                for (int v = 0; v < kNV; v++) fp[v] = to64(f[v], v);
                moments64(fp, a.F[0][0] + Bx, a.F[0][1] + By, rn, uxn, b.old[0]);
            }
            bcs[atomicAdd(&s_nbc, 1)] = b;
        }
    }
    if (outlet) tile_outlet_sum<T>(col, Ny, red);
    __syncthreads();
    // nine lanes per boundary site, seven sites per wavefront (bc_site.h);
    // the launch has wavefronts enough for all of them
    const int nbc = s_nbc;
    const int wave = t / 64, slot = t % 64 / kBCLanes, bv = t % 64 - slot * kBCLanes;
    const int bk = wave * kBCPerWave + slot;
    const bool bcl = slot < kBCPerWave && bk < nbc;
    double* share = reinterpret_cast<double*>(tile_lds + a.share_off) + bk * kNV;
    // site and lane in one word: what the boundary arithmetic derives from it
    // is formed again in each step, since held over the collision it would
    // cost the registers that let two workgroups share a CU
    unsigned bword = 0;
    if (bcl) {
        const TileBC& b = bcs[bk];
        bword = (unsigned)b.t | (unsigned)bv << 12 | (unsigned)b.type << 16 | (unsigned)(b.nx + 1) << 20 |
                (unsigned)(b.ny + 1) << 22 | (unsigned)b.nd << 24;
    }
    for (int s = 0; s < n; s++) {
        const double Fxm = a.F[s][0], Fym = a.F[s][1], Fx = a.F[s + 1][0], Fy = a.F[s + 1][1];
        if (act) {
            if (ONE && site) TileOps<T, CM, FORCE>::site(g, f, Fxm + Bx, Fym + By, Fx + Bx, Fy + By);
            else TileOps<T, CM, FORCE>::step(g, f, Fxm, Fym, Fx + 0.0, Fy + 0.0);
            // push; a value that leaves the tile's last column lands on the
            // next row's first entry, which no other source writes and whose
            // population is either rebuilt by its boundary condition or
            // already past the valid region
#pragma unroll
            for (int v = 0; v < kNV; v++) P[v * PS + t + kCX[v] * EJ + kCY[v]] = f[v];
        }
        __syncthreads();
        if (nbc) {
            asm volatile("" : "+v"(bword));
            const int bt = bword & 0xfff, v = bword >> 12 & 0xf, type = bword >> 16 & 0xf;
            const TileBC& b = bcs[bk];
            if (ONE && bcl && type == 5) {
                if (v == 2 || v == 6 || v == 8) {
                    // delU of GridClass::convectiveSpeed (Grid.cpp:488-494)
                    const double uOut = red[0] / (double)Ny;
                    const double* u = u3 + 2 * (bt % EJ);
                    const double dux = (-uOut / 2.0) * (3.0 * u[0] - 4.0 * u[2 * EJ] + u[4 * EJ]);
                    const double duy = (-uOut / 2.0) * (3.0 * u[1] - 4.0 * u[2 * EJ + 1] + u[4 * EJ + 1]);
                    Pops<T>::put(P, PS, v, bt, bc_convective(v, b.old[v == 2 ? 0 : (v == 6 ? 1 : 2)], dux, duy));
                }
            } else if (bcl) {
                const int nx = (int)(bword >> 20 & 3) - 1, ny = (int)(bword >> 22 & 3) - 1, nd = bword >> 24 & 1;
                const BCLane l = bc_lane(g, v, type, nx, ny, nd);
                double r1 = 0.0, u1 = 0.0, r2 = 0.0, u2 = 0.0;
                if (l.nbr) {
                    // one neighbour at a time, for the registers
#pragma unroll 1
                    for (int q = 1; q <= 2; q++) {
                        double fn[kNV];
                        r1 = r2;
                        u1 = u2;
                        load_site(P, PS, bt + q * (nx * EJ + ny), fn);
                        bc_neighbour(fn, nd, nd != 0 ? Fx : Fy, r2, u2);
                    }
                }
                const BCPops q = bc_read(l, [&](int u, double w) { return Pops<T>::from(P[u * PS + bt], w); });
                Pops<T>::put(P, PS, v, bt, bc_value<CM>(l, g, q, r1, u1, r2, u2, b.ux * a.ramp[s], b.uy * a.ramp[s],
                                                        b.rho_in, ONE ? b.old[0] : 0.0, share));
            }
            __syncthreads();
        }
#pragma unroll
        for (int v = 0; v < kNV; v++) f[v] = P[v * PS + tl];
        if (s + 1 < n) __syncthreads();  // the next push overwrites what others still read
    }
    if (act && li + ra >= i0 && li + ra < i1 && lj + rb >= j0 && lj + rb < j1) {
#pragma unroll
        for (int v = 0; v < kNV; v++) dst[v * S + id] = f[v];
    }
}

template <typename T, bool CM, bool FORCE, bool ONE, bool MARK>
void launch_tile_t(const T* src, T* dst, const GridScalars& g, const TileArgs& a, unsigned threads, size_t lds,
                   hipStream_t s) {
    // tiles of four steps with their rim exceed the default limit in FP64
    static LdsLimit limit;
    limit.allow((const void*)k_tile_step<T, CM, FORCE, ONE, MARK>, lds, 128 * 1024);
    k_tile_step<T, CM, FORCE, ONE, MARK><<<(unsigned)(a.ni * a.nj), threads, lds, s>>>(src, dst, g, a);
}

template <typename T, bool ONE, bool MARK>
void launch_tile_cf(const T* src, T* dst, const GridScalars& g, const TileArgs& a, bool force, unsigned threads,
                    size_t lds, hipStream_t s) {
    if (g.cm) {
        if (force) launch_tile_t<T, true, true, ONE, MARK>(src, dst, g, a, threads, lds, s);
        else launch_tile_t<T, true, false, ONE, MARK>(src, dst, g, a, threads, lds, s);
    } else {
        if (force) launch_tile_t<T, false, true, ONE, MARK>(src, dst, g, a, threads, lds, s);
        else launch_tile_t<T, false, false, ONE, MARK>(src, dst, g, a, threads, lds, s);
    }
}

}  // namespace

template <typename T>
void launch_tile_step(const T* src, T* dst, const GridScalars& g, TileArgs a, const TileShape& shape, hipStream_t s) {
    const int n = a.steps;
    a.ni = (g.Nx + shape.CI - 1) / shape.CI;
    a.nj = (g.Ny + shape.CJ - 1) / shape.CJ;
    a.qi = g.Nx / a.ni;
    a.ri = g.Nx % a.ni;
    a.qj = g.Ny / a.nj;
    a.rj = g.Ny % a.nj;
    const int ci = a.qi + (a.ri ? 1 : 0), cj = a.qj + (a.rj ? 1 : 0);  // largest tile
    const int EI = ci + 2 * n;
    a.EJ = cj + 2 * n;
    a.PS = EI * a.EJ + 2 * (a.EJ + 1);
    const size_t planes = ((size_t)kNV * a.PS * sizeof(T) + 15) / 16 * 16;
    a.bc_off = (unsigned)planes;
    // boundary sites of a tile and its rim: on the sides of the lattice it
    // reaches, both of them where the tile spans the lattice
    const int reach_i = a.per_i ? 0 : (a.ni == 1 || a.qi <= n ? 2 : 1);
    const int reach_j = a.per_j ? 0 : (a.nj == 1 || a.qj <= n ? 2 : 1);
    const int max_bc = reach_i * (a.EJ < g.Ny || a.per_j ? a.EJ : g.Ny) + reach_j * (EI < g.Nx || a.per_i ? EI : g.Nx);
    unsigned threads = (unsigned)((EI * a.EJ + 63) / 64 * 64);
    const unsigned bc_threads = (unsigned)((max_bc + kBCPerWave - 1) / kBCPerWave * 64);
    if (threads < bc_threads) threads = bc_threads;
    a.share_off = (unsigned)(planes + sizeof(TileBC) * (size_t)max_bc);
    a.out_off = a.share_off + (unsigned)(sizeof(double) * (threads / 64 * kBCPerWave * kNV));
    const bool one = a.one != 0;
    const size_t outlet = one && a.wall[1] == 5 ? 6 * (size_t)a.EJ + kConvThreads + (size_t)g.Ny : 0;
    const size_t lds = a.out_off + sizeof(double) * outlet;
    bool force = false;
    for (int k = 0; k <= n; k++) force = force || a.F[k][0] != 0.0 || a.F[k][1] != 0.0;
    if (one && a.markers > 0) launch_tile_cf<T, true, true>(src, dst, g, a, force, threads, lds, s);
    else if (one) launch_tile_cf<T, true, false>(src, dst, g, a, force, threads, lds, s);
    else launch_tile_cf<T, false, false>(src, dst, g, a, force, threads, lds, s);
}

template void launch_tile_step<double>(const double*, double*, const GridScalars&, TileArgs, const TileShape&,
                                       hipStream_t);
template void launch_tile_step<float>(const float*, float*, const GridScalars&, TileArgs, const TileShape&,
                                      hipStream_t);

}  // namespace life
