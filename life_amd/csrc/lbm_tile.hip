// Tiled lattice step: stream-collide, support sites and boundaries of one
// or several time steps in one launch.
//
// The plain step is a bulk push kernel followed by small launches (support
// sites, boundaries) that wait for each other.  On a lattice of up to about
// a million sites those small launches, each a few microseconds of launch
// and dependent memory latency, are most of the step.  Here a workgroup owns
// a tile of the lattice plus a rim of `steps` sites around it, keeps all
// nine populations of those sites on the CU, and runs the whole step on
// them: collide in registers, push through LDS, boundary sites from LDS.
// The rim is recomputed by every tile that needs it and shrinks by one site
// per step, so after `steps` steps exactly the tile is valid and is stored;
// the lattice crosses memory once per launch instead of once per step, and
// boundaries cost no launch of their own.
//
// Every site update is the arithmetic of the plain kernels (collide64 /
// collide32, bc_values), operand for operand, so the values are the same.
#include <hip/hip_runtime.h>

#include "d2q9_f32.h"
// (uncontracted from here on, see d2q9_f64.h)
#include "bc_site.h"
#include "dev_util.h"
#include "launch.h"

namespace life {

namespace {

// Site arithmetic by storage type: moments and collision of one site.
// Fm: force_xy of the previous step (moments), F: of this step, both with
// force_ibm where the lattice has immersed bodies.
template <typename T, bool CM>
struct TileOps;

template <bool CM>
struct TileOps<double, CM> {
    static __device__ __forceinline__ void step(const GridScalars& g, double f[kNV], double Fxm, double Fym, double Fx,
                                                double Fy) {
        double rho, ux, uy, fo[kNV];
        moments64(f, Fxm, Fym, rho, ux, uy);
        collide64<CM>(g, f, rho, ux, uy, Fx, Fy, fo);
#pragma unroll
        for (int v = 0; v < kNV; v++) f[v] = fo[v];
    }
};

template <bool CM>
struct TileOps<float, CM> {
    static __device__ __forceinline__ void step(const GridScalars& g, float f[kNV], double Fxm, double Fym, double Fx,
                                                double Fy) {
        // Scalars opaque to the optimiser: hoisted out of the step loop, they
        // would leave the compiler other multiply-add pairs to fuse than in
        // the plain kernels, and the results would differ in the last bit.
        float om = (float)g.omega, c2 = (float)g.cs2, c4 = (float)g.cs4;
        float xm = (float)Fxm, ym = (float)Fym, x = (float)Fx, y = (float)Fy;
        asm volatile("" : "+v"(om), "+v"(c2), "+v"(c4), "+v"(xm), "+v"(ym), "+v"(x), "+v"(y));
        float drho, ux, uy, fo[kNV];
        moments32(f, xm, ym, drho, ux, uy);
        if (CM) collide_cm32(om, c2, c4, f, drho, ux, uy, x, y, fo);
        else collide_bgk32(om, f, drho, ux, uy, x, y, fo);
#pragma unroll
        for (int v = 0; v < kNV; v++) f[v] = fo[v];
    }
};

// A boundary site of the tile: where it lies in the tile, and its type and
// normal (BCSite's, resolved from the walls alone).
struct TileBC {
    int t;       // tile-local index a * EJ + b
    int i, j;    // lattice coordinates
    signed char type, nx, ny, nd;
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
    b.i = i;
    b.j = j;
    b.type = (signed char)type;
    b.nx = (signed char)nx;
    b.ny = (signed char)ny;
    b.nd = (signed char)nd;
    return true;
}

// Value of population v at tile-local index t, in FP64 (Pops<T>::get on the
// tile's LDS planes).
template <typename T>
__device__ __forceinline__ void lds_site(const T* P, int PS, int t, double f[kNV]) {
#pragma unroll
    for (int v = 0; v < kNV; v++) f[v] = Pops<T>::get(P, PS, v, t);
}

// One tile of CI x CJ sites (at most) and its rim, one site per lane.  SUP:
// the lattice has immersed bodies, so force_ibm is added to every site's
// force (it is zero away from the supports of the last spread, which gives
// the plain kernels' values there); one step per launch then.
template <typename T, bool CM, bool SUP>
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
    const int i0 = (int)((long long)ti * Nx / a.ni), i1 = (int)((long long)(ti + 1) * Nx / a.ni);
    const int j0 = (int)((long long)tj * Ny / a.nj), j1 = (int)((long long)(tj + 1) * Ny / a.nj);
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
    T f[kNV];
#pragma unroll
    for (int v = 0; v < kNV; v++) f[v] = src[v * S + id];
    double Bx = 0.0, By = 0.0;
    if (SUP) {
        Bx = a.fibm[id];
        By = a.fibm[S + id];
    }
    if (t == 0) s_nbc = 0;
    __syncthreads();
    {
        TileBC b;
        if (act && tile_bc(a, Nx, Ny, i, j, b)) {
            b.t = t;
            bcs[atomicAdd(&s_nbc, 1)] = b;
        }
    }
    __syncthreads();
    // The boundary sites are gathered so that the first lanes take one each
    // (their FP64 arithmetic is several times a site's collision: in place,
    // every wavefront of a tile along a wall would pay for it).
    const int nbc = s_nbc;
    TileBC b{};
    double uwx = 0.0, uwy = 0.0, rin = 1.0;
    const bool bcl = t < nbc;
    if (bcl) {
        b = bcs[t];
        uwx = a.u_in[2 * b.j];
        uwy = a.u_in[2 * b.j + 1];
        rin = a.rho_in[b.j];
    }
    double dux = 0.0, duy = 0.0, fo2 = 0.0, fo6 = 0.0, fo8 = 0.0;
    double rn = 0.0, uxn = 0.0, uyn = 0.0;
    if (bcl && b.type == 5) {
        // convective outlet (one step per launch): its old populations and
        // the extrapolated velocity change
        const long long bid = (long long)b.i * Ny + b.j;
        dux = a.delU[2 * b.j];
        duy = a.delU[2 * b.j + 1];
        fo2 = Pops<T>::get(src, S, 2, bid);
        fo6 = Pops<T>::get(src, S, 6, bid);
        fo8 = Pops<T>::get(src, S, 8, bid);
    }
    if (bcl && b.type == 4 && b.nx != 0 && b.ny != 0) {
        // pressure corner (one step per launch): its previous moments
        const long long bid = (long long)b.i * Ny + b.j;
        double fp[kNV];
        load_site(src, S, bid, fp);
        moments64(fp, a.F[0][0] + a.fibm[bid], a.F[0][1] + a.fibm[S + bid], rn, uxn, uyn);
    }
    for (int s = 0; s < n; s++) {
        const double Fxm = a.F[s][0], Fym = a.F[s][1], Fx = a.F[s + 1][0], Fy = a.F[s + 1][1];
        if (act) {
            if (SUP) TileOps<T, CM>::step(g, f, Fxm + Bx, Fym + By, Fx + Bx, Fy + By);
            else TileOps<T, CM>::step(g, f, Fxm, Fym, Fx + 0.0, Fy + 0.0);
            // push; a value that leaves the tile's last column lands on the
            // next row's first entry, which no other source writes and whose
            // population is either rebuilt by its boundary condition or
            // already past the valid region
#pragma unroll
            for (int v = 0; v < kNV; v++) P[v * PS + t + kCX[v] * EJ + kCY[v]] = f[v];
        }
        __syncthreads();
        if (nbc) {
            if (bcl) {
                if (b.type == 5) {
                    Pops<T>::put(P, PS, 2, b.t, fo2 + 3.0 * w64(2) * (dux * kCX[2] + duy * kCY[2]));
                    Pops<T>::put(P, PS, 6, b.t, fo6 + 3.0 * w64(6) * (dux * kCX[6] + duy * kCY[6]));
                    Pops<T>::put(P, PS, 8, b.t, fo8 + 3.0 * w64(8) * (dux * kCX[8] + duy * kCY[8]));
                } else {
                    double fs[kNV], f1[kNV], f2[kNV];
                    const bool nbr = bc_reads_neighbours(b.type, b.nx, b.ny);
#pragma unroll
                    for (int v = 0; v < kNV; v++)
                        fs[v] = bc_unknown(b.nx, b.ny, b.nd, v) ? 0.0 : Pops<T>::get(P, PS, v, b.t);
                    if (nbr) {
                        lds_site(P, PS, b.t + b.nx * EJ + b.ny, f1);
                        lds_site(P, PS, b.t + 2 * (b.nx * EJ + b.ny), f2);
                    }
                    const double F12[2] = {Fx, Fy};
                    bc_values<CM>(g, b.type, b.nx, b.ny, b.nd, fs, f1, f2, uwx * a.ramp[s], uwy * a.ramp[s], rin, rn,
                                  uxn, uyn, F12, F12);
#pragma unroll
                    for (int v = 0; v < kNV; v++) Pops<T>::put(P, PS, v, b.t, fs[v]);
                }
            }
            __syncthreads();
        }
        if (act) {
#pragma unroll
            for (int v = 0; v < kNV; v++) f[v] = P[v * PS + t];
        }
        if (s + 1 < n) __syncthreads();  // the next push overwrites what others still read
    }
    if (act && li + ra >= i0 && li + ra < i1 && lj + rb >= j0 && lj + rb < j1) {
#pragma unroll
        for (int v = 0; v < kNV; v++) dst[v * S + id] = f[v];
    }
}

template <typename T, bool CM, bool SUP>
void launch_tile_t(const T* src, T* dst, const GridScalars& g, const TileArgs& a, unsigned threads, size_t lds,
                   hipStream_t s) {
    k_tile_step<T, CM, SUP><<<(unsigned)(a.ni * a.nj), threads, lds, s>>>(src, dst, g, a);
}

}  // namespace

template <typename T>
void launch_tile_step(const T* src, T* dst, const GridScalars& g, TileArgs a, const TileShape& shape, bool sup,
                      hipStream_t s) {
    const int n = a.steps;
    a.ni = (g.Nx + shape.CI - 1) / shape.CI;
    a.nj = (g.Ny + shape.CJ - 1) / shape.CJ;
    const int ci = (g.Nx + a.ni - 1) / a.ni, cj = (g.Ny + a.nj - 1) / a.nj;  // largest tile
    const int EI = ci + 2 * n;
    a.EJ = cj + 2 * n;
    a.PS = EI * a.EJ + 2 * (a.EJ + 1);
    const size_t planes = ((size_t)kNV * a.PS * sizeof(T) + 15) / 16 * 16;
    a.bc_off = (unsigned)planes;
    // boundary sites of a tile lie on at most two rows and two columns of it
    const size_t lds = planes + sizeof(TileBC) * (size_t)(2 * (EI + a.EJ));
    const unsigned threads = (unsigned)((EI * a.EJ + 63) / 64 * 64);
    if (sup) {
        if (g.cm) launch_tile_t<T, true, true>(src, dst, g, a, threads, lds, s);
        else launch_tile_t<T, false, true>(src, dst, g, a, threads, lds, s);
    } else {
        if (g.cm) launch_tile_t<T, true, false>(src, dst, g, a, threads, lds, s);
        else launch_tile_t<T, false, false>(src, dst, g, a, threads, lds, s);
    }
}

template void launch_tile_step<double>(const double*, double*, const GridScalars&, TileArgs, const TileShape&, bool,
                                       hipStream_t);
template void launch_tile_step<float>(const float*, float*, const GridScalars&, TileArgs, const TileShape&, bool,
                                      hipStream_t);

}  // namespace life
