// Immersed-boundary kernels: support search, marker spacing, epsilon
// matrix, interpolation + direct forcing, and the ordered spread.
//
// All arithmetic is FP64 with the reference's operation order
// (IBMNode.cpp, Objects.cpp:235-321), for both population storages.
// Compiled with -ffp-contract=off.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdlib>

#include "d2q9_f64.h"
#include "launch.h"
#include "lds_limit.h"

namespace life {

// The single-case coupling kernels run beside the next step's bulk
// stream-collide (launched early on another stream): their waves take the
// highest issue priority on a SIMD they share with stream-collide waves,
// since they are usually the critical path of the step.  The level (0..3)
// is set per device by set_coupling_priority (LIFE_COUPLING_PRIO, default 3).
__device__ int g_coupling_prio = 3;
__device__ __forceinline__ void coupling_priority() {
    const int p = g_coupling_prio;
    if (p >= 3) __builtin_amdgcn_s_setprio(3);
    else if (p == 2) __builtin_amdgcn_s_setprio(2);
    else if (p == 1) __builtin_amdgcn_s_setprio(1);
}

hipError_t set_coupling_priority(int level) {
    return hipMemcpyToSymbol(HIP_SYMBOL(g_coupling_prio), &level, sizeof(int));
}

// Orders LDS writes of some lanes before later reads by other lanes of the
// same wavefront (LDS operations of a wavefront complete in order; the
// fence stops the compiler from reordering them across lanes).
__device__ __forceinline__ void lane_exchange_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Supports and spacing take half a wavefront (kHalf lanes) per marker: one lane
// per site of the 5x5 block, and every 32nd marker of the body per lane.  With
// one lane per marker the 25 sites and the body's markers came one after the
// other in each lane, and one workgroup per body left all but a few CUs idle:
// 27 us for two bodies of 530 markers and 10 us for one filament, 5.5 us for both now.
constexpr int kHalf = 32;

// IBMNodeClass::findSupport (IBMNode.cpp:139-179): lattice sites within 1.5
// spacings of the marker in both directions, scanned i-major over the 5x5
// block around the nearest site, kept in scan order (at most 9).  l: lane of
// the half wavefront.
__device__ __forceinline__ void find_support_half(const MarkerDev& m, const GridScalars& g, int k, double x, double y,
                                                  int l) {
    const double Dx = g.Dx;
    const int inear = (int)round(x / Dx), jnear = (int)round(y / Dx);
    const int i = inear - 2 + l / 5, j = jnear - 2 + l % 5;
    const double dx = fabs(x / Dx - i), dy = fabs(y / Dx - j);
    const bool in = l < 25 && dx < 1.5 && dy < 1.5 && i >= 0 && i <= g.Nx - 1 && j >= 0 && j <= g.Ny - 1;
    const unsigned mask = (unsigned)(__ballot(in) >> (threadIdx.x & 32));  // this half's lanes
    const int at = __popc(mask & ((1u << l) - 1)), found = __popc(mask), n = min(found, kSupp);
    if (in && at < kSupp) {
        m.supp_site[k * kSupp + at] = i * g.Ny + j;
        m.supp_ij[(k * kSupp + at) * 2] = i;
        m.supp_ij[(k * kSupp + at) * 2 + 1] = j;
        m.supp_delta[k * kSupp + at] = dirac64(dx) * dirac64(dy);
    }
    if (l >= n && l < kSupp) {
        m.supp_site[k * kSupp + l] = -1;
        m.supp_ij[(k * kSupp + l) * 2] = 0;
        m.supp_ij[(k * kSupp + l) * 2 + 1] = 0;
        m.supp_delta[k * kSupp + l] = 0.0;
    }
    if (l == 0) {
        if (found > kSupp) *m.overflow = 1;
        const int first = n > 0 ? __ffs(mask) - 1 : 0, rows = __popc(mask & (31u << (first / 5 * 5)));
        m.supp_cnt[k] = n;
        int* box = m.supp_box + 4 * k;
        box[0] = n > 0 ? inear - 2 + first / 5 : 0;
        box[1] = n > 0 ? jnear - 2 + first % 5 : 0;
        box[2] = n > 0 ? n / rows : 0;
        box[3] = rows;
    }
}

// IBMNodeClass::computeDs (IBMNode.cpp:182-204): distance (lattice units) of
// marker q0 of a body, at (x, y), to the nearest of the body's other markers
// (positions P, cnt of them), starting from 10.  sqrt(.)/Dx is monotone, so
// the minimum of sqrt(d.d)/Dx over the other markers is sqrt(min d.d)/Dx; the
// minimum does not depend on the order of the comparisons.  The result is in
// every lane of the half wavefront.
__device__ __forceinline__ double spacing_half(const double* P, int cnt, int q0, double x, double y, double Dx, int l) {
    const double2* P2 = reinterpret_cast<const double2*>(P);
    constexpr int U = 4;  // positions loaded before the first is used
    double mn = INFINITY;
    for (int b = 0; b < cnt; b += U * kHalf) {
        double2 pq[U];
#pragma unroll
        for (int u = 0; u < U; u++) pq[u] = P2[min(b + u * kHalf + l, cnt - 1)];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int q = b + u * kHalf + l;
            const double dx = x - pq[u].x, dy = y - pq[u].y;
            const double d2 = 0.0 + dx * dx + dy * dy;
            if (q < cnt && q != q0 && d2 < mn) mn = d2;
        }
    }
#pragma unroll
    for (int o = kHalf / 2; o > 0; o /= 2) {
        const double other = __shfl_xor(mn, o, kHalf);
        if (other < mn) mn = other;
    }
    const double mag = sqrt(mn) / Dx;
    return mag < 10.0 ? mag : 10.0;
}

// Both for the markers of this workgroup: the two are independent (the
// spacing reads only positions), so the coupling chain has one kernel fewer
// to wait for.
constexpr int kSupportThreads = 256;

__device__ __forceinline__ void support_ds_body(const MarkerDev& m, const GridScalars& g, int flexible_only) {
    const int k = (int)(blockIdx.x * (kSupportThreads / kHalf) + threadIdx.x / kHalf), l = (int)threadIdx.x % kHalf;
    if (k >= m.n) return;
    const int b = m.body[k];
    const double x = m.pos[2 * k], y = m.pos[2 * k + 1];
    const int first = m.body_first[b], cnt = m.body_n[b];
    if (flexible_only && m.body_flex[b] != 0) return;
    find_support_half(m, g, k, x, y, l);
    const double ds = spacing_half(m.pos + 2 * first, cnt, k - first, x, y, g.Dx, l);
    if (l == 0) m.ds[k] = ds;
}

__global__ __launch_bounds__(kSupportThreads) void k_support_ds(MarkerDev m, GridScalars g, int flexible_only) {
    coupling_priority();
    support_ds_body(m, g, flexible_only);
}

__global__ __launch_bounds__(kSupportThreads) void k_support_ds_batch(const CaseDev* __restrict__ cases,
                                                                      const int* __restrict__ list,
                                                                      int flexible_only) {
    const CaseDev& c = cases[list[blockIdx.y]];
    support_ds_body(c.m, c.g, flexible_only);
}

// A_ij of ObjectsClass::computeEpsilon (Objects.cpp:271-300) for the system
// of markers [first, first+n): sum over the supports s of marker i of
// delta_i(s) * delta(x_j - s), times ds_j.
// The sum over the supports of marker mi of delta_s * d(xj - i_s) d(yj - j_s)
// in support order (an epsilon matrix entry before the spacing factor,
// Objects.cpp:271-300).  find_support keeps the sites with |x - i| < 1.5 and
// |y - j| < 1.5 inside the lattice, scanned i-major in ascending order: a
// block of at most three consecutive columns by three consecutive rows, the
// first support being the lowest of each.  So the kernel values of the x
// and y distances are evaluated once per column and per row (six
// evaluations instead of eighteen) and picked per support: the same values,
// products and sum as evaluating them support by support.
__device__ __forceinline__ double support_sum(const MarkerDev& m, int mi, double xj, double yj) {
    const int cnt = m.supp_cnt[mi];
    int sij[2 * kSupp];
    double sd[kSupp];
#pragma unroll
    for (int s = 0; s < 2 * kSupp; s++) sij[s] = m.supp_ij[mi * kSupp * 2 + s];
#pragma unroll
    for (int s = 0; s < kSupp; s++) sd[s] = m.supp_delta[mi * kSupp + s];
    const int i0 = sij[0], j0 = sij[1];
    const double x0 = dirac64(fabs(xj - i0)), x1 = dirac64(fabs(xj - (i0 + 1))), x2 = dirac64(fabs(xj - (i0 + 2)));
    const double y0 = dirac64(fabs(yj - j0)), y1 = dirac64(fabs(yj - (j0 + 1))), y2 = dirac64(fabs(yj - (j0 + 2)));
    double a = 0.0;
#pragma unroll
    for (int s = 0; s < kSupp; s++) {
        if (s < cnt) {
            const int kx = sij[2 * s] - i0, ky = sij[2 * s + 1] - j0;
            const double dx = kx == 0 ? x0 : (kx == 1 ? x1 : x2);
            const double dy = ky == 0 ? y0 : (ky == 1 ? y1 : y2);
            a += sd[s] * (dx * dy);
        }
    }
    return a;
}

__global__ void k_epsilon_matrix(MarkerDev m, GridScalars g, int first, int n, double* __restrict__ A) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * n) return;
    const int r = (int)(t / n), c = (int)(t - (long long)r * n);
    const int mi = first + r, mj = first + c;
    const double Dx = g.Dx;
    const double xj = m.pos[2 * mj] / Dx, yj = m.pos[2 * mj + 1] / Dx;
    A[t] = support_sum(m, mi, xj, yj) * m.ds[mj];
}

// Entry (mi, mj) from the positions of the two markers and the column's
// spacing.  Markers three spacings apart in x or y have no site in common:
// their entry is zero.  The supports are those of the positions (every caller
// forms the system before the markers move on).
__device__ __forceinline__ double eps_entry(const MarkerDev& m, double Dx, int mi, double xi, double yi, double xj,
                                            double yj, double dsj) {
    const double lim = 3.01 * Dx;
    if (fabs(xi - xj) >= lim || fabs(yi - yj) >= lim) return 0.0;  // (a position of NaN shows in the entry)
    return support_sum(m, mi, xj / Dx, yj / Dx) * dsj;
}

// The matrix row by row, non-zeros only: a marker couples to the few others
// within three spacings (a support of marker i lies within 1.5 of x_i and
// reaches 1.5), so of n^2 entries about ten a row are computed and brought to
// the host.  One wavefront per row: 64 columns a round, the entries that are
// near evaluated, the non-zero ones packed by a ballot.  530 markers: 16 us
// for the whole matrix and 45 us for its copy before, 10 us and 3 us now.
__global__ __launch_bounds__(256) void k_epsilon_rows(MarkerDev m, GridScalars g, int first, int n,
                                                      int* __restrict__ count, int* __restrict__ col,
                                                      double* __restrict__ val) {
    const int r = blockIdx.x * 4 + (int)threadIdx.x / 64, lane = threadIdx.x % 64;
    if (r >= n) return;
    const double Dx = g.Dx;
    const int mi = first + r;
    const double xi = m.pos[2 * mi], yi = m.pos[2 * mi + 1];
    int have = 0;
    for (int c0 = 0; c0 < n; c0 += 64) {
        const int c = c0 + lane, mj = first + (c < n ? c : 0);
        const double xj = m.pos[2 * mj], yj = m.pos[2 * mj + 1];
        double a = 0.0;
        if (c < n) a = eps_entry(m, Dx, mi, xi, yi, xj, yj, m.ds[mj]);
        const unsigned long long mask = __ballot(a != 0.0);
        const int at = have + __popcll(mask & ((1ull << lane) - 1));
        if (a != 0.0 && at < kEpsRowCap) {
            col[r * kEpsRowCap + at] = c;
            val[r * kEpsRowCap + at] = a;
        }
        have += __popcll(mask);
    }
    if (lane == 0) count[r] = have;
}

// ---------------------------------------------------------------- epsilon, banded
// Batched form of computeEpsilon for systems whose matrix is banded (every
// filament: A_ij = 0 unless markers i and j are within 3 lattice spacings).
// Band storage: row r holds columns r-KB .. r+2KB (width 3KB+1, the upper
// part leaves room for the fill-in of partial pivoting).  A system with a
// coupling pair outside the band is flagged and solved on the host with the
// dense path instead.

// One thread per band entry, diagonal by diagonal: of the 3KB + 1 a row is
// stored with, the few near the main one are formed, the other diagonals'
// wavefronts only write zeros (row by row: 5.2 us for a filament of 91 markers,
// 35 for the canopy's 64 on two XCDs, 4.3 and 26 now).  grid.y = system.
__device__ inline void eps_band_entry(const MarkerDev& m, const GridScalars& g, int first, int n, int KB,
                                      double* __restrict__ band, long long t) {
    const int W = 3 * KB + 1;
    if (t >= (long long)n * W) return;
    const int q = (int)(t / n), r = (int)(t - (long long)q * n);
    const int c = r - KB + q;
    double a = 0.0;
    if (q <= 2 * KB && c >= 0 && c < n) {
        const int mi = first + r, mj = first + c;
        a = eps_entry(m, g.Dx, mi, m.pos[2 * mi], m.pos[2 * mi + 1], m.pos[2 * mj], m.pos[2 * mj + 1], m.ds[mj]);
    }
    band[(size_t)r * W + q] = a;
}

// The out-of-band check of one system: pairs r < c - KB that could couple
// (support of i within 1.5 of x_i, delta of j within 1.5 of the support: |x_i -
// x_j| < 3 spacings; the test is symmetric).  One workgroup, which writes the
// system's flag (1: a pair outside the band couples, 0: none), also to out if
// that is given (page-locked host memory).  Positions are staged in LDS (P: 2n doubles, or null to
// read them from device memory).  Eight lanes share a row r and take every
// eighth column beyond the band, four columns at a time; rows are dealt out
// in steps of blockDim / 8, so every lane sees about the same number of
// pairs.
__device__ inline void eps_far_rows(const MarkerDev& m, const GridScalars& g, int first, int n, int KB,
                                    int* __restrict__ outside, int* __restrict__ out, double* __restrict__ P) {
    __shared__ int far_sh;
    const double* X = m.pos + 2 * first;
    if (threadIdx.x == 0) far_sh = 0;
    if (P)
        for (int k = threadIdx.x; k < 2 * n; k += blockDim.x) P[k] = X[k];
    __syncthreads();
    if (P) X = P;
    const double lim = 3.01 * g.Dx;
    constexpr int CL = 8, U = 4;
    const int rl = threadIdx.x / CL, cl = threadIdx.x % CL, nrl = blockDim.x / CL;
    int far = 0;
    for (int r = rl; r < n; r += nrl) {
        const double xr = X[2 * r], yr = X[2 * r + 1];
        for (int c0 = r + KB + 1 + cl; c0 < n; c0 += U * CL) {
            double xs[U], ys[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = min(c0 + u * CL, n - 1);
                xs[u] = X[2 * c];
                ys[u] = X[2 * c + 1];
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (c0 + u * CL < n && fabs(xr - xs[u]) < lim && fabs(yr - ys[u]) < lim) far = 1;
        }
    }
    if (far) atomicOr(&far_sh, 1);
    __syncthreads();
    if (threadIdx.x == 0) {
        *outside = far_sh;
        if (out) *out = far_sh;
    }
}

// Launches whose systems have up to this many markers stage the positions
// for the out-of-band check in LDS.
constexpr int kFarLdsMarkers = 1024;

// Band entries (the first be workgroups of grid.x) and the out-of-band
// check (the last workgroup, which also writes the flag) of each system in
// one launch: the two are independent and the solve needs both, so the
// coupling chain waits for one kernel.
__global__ void k_eps_band_prep(MarkerDev m, GridScalars g, const int* __restrict__ sys_first,
                                const int* __restrict__ sys_n, int KB, double* __restrict__ band,
                                const long long* __restrict__ band_off, int* __restrict__ outside, int be,
                                int stage_far) {
    extern __shared__ double P[];
    coupling_priority();
    const int sys = blockIdx.y;
    const int bx = (int)blockIdx.x;
    if (bx < be)
        eps_band_entry(m, g, sys_first[sys], sys_n[sys], KB, band + band_off[sys],
                       (long long)bx * blockDim.x + threadIdx.x);
    else
        eps_far_rows(m, g, sys_first[sys], sys_n[sys], KB, outside + sys, nullptr, stage_far ? P : nullptr);
}

// Batched: grid.y = entry of the system table, whose flag goes to out as well.
// With k_support_ds_batch and the solve 31 us for 12 served filaments, 62 for
// one workgroup per body that did everything (and the flags' gathering).
__global__ void k_eps_band_prep_batch(const CaseDev* __restrict__ cases, const CaseSys* __restrict__ sys, int KB, int be,
                                      int stage_far, int* __restrict__ out) {
    extern __shared__ double P[];
    const CaseSys q = sys[blockIdx.y];
    const CaseDev& c = cases[q.c];
    const int bx = (int)blockIdx.x, first = c.eps.first[q.k], n = c.eps.n[q.k];
    if (bx < be)
        eps_band_entry(c.m, c.g, first, n, KB, c.eps.band + c.eps.off[q.k], (long long)bx * blockDim.x + threadIdx.x);
    else
        eps_far_rows(c.m, c.g, first, n, KB, c.eps.outside + q.k, out ? out + blockIdx.y : nullptr,
                     stage_far ? P : nullptr);
}

// Canonical elimination (partial pivoting, first maximum) of one banded
// system per wavefront, right-hand side of ones, writing epsilon.
//
// With lower and upper bandwidth KB, every non-zero that step k of the
// dense elimination reads or writes lies in rows k..k+KB and columns
// k..k+2KB (row swaps widen the upper band by KB).  Row r lives in the
// registers of lane r % 64, column c of it in register c % C, C = 2KB + 1: rows
// and columns stay where they are for the whole elimination, the steps are
// unrolled C times so that every register index is a constant, and the lanes
// of rows k+1..k+KB are selected by an execution mask that moves up by one a
// step.  Step k:
//  - the pivot's lane is read by every lane (v_readlane); if no entry of
//    column k in the window reaches its magnitude, it is the pivot;
//  - otherwise the first row of maximum magnitude is found, and the two lanes'
//    registers change places;
//  - every lane divides (l = a(i, k) / a(k, k)) and the window's lanes take
//    l times row k from their own row: columns k+1..k+KB, and those up to
//    k+d+KB that a row come up by d has brought in.
// Rows of U stay in place; half the lanes at a time store theirs and take the
// rows 64 further on.  The skipped dense operations all involve an exact
// zero, so the values equal the dense elimination's.
//
// A single wavefront is bound by the chain of dependent FP64 operations here
// (readlane, compare, a division of ten operations, product, difference), about
// 330 cycles a step at KB = 3; the back substitution, with the diagonal's
// reciprocals formed beforehand, 175.  Columns in lanes and rows in registers,
// shifted every step, took 950 for both.  A moved row costs its exchange and the
// columns that it brings in.  Markers one spacing apart, or up to half a per cent
// less, move none; 2 % less, nearly every second row.  97 rows, before | now: none
// moved, KB = 3, 45.8 | 28.9 us; 14 % 46.2 | 34.0; 58 % 48.5 | 46.4; KB = 4, 71 %
// 55.3 | 54.9; 76 % 78.3 | 76.4.  (With the exchange by readlane, all
// KB further columns for KB steps and divisions in the back substitution 28.1,
// 42.0, 61.0, 78.2, 131.)  91 markers, KB = 3: 39 us before, 25 us with the staging
// by four wavefronts.

// Lane `lane`'s value as a wavefront-uniform (SGPR) value.
__device__ inline double uniform64(double v, int lane) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// This lane's bit of a wavefront-uniform mask.
__device__ __forceinline__ bool lane_in(unsigned long long mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// The band is stored with half-bandwidth KBS (W = 3KBS + 1 per row); the
// elimination window has half-bandwidth KB <= KBS, which must bound every
// non-zero of the matrix (|column - row| <= KB).
template <int KB, int KBS>
struct BandRows {
    static constexpr int C = 2 * KB + 1, W = 3 * KBS + 1;
    double w[C], wr;       // this lane's row and its right-hand side
    int moved = 0;         // most rows a pivot has come up by

    // Row r of the band (zero past n): register j takes column
    // (r - KB) + (j - (r - KB)) mod C.
    __device__ __forceinline__ void load(int r, int n, const double* __restrict__ B) {
        const bool in = r < n;
        const double* src = B + (size_t)(in ? r : 0) * W + (KBS - KB);
        int q = (KB - r) % C;
        if (q < 0) q += C;
#pragma unroll
        for (int j = 0; j < C; j++) {
            const double v = src[q];
            w[j] = in ? v : 0.0;
            q = q + 1 == C ? 0 : q + 1;
        }
        wr = in ? 1.0 : 0.0;
    }

    // Row r of U (columns r .. r + 2KB) in place of row r of the band.
    __device__ __forceinline__ void store(int r, int n, double* __restrict__ B, double* __restrict__ y) const {
        if (r >= n) return;
        double* dst = B + (size_t)r * W + KBS;
        int q = (-r) % C;
        if (q < 0) q += C;
#pragma unroll
        for (int j = 0; j < C; j++) {
            dst[q] = w[j];
            q = q + 1 == C ? 0 : q + 1;
        }
        y[r] = wr;
    }

    // The rows of lanes a and b change places, each value by one exchange over
    // the LDS crossbar (all of them in flight together).
    __device__ __forceinline__ void swap_lanes(int L, int a, int b) {
        const int from = L == a ? b : (L == b ? a : L);
#pragma unroll
        for (int j = 0; j < C; j++) w[j] = __shfl(w[j], from);
        wr = __shfl(wr, from);
    }

    // Step k, column k in register J; window: the lanes of rows k+1..k+KB;
    // reach: a pivot row, widened by swaps, has no entry past this column or
    // column k+KB.
    template <int J>
    __device__ __forceinline__ void step(int k, unsigned long long window, int& reach, int L) {
        const int a = k & 63;
        const double p0 = uniform64(w[J], a);
        double piv = p0;
        const unsigned long long reached = __ballot(fabs(w[J]) >= fabs(p0)) & window;
        if (__builtin_expect(reached != 0, 0)) {
            const unsigned long long above = __ballot(fabs(w[J]) > fabs(p0)) & window;
            // the first largest, among the rows above the diagonal's magnitude,
            // in row order (bit d of m: row k + d)
            unsigned long long m = (above >> a) | (above << ((64 - a) & 63));
            double best = fabs(p0);
            int b = a;
            for (; m; m &= m - 1) {
                const int lane = (a + __builtin_ctzll(m)) & 63;
                const double v = uniform64(w[J], lane);
                if (fabs(v) > best) {
                    best = fabs(v);
                    piv = v;
                    b = lane;
                }
            }
            if (b != a) {
                swap_lanes(L, a, b);
                // row k + d has entries up to column k + d + KB
                const int up = (b - a) & 63;
                reach = max(reach, k + up + KB);
                moved = max(moved, up);
            }
            if (piv == 0.0) piv = 1.0;  // zero column: all multipliers 0
        }
        double p[KB + 1];
#pragma unroll
        for (int d = 1; d <= KB; d++) p[d] = uniform64(w[(J + d) % C], a);
        const double pr = uniform64(wr, a);
        const double l = w[J] / piv;
        if (lane_in(window)) {
            w[J] = 0.0;  // column k + C from here on
#pragma unroll
            for (int d = 1; d <= KB; d++) w[(J + d) % C] = w[(J + d) % C] - l * p[d];
            wr = wr - l * pr;
        }
        if (__builtin_expect(reach > k + KB, 0)) {
#pragma unroll
            for (int d = KB + 1; d <= 2 * KB; d++)
                if (d <= reach - k) {
                    const double q = uniform64(w[(J + d) % C], a);
                    if (lane_in(window)) w[(J + d) % C] = w[(J + d) % C] - l * q;
                }
        }
    }

    // Steps k .. k+C-1 (FULL) or those of them below kend.
    template <bool FULL, int J = 0>
    __device__ __forceinline__ void steps(int k, int kend, unsigned long long& window, int& reach, int L) {
        if constexpr (J < C) {
            if (FULL || k < kend) {
                step<J>(k, window, reach, L);
                window = (window << 1) | (window >> 63);
                steps<FULL, J + 1>(k + 1, kend, window, reach, L);
            }
        }
    }
};

// One wavefront; returns the most rows a pivot has come up by, which widen U.
template <int KB, int KBS>
__device__ __forceinline__ int band_eliminate(int n, double* __restrict__ B, double* __restrict__ y) {
    constexpr int C = 2 * KB + 1;
    const int L = threadIdx.x;
    BandRows<KB, KBS> s;
    s.load(L, n, B);
    unsigned long long window = ((1ull << KB) - 1) << 1;
    int reach = 0, saved = 0;
    for (int k = 0; k < n; k += C) {
        // the half wavefront whose rows are done: a block of C steps and its
        // window stay within the 64 rows from `saved`
        if (k >= saved + 32) {
            if (L / 32 == (saved / 32) % 2) {
                const int r = saved + L % 32;
                s.store(r, n, B, y);
                s.load(r + 64, n, B);
            }
            saved += 32;
        }
        if (k + C <= n) s.template steps<true>(k, n, window, reach, L);
        else s.template steps<false>(k, n, window, reach, L);
    }
    for (int end = saved + 64; saved < end; saved += 32)
        if (L / 32 == (saved / 32) % 2) s.store(saved + L % 32, n, B, y);
    return s.moved;
}

// Between the solve's phases: writes of some lanes, reads by others of the
// same wavefront, in LDS or in device memory.
template <bool LDS_>
__device__ __forceinline__ void band_fence() {
    if (LDS_) lane_exchange_fence();
    else __threadfence_block();
}

__device__ __forceinline__ bool mid_range(double v) {
    const double a = fabs(v);
    return a > 0x1p-300 && a < 0x1p300;
}

// a / b from y, the correctly rounded 1 / b (Markstein, IBM J. Res. Dev. 34,
// 1990): the first correction leaves a quotient within one unit in the last
// place, the second rounds it correctly.  For values clear of overflow and
// underflow (mid_range).
__device__ __forceinline__ double div_by(double a, double b, double y) {
    double q = a * y;
    q = __builtin_fma(__builtin_fma(-b, q, a), y, q);
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

// Back substitution by one wavefront (every lane the same), in increasing
// column order: rows of U of half-bandwidth T, KB where no swap has widened
// them.  Terms past n are 0 * 0, which leaves a sum unchanged.  The
// reciprocals and the results go into the two sub-diagonal entries that the
// elimination left unused.  False, with nothing of use written, if a diagonal
// entry or a result is not mid_range (a singular matrix among them).
template <int T, int KBS, bool LDS_>
__device__ __forceinline__ bool band_back_fast(int first, int n, double* __restrict__ B, const double* __restrict__ y,
                                               double* __restrict__ eps) {
    constexpr int W = 3 * KBS + 1;
    bool ok = true;
    for (int r = threadIdx.x; r < n; r += 64) {
        const double d = B[(size_t)r * W + KBS];
        ok = ok && mid_range(d);
        B[(size_t)r * W + KBS - 1] = 1.0 / d;
    }
    if (__ballot(!ok)) return false;
    band_fence<LDS_>();
    struct Row {
        double u[T + 1], r, s;
    };
    auto load = [&](Row& v, int i) {
        const double* U = B + (size_t)max(i, 0) * W + KBS;
#pragma unroll
        for (int q = 0; q <= T; q++) v.u[q] = U[q];
        v.r = U[-1];
        v.s = y[max(i, 0)];
    };
    double x[T];  // x[q] = solution at i + 1 + q
#pragma unroll
    for (int q = 0; q < T; q++) x[q] = 0.0;
    auto solve = [&](const Row& v, int i) {
        double t = v.s;
#pragma unroll
        for (int q = 0; q < T; q++) t = t - v.u[1 + q] * x[q];
        const double xi = div_by(t, v.u[0], v.r);
        if (i >= 0) B[(size_t)i * W + KBS - 2] = xi;
#pragma unroll
        for (int q = T - 1; q > 0; q--) x[q] = x[q - 1];
        x[0] = xi;
    };
    // rows loaded two ahead
    Row a, b, c;
    load(a, n - 1);
    load(b, n - 2);
    for (int i = n - 1; i >= 0; i -= 3) {
        load(c, i - 2);
        solve(a, i);
        load(a, i - 3);
        solve(b, i - 1);
        load(b, i - 4);
        solve(c, i - 2);
    }
    band_fence<LDS_>();
    for (int r = threadIdx.x; r < n; r += 64) {
        const double v = B[(size_t)r * W + KBS - 2];
        ok = ok && mid_range(v);
        eps[first + r] = v;
    }
    return !__ballot(!ok);
}

// The same for any U of half-bandwidth T, with divisions.
template <int T, int KBS>
__device__ __forceinline__ void band_back_rows(int first, int n, const double* __restrict__ B,
                                               const double* __restrict__ y, double* __restrict__ eps) {
    constexpr int W = 3 * KBS + 1;
    double x[T];
#pragma unroll
    for (int q = 0; q < T; q++) x[q] = 0.0;
    for (int i = n - 1; i >= 0; i--) {
        const double* U = B + (size_t)i * W + KBS;
        double s = y[i];
#pragma unroll
        for (int q = 0; q < T; q++) s = s - U[1 + q] * x[q];
        const double xi = s / U[0];
        if (threadIdx.x == 0) eps[first + i] = xi;
#pragma unroll
        for (int q = T - 1; q > 0; q--) x[q] = x[q - 1];
        x[0] = xi;
    }
}

// B: the band (rows of U replace it), y: the right-hand side; both either
// in LDS or in global memory (LDS_ selects the instantiation, so that every
// access is compiled for its own address space).  Wavefront 0 of the workgroup.
template <int KB, int KBS, bool LDS_>
__device__ __forceinline__ void eps_band_solve_impl(int first, int n, double* __restrict__ B, double* __restrict__ y,
                                                    double* __restrict__ eps) {
    static_assert(KB <= KBS && KB >= 2, "window wider than the stored band, or no sub-diagonal pair");
    if (threadIdx.x >= 64) return;
    const int moved = band_eliminate<KB, KBS>(n, B, y);
    band_fence<LDS_>();
    bool done;
    if (moved == 0) done = band_back_fast<KB, KBS, LDS_>(first, n, B, y, eps);
    else if (moved <= 2) done = band_back_fast<KB + 2, KBS, LDS_>(first, n, B, y, eps);
    else done = band_back_fast<2 * KB, KBS, LDS_>(first, n, B, y, eps);
    if (!done) band_back_rows<2 * KB, KBS>(first, n, B, y, eps);
}

// Largest |column - row| over the non-zero entries of rows [r0, r1) of a
// band stored with half-bandwidth KBS (entries q = 0..2KBS of each row).
template <int KBS>
__device__ __forceinline__ int band_width_rows(const double* __restrict__ B, long long t0, long long t1, int stride) {
    constexpr int W = 3 * KBS + 1;
    int bw = 0;
    for (long long t = t0; t < t1; t += stride) {
        const int q = (int)(t % W);
        if (q <= 2 * KBS && B[t] != 0.0) bw = max(bw, q < KBS ? KBS - q : q - KBS);
    }
    return bw;
}

// Elimination with the narrowest window that holds the matrix's non-zeros
// (bandwidth bw): the same operations on the non-zero entries, fewer on
// structural zeros, so the same values.
template <int KBS, bool LDS_>
__device__ __forceinline__ void eps_band_solve_bw(int bw, int first, int n, double* __restrict__ B,
                                                  double* __restrict__ y, double* __restrict__ eps) {
    if (bw <= 2) eps_band_solve_impl<2, KBS, LDS_>(first, n, B, y, eps);
    else if (bw == 3) eps_band_solve_impl<3, KBS, LDS_>(first, n, B, y, eps);
    else if (bw == 4) eps_band_solve_impl<4, KBS, LDS_>(first, n, B, y, eps);
    else eps_band_solve_impl<KBS, KBS, LDS_>(first, n, B, y, eps);
}

// One system per workgroup of kBandThreads lanes: all of them stage the band in
// LDS when it fits and measure its bandwidth on the way, the first wavefront
// solves with the matching window.  bw_sh: one int of LDS.
constexpr int kBandThreads = 256;

template <int KB>
__device__ __forceinline__ void eps_band_solve_body(int first, int n, double* __restrict__ G, double* __restrict__ ywork,
                                                    double* __restrict__ eps, int lds_rows, double* sm, int* bw_sh) {
    constexpr int W = 3 * KB + 1;
    const int nw = n * W;
    if (threadIdx.x == 0) *bw_sh = 0;
    __syncthreads();
    int bw = 0;
    if (n <= lds_rows) {
        constexpr int U = 8;  // loads in flight
        for (int t0 = threadIdx.x; t0 < nw; t0 += U * kBandThreads) {
            double v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = G[min(t0 + u * kBandThreads, nw - 1)];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = t0 + u * kBandThreads, q = t % W;
                if (t < nw) {
                    sm[t] = v[u];
                    if (q <= 2 * KB && v[u] != 0.0) bw = max(bw, q < KB ? KB - q : q - KB);
                }
            }
        }
    } else {
        bw = band_width_rows<KB>(G, threadIdx.x, nw, kBandThreads);
    }
    if (bw) atomicMax(bw_sh, bw);
    __syncthreads();
    bw = *bw_sh;
    if (n <= lds_rows) eps_band_solve_bw<KB, true>(bw, first, n, sm, sm + (long long)nw, eps);
    else eps_band_solve_bw<KB, false>(bw, first, n, G, ywork + first, eps);
}

template <int KB>
__global__ __launch_bounds__(kBandThreads) void k_eps_band_solve(const int* __restrict__ sys_first,
                                                                 const int* __restrict__ sys_n,
                                                                 const int* __restrict__ outside,
                                                                 double* __restrict__ band,
                                                                 const long long* __restrict__ band_off,
                                                                 double* __restrict__ ywork, double* __restrict__ eps,
                                                                 int lds_rows, int skip_upto) {
    extern __shared__ double sm[];
    __shared__ int bw;
    const int sys = blockIdx.x;
    coupling_priority();
    // skip_upto: systems of up to that many rows are the reduction's
    if (outside[sys] || sys_n[sys] <= skip_upto) return;
    eps_band_solve_body<KB>(sys_first[sys], sys_n[sys], band + band_off[sys], ywork, eps, lds_rows, sm, &bw);
}

template <int KB>
__global__ __launch_bounds__(kBandThreads) void k_eps_band_solve_batch(const CaseDev* __restrict__ cases,
                                                                       const CaseSys* __restrict__ sys, int lds_rows,
                                                                       int skip_upto) {
    extern __shared__ double sm[];
    __shared__ int bw;
    const CaseSys q = sys[blockIdx.x];
    const CaseDev& c = cases[q.c];
    if (c.eps.outside[q.k] || c.eps.n[q.k] <= skip_upto) return;
    eps_band_solve_body<KB>(c.eps.first[q.k], c.eps.n[q.k], c.eps.band + c.eps.off[q.k], c.eps.y, c.m.eps, lds_rows,
                            sm, &bw);
}

// ---------------------------------------------------------------- epsilon by cyclic reduction
// FP32-shifted cases: the banded epsilon system A eps = 1 of a body solved by
// block cyclic reduction instead of the pivoted elimination above.  With
// half-bandwidth bw <= Bk, A is block tridiagonal in Bk x Bk blocks (block
// row I: rows I*Bk .. I*Bk+Bk-1; padding rows beyond n are identity rows
// with a zero right-hand side).  At stride s = 1, 2, 4, ... the blocks at
// odd multiples of s are eliminated from their neighbours' equations, one
// lane per entry of each surviving block, and back substitution runs the
// levels in reverse: log2(n / Bk) dependent levels instead of n pivot
// steps.  A_ij = S_ij ds_j with S the Gram matrix of the markers' delta
// functions over the lattice (symmetric positive definite for distinct
// markers), so every Schur complement the reduction forms is S's Schur
// complement scaled by ds: no pivoting is needed.  The values agree with the
// pivoted elimination to rounding (the plain method keeps that one, whose
// operations are the reference's).  Systems of up to kCrMaxRows rows and
// half-bandwidth up to kCrMaxBw (blocks of 2 x 2 or 4 x 4); a wider band is
// solved by the pivoted elimination on wavefront 0 of the same kernel, and
// larger systems by the pivoted kernel.  The markers of a filament lie one
// lattice spacing apart, which bounds the half-bandwidth at 4; a lower limit
// (cr_max_bw) sends narrower bands to the fallback as well.
constexpr int kCrMaxRows = 384;
constexpr int kCrMaxBw = 4;

// Widest half-bandwidth the reduction takes: environment LIFE_EPS_CR_MAX_BW
// (0 .. 4, default 4; 0: every system by the pivoted elimination), read at
// each launch.
static int cr_max_bw() {
    const char* e = std::getenv("LIFE_EPS_CR_MAX_BW");
    const int v = e && *e ? std::atoi(e) : kCrMaxBw;
    return v < 0 ? 0 : (v > kCrMaxBw ? kCrMaxBw : v);
}

// LDS (doubles) of the reduction with Bk x Bk blocks over n rows: blocks,
// staged new blocks of a level, solution.
__host__ __device__ constexpr size_t cr_lds_doubles(int Bk, int n) {
    return (size_t)((n + Bk - 1) / Bk) * (3 * Bk * Bk + Bk) + (size_t)(((n + Bk - 1) / Bk + 1) / 2) * (3 * Bk * Bk + Bk) +
           (size_t)((n + Bk - 1) / Bk) * Bk;
}

// In-place inverse of a Bk x Bk block (row-major) by Gauss-Jordan
// elimination without pivoting, in registers.
template <int Bk>
__device__ __forceinline__ void cr_inverse(double* __restrict__ D) {
    double a[Bk][Bk];
#pragma unroll
    for (int i = 0; i < Bk; i++)
#pragma unroll
        for (int j = 0; j < Bk; j++) a[i][j] = D[Bk * i + j];
#pragma unroll
    for (int k = 0; k < Bk; k++) {
        const double p = 1.0 / a[k][k];
        a[k][k] = 1.0;
#pragma unroll
        for (int j = 0; j < Bk; j++) a[k][j] = a[k][j] * p;
#pragma unroll
        for (int i = 0; i < Bk; i++) {
            if (i == k) continue;
            const double f = a[i][k];
            a[i][k] = 0.0;
#pragma unroll
            for (int j = 0; j < Bk; j++) a[i][j] = a[i][j] - f * a[k][j];
        }
    }
#pragma unroll
    for (int i = 0; i < Bk; i++)
#pragma unroll
        for (int j = 0; j < Bk; j++) D[Bk * i + j] = a[i][j];
}

// The reduction of one system by the whole workgroup.  G: the band (KB = 8
// storage, LDS or global memory), read once into the blocks; blk: LDS for
// the blocks; work: LDS for the staged blocks and the solution (it may
// alias G when G is in LDS: G is read only before the first level).
template <int Bk>
__device__ __forceinline__ void eps_cr_solve(const double* __restrict__ G, int n, double* __restrict__ eps,
                                             double* __restrict__ blk, double* __restrict__ work) {
    constexpr int KB = 8, W = 3 * KB + 1;
    constexpr int BB = Bk * Bk, BLK = 3 * BB + Bk;  // A (sub), D (diagonal), C (super), f
    constexpr int oA = 0, oD = BB, oC = 2 * BB, oF = 3 * BB;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int nb = (n + Bk - 1) / Bk;
    // blocks from the band: eight entries per lane at a time, their loads
    // (unconditional, clamped address) issued before any is used
    constexpr int U = 8;
    const int total = nb * BLK;
    for (int base = 0; base < total; base += U * nt) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = base + u * nt + tid;
            const int I = t / BLK, q = t - I * BLK;
            const int part = q / BB, i = (q % BB) / Bk, j = q % Bk;
            const int r = I * Bk + i, c = (I + part - 1) * Bk + j, o = c - r;
            const bool band_entry = q < oF && r < n && c >= 0 && c < n && o >= -KB && o <= KB;
            const double a = G[band_entry ? (size_t)r * W + (o + KB) : 0];
            double val;
            if (q >= oF) val = I * Bk + (q - oF) < n ? 1.0 : 0.0;
            else if (r >= n) val = (part == 1 && i == j) ? 1.0 : 0.0;
            else val = band_entry ? a : 0.0;
            v[u] = val;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = base + u * nt + tid;
            if (t < total) blk[t] = v[u];
        }
    }
    __syncthreads();
    double* stage = work;
    double* x = work + (size_t)((nb + 1) / 2) * BLK;
    int s = 1;
    for (; s < nb; s *= 2) {
        for (int j = s + 2 * s * tid; j < nb; j += 2 * s * nt) cr_inverse<Bk>(blk + (size_t)BLK * j + oD);
        __syncthreads();
        const int nr = (nb - 1) / (2 * s) + 1;
        for (int t = tid; t < BB * nr; t += nt) {
            const int k = t / BB, r = (t % BB) / Bk, c = t % Bk, i = 2 * s * k;
            const double* bi = blk + (size_t)BLK * i;
            double Dn = bi[oD + Bk * r + c], An = 0.0, Cn = 0.0, fn = bi[oF + r];
            if (i - s >= 0) {
                const double* bj = blk + (size_t)BLK * (i - s);
                double al[Bk];
#pragma unroll
                for (int q = 0; q < Bk; q++) {
                    double a = 0.0;
#pragma unroll
                    for (int m = 0; m < Bk; m++) a += bi[oA + Bk * r + m] * bj[oD + Bk * m + q];
                    al[q] = a;
                }
                double dc = 0.0, da = 0.0, df = 0.0;
#pragma unroll
                for (int q = 0; q < Bk; q++) {
                    dc += al[q] * bj[oC + Bk * q + c];
                    da += al[q] * bj[oA + Bk * q + c];
                    df += al[q] * bj[oF + q];
                }
                Dn = Dn - dc;
                An = -da;
                fn = fn - df;
            }
            if (i + s < nb) {
                const double* bj = blk + (size_t)BLK * (i + s);
                double ga[Bk];
#pragma unroll
                for (int q = 0; q < Bk; q++) {
                    double a = 0.0;
#pragma unroll
                    for (int m = 0; m < Bk; m++) a += bi[oC + Bk * r + m] * bj[oD + Bk * m + q];
                    ga[q] = a;
                }
                double da = 0.0, dc = 0.0, df = 0.0;
#pragma unroll
                for (int q = 0; q < Bk; q++) {
                    da += ga[q] * bj[oA + Bk * q + c];
                    dc += ga[q] * bj[oC + Bk * q + c];
                    df += ga[q] * bj[oF + q];
                }
                Dn = Dn - da;
                Cn = -dc;
                fn = fn - df;
            }
            double* o = stage + (size_t)BLK * k;
            o[oA + Bk * r + c] = An;
            o[oD + Bk * r + c] = Dn;
            o[oC + Bk * r + c] = Cn;
            if (c == 0) o[oF + r] = fn;
        }
        __syncthreads();
        for (int t = tid; t < BLK * nr; t += nt) blk[(size_t)BLK * 2 * s * (t / BLK) + t % BLK] = stage[t];
        __syncthreads();
    }
    // block 0 alone: x_0 = inv(D_0) f_0
    if (tid == 0) cr_inverse<Bk>(blk + oD);
    __syncthreads();
    if (tid < Bk) {
        double a = 0.0;
#pragma unroll
        for (int m = 0; m < Bk; m++) a += blk[oD + Bk * tid + m] * blk[oF + m];
        x[tid] = a;
    }
    __syncthreads();
    // back substitution: x_j = inv(D_j) (f_j - A_j x_{j-s} - C_j x_{j+s})
    for (s /= 2; s >= 1; s /= 2) {
        const int ne = (nb + s - 1) / (2 * s);
        for (int t = tid; t < Bk * ne; t += nt) {
            const int j = s + 2 * s * (t / Bk), r = t % Bk;
            const double* bj = blk + (size_t)BLK * j;
            const double* xl = x + (size_t)Bk * (j - s);
            const bool right = j + s < nb;
            const double* xr = x + (size_t)Bk * (right ? j + s : j - s);
            double v[Bk];
#pragma unroll
            for (int a = 0; a < Bk; a++) {
                double ax = 0.0, cx = 0.0;
#pragma unroll
                for (int m = 0; m < Bk; m++) {
                    ax += bj[oA + Bk * a + m] * xl[m];
                    cx += bj[oC + Bk * a + m] * xr[m];
                }
                v[a] = bj[oF + a] - ax - (right ? cx : 0.0);
            }
            double xv = 0.0;
#pragma unroll
            for (int m = 0; m < Bk; m++) xv += bj[oD + Bk * r + m] * v[m];
            x[(size_t)Bk * j + r] = xv;
        }
        __syncthreads();
    }
    for (int k = tid; k < n; k += nt) eps[k] = x[k];
}

// Block size for a measured half-bandwidth (at most kCrMaxBw).
__device__ __forceinline__ void eps_cr_dispatch(int bw, const double* G, int n, double* eps, double* blk,
                                                double* work) {
    if (bw <= 2) eps_cr_solve<2>(G, n, eps, blk, work);
    else eps_cr_solve<4>(G, n, eps, blk, work);
}

// Half-bandwidth of a system's band in global memory (largest |column - row|
// over its non-zero entries), reduced over the workgroup.
__device__ __forceinline__ int band_width_wg(const double* __restrict__ G, int n, int* bw_sh) {
    constexpr int KB = 8, W = 3 * KB + 1;
    if (threadIdx.x == 0) *bw_sh = 0;
    __syncthreads();
    // sixteen loads in flight per lane (clamped addresses)
    constexpr int U = 16;
    const int total = n * W, nt = blockDim.x;
    int bw = 0;
    for (int base = 0; base < total; base += U * nt) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = G[min(base + u * nt + (int)threadIdx.x, total - 1)];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = base + u * nt + (int)threadIdx.x;
            const int q = t % W;
            if (t < total && q <= 2 * KB && v[u] != 0.0) bw = max(bw, q < KB ? KB - q : q - KB);
        }
    }
    atomicMax(bw_sh, bw);
    __syncthreads();
    return *bw_sh;
}

// LDS of the reduction kernels for systems of up to max_n rows (blocks of
// the widest size, 4).
static size_t eps_cr_lds(int max_n) {
    const int n = max_n < kCrMaxRows ? max_n : kCrMaxRows;
    return sizeof(double) * cr_lds_doubles(kCrMaxBw, n);
}

// One system per workgroup: the reduction, or for a band wider than
// kCrMaxBw the pivoted elimination on the band in device memory (ywork: its
// right-hand side) by wavefront 0.
__device__ __forceinline__ void eps_cr_or_pivot(double* __restrict__ G, int first, int n, double* __restrict__ ywork,
                                                double* __restrict__ eps, double* sm, int* bw_sh, int maxbw) {
    const int bw = band_width_wg(G, n, bw_sh);
    if (bw > maxbw) {
        eps_band_solve_bw<8, false>(bw, first, n, G, ywork + first, eps);
        return;
    }
    const int nb = (n + kCrMaxBw - 1) / kCrMaxBw;
    eps_cr_dispatch(bw, G, n, eps + first, sm, sm + (size_t)nb * (3 * kCrMaxBw * kCrMaxBw + kCrMaxBw));
}

__global__ __launch_bounds__(256) void k_eps_band_cr(const int* __restrict__ sys_first, const int* __restrict__ sys_n,
                                                     const int* __restrict__ outside, double* __restrict__ band,
                                                     const long long* __restrict__ band_off,
                                                     double* __restrict__ ywork, double* __restrict__ eps, int maxbw) {
    extern __shared__ double sm[];
    __shared__ int bw_sh;
    const int sys = blockIdx.x, n = sys_n[sys];
    coupling_priority();
    if (outside[sys] || n > kCrMaxRows) return;
    eps_cr_or_pivot(band + band_off[sys], sys_first[sys], n, ywork, eps, sm, &bw_sh, maxbw);
}

__global__ __launch_bounds__(256) void k_eps_band_cr_batch(const CaseDev* __restrict__ cases,
                                                           const CaseSys* __restrict__ sys, int maxbw) {
    extern __shared__ double sm[];
    __shared__ int bw_sh;
    const CaseSys q = sys[blockIdx.x];
    const CaseDev& c = cases[q.c];
    const int n = c.eps.n[q.k];
    if (c.eps.outside[q.k] || n > kCrMaxRows) return;
    eps_cr_or_pivot(c.eps.band + c.eps.off[q.k], c.eps.first[q.k], n, c.eps.y, c.m.eps, sm, &bw_sh, maxbw);
}

// ---------------------------------------------------------------- interpolation
// ObjectsClass::ibmKernelInterp body (IBMNode.cpp:26-58): rho and rho*u at
// the supports (GridClass::macroscopic values: force_xy only) interpolated
// with the support deltas, then F = 2 (Dt/Dx rho_I U - (rho u)_I).  One
// lane per (marker, support slot): each lane takes its support's moments
// and weighted terms, and the marker's first lane adds them up in support
// order, as the reference's loop does, so the nine gathers of nine
// populations are in flight at once.  kInterpMarkers markers per workgroup
// of kSupp lanes each.
constexpr int kInterpMarkers = 28;
constexpr int kInterpThreads = kInterpMarkers * kSupp;  // 252

template <typename T>
__device__ inline void interpolate_slots(const T* __restrict__ f, const MarkerDev& m, const GridScalars& g,
                                         int k0, double* __restrict__ sh, int t) {
    const int km = t / kSupp, s = t - km * kSupp;
    const int k = k0 + km;
    double* a = sh;
    double* bx = sh + kInterpThreads;
    double* by = sh + 2 * kInterpThreads;
    if (t < kInterpThreads && k < m.n && s < m.supp_cnt[k]) {
        const long long id = m.supp_site[k * kSupp + s];
        interpolate_terms(f, g.S, id, g.fcur ? g.fcur[id] : g.Fx, g.fcur ? g.fcur[g.S + id] : g.Fy,
                          m.supp_delta[k * kSupp + s], a[t], bx[t], by[t]);
    }
    __syncthreads();
    if (t < kInterpThreads && s == 0 && k < m.n) {
        double iR = 0.0, mx = 0.0, my = 0.0;
        const int cnt = m.supp_cnt[k];
        for (int q = 0; q < cnt; q++) {
            iR += a[t + q];
            mx += bx[t + q];
            my += by[t + q];
        }
        const double vs = g.velScale;
        m.force[2 * k] = 2.0 * (vs * iR * m.vel[2 * k] - mx);
        m.force[2 * k + 1] = 2.0 * (vs * iR * m.vel[2 * k + 1] - my);
    }
}

__device__ inline void spread_clear_one(double* __restrict__ fibm, long long S, const int* __restrict__ uniq,
                                        const int* __restrict__ uniq_n, int k);

// Workgroups past the first ib zero the force at the sites of the last spread,
// for a launch that a spread with new supports follows: the interpolation does
// not read that force, so the clear costs the chain no launch of its own.
template <typename T>
__global__ __launch_bounds__(256) void k_interpolate(const T* __restrict__ f, MarkerDev m, GridScalars g, int ib,
                                                     SpreadScratch sc, double* __restrict__ fibm) {
    __shared__ double sh[3 * kInterpThreads];
    coupling_priority();
    if ((int)blockIdx.x >= ib) {
        spread_clear_one(fibm, g.S, sc.uniq, sc.uniq_n, ((int)blockIdx.x - ib) * kInterpThreads + (int)threadIdx.x);
        return;
    }
    interpolate_slots(f, m, g, blockIdx.x * kInterpMarkers, sh, (int)threadIdx.x);
}

// Batched: the populations after this step's stream-collide.
template <typename T>
__global__ __launch_bounds__(256) void k_interpolate_batch(const CaseDev* __restrict__ cases,
                                                           const int* __restrict__ list) {
    __shared__ double sh[3 * kInterpThreads];
    const CaseDev& c = cases[list[blockIdx.y]];
    interpolate_slots(static_cast<const T*>(c.dst), c.m, c.g, blockIdx.x * kInterpMarkers, sh, (int)threadIdx.x);
}

// ---------------------------------------------------------------- spread
// The reference adds marker contributions to each site in marker order
// (ORDERED, IBMNode.cpp:67-83).  Here every (marker, support) pair takes a
// slot at its site, each touched site gets a compact index, the pairs are
// scattered into per-site lists, and one thread per site sorts its list by
// marker and sums it from zero: the same additions in the same order.

__device__ inline void spread_clear_one(double* __restrict__ fibm, long long S, const int* __restrict__ uniq,
                                        const int* __restrict__ uniq_n, int k) {
    if (k >= *uniq_n) return;
    const long long id = uniq[k];
    if (id < 0) return;
    fibm[id] = 0.0;
    fibm[S + id] = 0.0;
}

__device__ inline void spread_count_one(const MarkerDev& m, const SpreadScratch& sc, int p) {
    if (p >= m.n * kSupp) return;
    const int k = p / kSupp, s = p - k * kSupp;
    if (s >= m.supp_cnt[k]) return;
    const int site = m.supp_site[p];
    const int slot = atomicAdd(&sc.site_count[site], 1);
    sc.pair_slot[p] = slot;
    if (slot == 0) {
        const int u = atomicAdd(sc.uniq_n, 1);
        sc.uniq[u] = site;
        sc.site_uid[site] = u;
    }
}

__device__ inline void spread_scatter_one(const MarkerDev& m, const SpreadScratch& sc, int p) {
    if (p >= m.n * kSupp) return;
    const int k = p / kSupp, s = p - k * kSupp;
    if (s >= m.supp_cnt[k]) return;
    const int site = m.supp_site[p];
    const int slot = sc.pair_slot[p];
    if (slot >= kMaxPerSite) {
        *sc.overflow = 1;
        return;
    }
    sc.list[(long long)sc.site_uid[site] * kMaxPerSite + slot] = p;
}

__device__ inline void spread_reduce_one(const MarkerDev& m, const SpreadScratch& sc, double* __restrict__ fibm,
                                         long long S, int u) {
    if (u >= *sc.uniq_n) return;
    const int site = sc.uniq[u];
    int n = sc.site_count[site];
    if (n > kMaxPerSite) n = kMaxPerSite;
    int pairs[kMaxPerSite];
    for (int q = 0; q < n; q++) {
        const int p = sc.list[(long long)u * kMaxPerSite + q];
        int r = q - 1;
        while (r >= 0 && pairs[r] > p) {
            pairs[r + 1] = pairs[r];
            r--;
        }
        pairs[r + 1] = p;
    }
    double fx = 0.0, fy = 0.0;
    for (int q = 0; q < n; q++) {
        const int p = pairs[q];
        const int k = p / kSupp;
        const double d = m.supp_delta[p];
        const double e = m.eps[k], ds = m.ds[k];
        fx += m.force[2 * k] * e * ds * 1.0 * d;
        fy += m.force[2 * k + 1] * e * ds * 1.0 * d;
    }
    fibm[site] = fx;
    fibm[S + site] = fy;
    sc.site_count[site] = 0;
}

__global__ void k_spread_clear(double* __restrict__ fibm, long long S, const int* __restrict__ uniq,
                               const int* __restrict__ uniq_n) {
    spread_clear_one(fibm, S, uniq, uniq_n, blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void k_spread_reset(int* uniq_n) { *uniq_n = 0; }

__global__ void k_spread_count(MarkerDev m, SpreadScratch sc) {
    coupling_priority();
    spread_count_one(m, sc, blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void k_spread_scatter(MarkerDev m, SpreadScratch sc) {
    coupling_priority();
    spread_scatter_one(m, sc, blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void k_spread_reduce(MarkerDev m, SpreadScratch sc, double* __restrict__ fibm, long long S) {
    coupling_priority();
    spread_reduce_one(m, sc, fibm, S, blockIdx.x * blockDim.x + threadIdx.x);
}

// Spread of a case with few markers without lists: one wavefront per marker k
// finds the markers whose support blocks overlap k's (all blocks compared, 64
// a round, in ascending order; the four wavefronts of a workgroup share the
// reading, a quarter each), forms their contributions, seven markers of
// nine support lanes at a time, in a table by k's own sites, and lane o < 9
// adds up site o in marker order.  The first marker at a site owns it and
// writes its sum; the same additions in the same order as the passes above,
// with no atomics and no sorting.  The site list of the last spread has one
// entry per marker-support pair here, -1 where another marker owns the site.
// Every support site is overwritten, so only sites outside the present
// supports have to be cleared before.
//
// INTERP: the forces are not read but interpolated from the populations f on
// the way, by every wavefront that needs them (those of about seven markers
// each; the marker's own wavefront stores its force): interpolation and
// spread of rigid bodies in one launch without a wait between them.
//
// Bound by the launch and a chain of four dependent reads (blocks, supports,
// populations, sums in LDS).  The passes in one workgroup, with their atomics
// and lists in device memory, took 26 us for 530 markers against 6 us here; with
// the interpolation 17 us for 126 markers against 6 us.
// Up to kScanMaxMarkers markers: the comparisons grow with the square of their
// number, the five passes do not.  The markers of a case lie one after the other
// along its bodies, so the four of a workgroup are close together and most rounds
// of 64 meet none of them; a caller's may lie anywhere, and then every round is
// opened: hence limits of their own.  Spread alone at 2000, 4000, 6000 and 8192
// markers, here | passes: filaments 6.0 | 21.0, 8.5 | 23.3, 11.7 | 26.2, 17.6 |
// 29.7 us, scattered 8.6 | 20.3, 18.5 | 23.9, 31.6 | 27.9, 51.4 | 32.8.  Where
// the coupling keeps to a quarter of the device (few_cus), the comparisons take
// longer and the passes, atomics most of them, hardly: in a step of 4096 x 1040,
// 2420, 4840 and 7744 markers of filaments 14 | 26, 28 | 30, 52 | 36 us of kernels;
// scattered, spread alone, 1000, 2000 and 3000 markers 7.8 | 15.4, 17.2 | 17.9,
// 31 | 20.
constexpr int kScanMaxMarkers = 8192, kScanMaxMarkersFew = 5000;
constexpr int kScanMaxScattered = 5000, kScanMaxScatteredFew = 2000;
constexpr int kScanWaves = 4;    // markers per workgroup
constexpr int kScanGroup = 7;    // neighbours at a time, of kSupp lanes each
// More overlapping markers than this put more than kMaxPerSite pairs on one
// of the nine sites.
constexpr int kScanNear = kSupp * kMaxPerSite;

template <typename T, bool INTERP>
__device__ __forceinline__ void spread_scan_wg(const T* __restrict__ f, const MarkerDev& m, const GridScalars& g,
                                               const SpreadScratch& sc, double* __restrict__ fibm) {
    __shared__ unsigned short near_s[kScanWaves][kScanWaves][kScanNear];  // marker, quarter
    __shared__ int near_n[kScanWaves][kScanWaves];
    __shared__ double tx_s[kScanWaves][64], ty_s[kScanWaves][64];
    __shared__ int has_s[kScanWaves][64];
    __shared__ double terms_s[kScanWaves][INTERP ? 3 * 64 : 1];
    const int wv = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64;
    const int k = (int)blockIdx.x * kScanWaves + wv;
    const int4* box = reinterpret_cast<const int4*>(m.supp_box);
    const int k0 = (int)blockIdx.x * kScanWaves;
    const int4 bk = box[min(k, m.n - 1)];
    // each wavefront compares a quarter of the markers with all four of the
    // workgroup
    int4 bs[kScanWaves];
    int have[kScanWaves], lx = INT_MAX, ly = INT_MAX, hx = INT_MIN, hy = INT_MIN;
#pragma unroll
    for (int w = 0; w < kScanWaves; w++) {
        bs[w] = box[min(k0 + w, m.n - 1)];
        have[w] = 0;
        lx = min(lx, bs[w].x);
        ly = min(ly, bs[w].y);
        hx = max(hx, bs[w].x + bs[w].z);
        hy = max(hy, bs[w].y + bs[w].w);
    }
    const int part = (m.n + kScanWaves - 1) / kScanWaves, cb = wv * part, ce = min(cb + part, m.n);
    constexpr int U = 4;
    for (int c0 = cb; c0 < ce; c0 += 64 * U) {
        int4 bc[U];
#pragma unroll
        for (int u = 0; u < U; u++) bc[u] = box[min(c0 + 64 * u + lane, m.n - 1)];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = c0 + 64 * u + lane;
            const int4 b = bc[u];
            // mostly none of the 64 is near any of the four
            const bool any = (b.x < hx && lx < b.x + b.z && b.y < hy && ly < b.y + b.w) || c / kScanWaves == (int)blockIdx.x;
            if (!__ballot(any)) continue;
#pragma unroll
            for (int w = 0; w < kScanWaves; w++) {
                const bool overlap = b.z > 0 && bs[w].z > 0 && b.x < bs[w].x + bs[w].z && bs[w].x < b.x + b.z &&
                                     b.y < bs[w].y + bs[w].w && bs[w].y < b.y + b.w;
                const bool in = c < ce && (overlap || c == k0 + w);
                const unsigned long long mask = __ballot(in);
                const int at = have[w] + __popcll(mask & ((1ull << lane) - 1));
                if (in && at < kScanNear) near_s[w][wv][at] = (unsigned short)c;
                have[w] += __popcll(mask);
            }
        }
    }
    if (lane == 0)
#pragma unroll
        for (int w = 0; w < kScanWaves; w++) near_n[w][wv] = have[w];
    __syncthreads();
    if (k >= m.n) return;  // the whole wavefront; no workgroup barriers below
    double *tx = tx_s[wv], *ty = ty_s[wv];
    int* has = has_s[wv];
    const int own_site = lane < kSupp ? m.supp_site[k * kSupp + lane] : -1;
    // the quarters one after the other: neighbour e is entry e - end[h - 1] of
    // quarter h
    int end[kScanWaves], total = 0;
    bool full = false;
#pragma unroll
    for (int h = 0; h < kScanWaves; h++) {
        const int c = near_n[wv][h];
        full = full || c > kScanNear;
        end[h] = total += min(c, kScanNear);
    }
    if (full && lane == 0) *sc.overflow = 1;
    auto near = [&](int e) -> int {
        int h = 0, at = e;
#pragma unroll
        for (int r = 0; r + 1 < kScanWaves; r++)
            if (e >= end[r]) {
                h = r + 1;
                at = e - end[r];
            }
        return near_s[wv][h][at];
    };
    const int q = lane / kSupp, s = lane - q * kSupp;
    double fx = 0.0, fy = 0.0;
    int pairs = 0;
    bool owner = false;
    for (int g0 = 0; g0 < total; g0 += kScanGroup) {
        const int qn = min(kScanGroup, total - g0);
        const bool on = q < qn;
        const int j = near(on ? g0 + q : 0), p = j * kSupp + s;
        const int4 bj = box[j];
        const bool act = on && s < bj.z * bj.w;
        const int site = m.supp_site[p];
        const double d = m.supp_delta[p], e = m.eps[j], ds = m.ds[j];
        double Fx, Fy;
        if constexpr (INTERP) {
            double *ta = terms_s[wv], *tbx = ta + 64, *tby = ta + 128;
            const double vx = m.vel[2 * j], vy = m.vel[2 * j + 1];
            if (act)
                interpolate_terms(f, g.S, site, g.fcur ? g.fcur[site] : g.Fx, g.fcur ? g.fcur[g.S + site] : g.Fy, d,
                                  ta[lane], tbx[lane], tby[lane]);
            lane_exchange_fence();
            // every lane of the marker adds the terms up in support order
            double iR = 0.0, mx = 0.0, my = 0.0;
            const int first = q * kSupp, cnt = on ? bj.z * bj.w : 0;
#pragma unroll
            for (int r = 0; r < kSupp; r++) {
                const double va = ta[min(first + r, 63)], vbx = tbx[min(first + r, 63)], vby = tby[min(first + r, 63)];
                if (r < cnt) {
                    iR += va;
                    mx += vbx;
                    my += vby;
                }
            }
            Fx = 2.0 * (g.velScale * iR * vx - mx);
            Fy = 2.0 * (g.velScale * iR * vy - my);
            if (on && s == 0 && j == k) {
                m.force[2 * k] = Fx;
                m.force[2 * k + 1] = Fy;
            }
        } else {
            Fx = m.force[2 * j];
            Fy = m.force[2 * j + 1];
        }
        has[lane] = 0;
        lane_exchange_fence();
        const int w = max(bj.w, 1), i = bj.x + s / w - bk.x, jj = bj.y + s % w - bk.y;
        if (act && i >= 0 && i < bk.z && jj >= 0 && jj < bk.w) {
            const int o = q * kSupp + i * bk.w + jj;
            has[o] = 1;
            tx[o] = Fx * e * ds * 1.0 * d;
            ty[o] = Fy * e * ds * 1.0 * d;
        }
        lane_exchange_fence();
        if (lane < kSupp) {
#pragma unroll
            for (int r = 0; r < kScanGroup; r++) {
                const int o = r * kSupp + lane;
                const bool hit = r < qn && has[o] != 0;
                const double cx = tx[o], cy = ty[o];
                if (hit) {
                    if (pairs == 0) owner = near(g0 + r) == k;
                    pairs++;
                    fx += cx;
                    fy += cy;
                }
            }
        }
        lane_exchange_fence();
    }
    if (lane < kSupp) {
        const int p = k * kSupp + lane;
        const bool mine = owner && own_site >= 0;
        sc.uniq[p] = mine ? own_site : -1;
        if (mine) {
            sc.site_uid[own_site] = p;
            fibm[own_site] = fx;
            fibm[g.S + own_site] = fy;
            if (pairs > kMaxPerSite) *sc.overflow = 1;
        }
        if (p == 0) *sc.uniq_n = m.n * kSupp;
    }
}

template <typename T, bool INTERP>
__global__ __launch_bounds__(64 * kScanWaves) void k_spread_scan(const T* __restrict__ f, MarkerDev m, GridScalars g,
                                                                 SpreadScratch sc, double* __restrict__ fibm) {
    coupling_priority();
    spread_scan_wg<T, INTERP>(f, m, g, sc, fibm);
}

// Batched, grid.y = case.  Twelve cases of up to 129 markers: clear and scan
// 11 us, the five passes 22 us and three more launches.
__global__ __launch_bounds__(64 * kScanWaves) void k_spread_scan_batch(const CaseDev* __restrict__ cases,
                                                                       const int* __restrict__ list) {
    const CaseDev& c = cases[list[blockIdx.y]];
    if ((int)blockIdx.x * kScanWaves >= c.m.n) return;  // the whole workgroup
    spread_scan_wg<double, false>(nullptr, c.m, c.g, c.sc, c.fibm);
}

// Batched spread by passes, grid.y = case (the reset: one thread per case).
__global__ void k_spread_clear_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list) {
    const CaseDev& c = cases[list[blockIdx.y]];
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < c.sc.cap; k += gridDim.x * blockDim.x)
        spread_clear_one(c.fibm, c.g.S, c.sc.uniq, c.sc.uniq_n, k);
}

__global__ void k_spread_reset_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list, int n) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) *cases[list[q]].sc.uniq_n = 0;
}

__global__ void k_spread_count_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list) {
    const CaseDev& c = cases[list[blockIdx.y]];
    spread_count_one(c.m, c.sc, blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void k_spread_scatter_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list) {
    const CaseDev& c = cases[list[blockIdx.y]];
    spread_scatter_one(c.m, c.sc, blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void k_spread_reduce_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list) {
    const CaseDev& c = cases[list[blockIdx.y]];
    spread_reduce_one(c.m, c.sc, c.fibm, c.g.S, blockIdx.x * blockDim.x + threadIdx.x);
}

// Packed marker staging <-> per-case marker arrays.
__global__ void k_markers_in_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list,
                                   const double* __restrict__ stage) {
    const CaseDev& c = cases[list[blockIdx.y]];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= c.m.n) return;
    const double* q = stage + 4 * (long long)(c.moff + k);
    c.m.pos[2 * k] = q[0];
    c.m.pos[2 * k + 1] = q[1];
    c.m.vel[2 * k] = q[2];
    c.m.vel[2 * k + 1] = q[3];
}

__global__ void k_markers_out_batch(const CaseDev* __restrict__ cases, const int* __restrict__ list,
                                    double* __restrict__ stage) {
    const CaseDev& c = cases[list[blockIdx.y]];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= c.m.n) return;
    double* q = stage + 3 * (long long)(c.moff + k);
    q[0] = c.m.force[2 * k];
    q[1] = c.m.force[2 * k + 1];
    q[2] = c.m.eps[k];
}

static int eps_lds_rows(int KB, int max_n) {
    const int W = 3 * KB + 1;
    const int lds_rows = (int)((60 * 1024) / (sizeof(double) * (W + 1)));
    return max_n < lds_rows ? max_n : lds_rows;
}

void launch_eps_band(const MarkerDev& m, const GridScalars& g, const int* sys_first, const int* sys_n,
                     const int* host_n, int nsys, int KB, double* band, const long long* band_off, int* outside,
                     double* ywork, bool cr, hipStream_t s) {
    if (nsys <= 0 || KB != 8) return;
    int max_n = 0;
    for (int k = 0; k < nsys; k++) max_n = max_n > host_n[k] ? max_n : host_n[k];
    const int W = 3 * KB + 1;
    const long long ne = (long long)max_n * W;
    const int be = (int)((ne + 255) / 256);
    const bool stage_far = max_n <= kFarLdsMarkers;
    const size_t far_lds = stage_far ? sizeof(double) * 2 * (size_t)max_n : 0;
    k_eps_band_prep<<<dim3((unsigned)(be + 1), nsys), 256, far_lds, s>>>(m, g, sys_first, sys_n, KB, band, band_off,
                                                                          outside, be, stage_far ? 1 : 0);
    if (cr) {
        const size_t lds = eps_cr_lds(max_n);
        static LdsLimit limit;
        limit.allow((const void*)k_eps_band_cr, lds, eps_cr_lds(kCrMaxRows));
        k_eps_band_cr<<<nsys, 256, lds, s>>>(sys_first, sys_n, outside, band, band_off, ywork, m.eps, cr_max_bw());
        if (max_n <= kCrMaxRows) return;
    }
    // band, then right-hand side, in LDS for systems of up to lds_rows rows
    const int rows = eps_lds_rows(KB, max_n);
    k_eps_band_solve<8><<<nsys, kBandThreads, sizeof(double) * (size_t)rows * (W + 1), s>>>(
        sys_first, sys_n, outside, band, band_off, ywork, m.eps, rows, cr ? kCrMaxRows : 0);
}

static unsigned support_blocks(int markers) {
    constexpr int per = kSupportThreads / kHalf;
    return (unsigned)((markers + per - 1) / per);
}

void launch_support_ds(const MarkerDev& m, const GridScalars& g, int flexible_only, hipStream_t s) {
    if (m.n <= 0) return;
    k_support_ds<<<support_blocks(m.n), kSupportThreads, 0, s>>>(m, g, flexible_only);
}

void launch_epsilon_matrix(const MarkerDev& m, const GridScalars& g, int first, int n, double* A, hipStream_t s) {
    const long long t = (long long)n * n;
    if (t <= 0) return;
    k_epsilon_matrix<<<(unsigned)((t + 255) / 256), 256, 0, s>>>(m, g, first, n, A);
}

void launch_epsilon_rows(const MarkerDev& m, const GridScalars& g, int first, int n, int* count, int* col, double* val,
                         hipStream_t s) {
    if (n <= 0) return;
    k_epsilon_rows<<<(unsigned)((n + 3) / 4), 256, 0, s>>>(m, g, first, n, count, col, val);
}

template <typename T>
void launch_interpolate(const T* f, const MarkerDev& m, const GridScalars& g, bool clear, double* fibm,
                        const SpreadScratch& sc, hipStream_t s) {
    if (m.n <= 0) return;
    const int ib = (m.n + kInterpMarkers - 1) / kInterpMarkers;
    const int cb = clear ? (sc.cap + kInterpThreads - 1) / kInterpThreads : 0;
    k_interpolate<T><<<ib + cb, kInterpThreads, 0, s>>>(f, m, g, ib, sc, fibm);
}
template void launch_interpolate<double>(const double*, const MarkerDev&, const GridScalars&, bool, double*,
                                         const SpreadScratch&, hipStream_t);
template void launch_interpolate<float>(const float*, const MarkerDev&, const GridScalars&, bool, double*,
                                        const SpreadScratch&, hipStream_t);

bool spread_scans(const MarkerDev& m) {
    if (m.few_cus) return m.n <= (m.along_bodies ? kScanMaxMarkersFew : kScanMaxScatteredFew);
    return m.n <= (m.along_bodies ? kScanMaxMarkers : kScanMaxScattered);
}

static unsigned scan_blocks(const MarkerDev& m) { return (unsigned)((m.n + kScanWaves - 1) / kScanWaves); }

void launch_spread(const MarkerDev& m, const GridScalars& g, double* fibm, SpreadScratch& sc, SpreadClear clear,
                   hipStream_t s) {
    const int np = m.n * kSupp;
    const int cap = sc.cap;
    const bool scan = np > 0 && spread_scans(m);
    if (clear == SpreadClear::kAll) {
        launch_fill_f64(fibm, 0.0, g.S * 2, s);
    } else if (cap > 0 && (clear == SpreadClear::kList || !scan)) {
        k_spread_clear<<<(cap + 255) / 256, 256, 0, s>>>(fibm, g.S, sc.uniq, sc.uniq_n);
    }
    if (scan) {
        k_spread_scan<double, false><<<scan_blocks(m), 64 * kScanWaves, 0, s>>>(nullptr, m, g, sc, fibm);
        return;
    }
    k_spread_reset<<<1, 1, 0, s>>>(sc.uniq_n);
    if (np <= 0) return;
    k_spread_count<<<(np + 255) / 256, 256, 0, s>>>(m, sc);
    k_spread_scatter<<<(np + 255) / 256, 256, 0, s>>>(m, sc);
    k_spread_reduce<<<(cap + 127) / 128, 128, 0, s>>>(m, sc, fibm, g.S);
}

template <typename T>
void launch_interp_spread(const T* f, const MarkerDev& m, const GridScalars& g, double* fibm, SpreadScratch& sc,
                          hipStream_t s) {
    k_spread_scan<T, true><<<scan_blocks(m), 64 * kScanWaves, 0, s>>>(f, m, g, sc, fibm);
}
template void launch_interp_spread<double>(const double*, const MarkerDev&, const GridScalars&, double*, SpreadScratch&,
                                           hipStream_t);
template void launch_interp_spread<float>(const float*, const MarkerDev&, const GridScalars&, double*, SpreadScratch&,
                                          hipStream_t);

// ---------------------------------------------------------------- batched launchers
void launch_support_ds_batch(const CaseDev* cases, const int* list, int n, int max_markers, int flexible_only,
                             hipStream_t s) {
    if (n <= 0 || max_markers <= 0) return;
    k_support_ds_batch<<<dim3(support_blocks(max_markers), (unsigned)n), kSupportThreads, 0, s>>>(cases, list,
                                                                                                flexible_only);
}

void launch_eps_band_batch(const CaseDev* cases, const CaseSys* sys, int nsys, int max_n, int* outside_out,
                           bool cr, hipStream_t s) {
    constexpr int KB = 8, W = 3 * KB + 1;
    if (nsys <= 0 || max_n <= 0) return;
    const int be = (int)(((long long)max_n * W + 255) / 256);
    const bool stage_far = max_n <= kFarLdsMarkers;
    k_eps_band_prep_batch<<<dim3((unsigned)(be + 1), (unsigned)nsys), 256, stage_far ? 16 * (size_t)max_n : 0, s>>>(
        cases, sys, KB, be, stage_far ? 1 : 0, outside_out);
    if (cr) {
        static LdsLimit limit;
        const size_t lds = eps_cr_lds(max_n);
        limit.allow((const void*)k_eps_band_cr_batch, lds, eps_cr_lds(kCrMaxRows));
        k_eps_band_cr_batch<<<(unsigned)nsys, 256, lds, s>>>(cases, sys, cr_max_bw());
    }
    if (!cr || max_n > kCrMaxRows) {
        const int rows = eps_lds_rows(KB, max_n);
        k_eps_band_solve_batch<KB><<<(unsigned)nsys, kBandThreads, sizeof(double) * (size_t)rows * (W + 1), s>>>(
            cases, sys, rows, cr ? kCrMaxRows : 0);
    }
}

template <typename T>
void launch_interpolate_batch(const CaseDev* cases, const int* list, int n, int max_markers, hipStream_t s) {
    if (n <= 0 || max_markers <= 0) return;
    k_interpolate_batch<T><<<dim3((unsigned)((max_markers + kInterpMarkers - 1) / kInterpMarkers), (unsigned)n),
                             kInterpThreads, 0, s>>>(cases, list);
}
template void launch_interpolate_batch<double>(const CaseDev*, const int*, int, int, hipStream_t);
template void launch_interpolate_batch<float>(const CaseDev*, const int*, int, int, hipStream_t);

void launch_spread_batch(const CaseDev* cases, const int* list, int n, int max_markers, hipStream_t s) {
    if (n <= 0) return;
    const int np = max_markers * kSupp;
    const unsigned nc = (unsigned)((np + 255) / 256);
    if (np > 0) k_spread_clear_batch<<<dim3(nc, (unsigned)n), 256, 0, s>>>(cases, list);
    if (np > 0 && max_markers <= kScanMaxMarkers) {
        k_spread_scan_batch<<<dim3((unsigned)((max_markers + kScanWaves - 1) / kScanWaves), (unsigned)n),
                              64 * kScanWaves, 0, s>>>(cases, list);
        return;
    }
    k_spread_reset_batch<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(cases, list, n);
    if (np <= 0) return;
    k_spread_count_batch<<<dim3(nc, (unsigned)n), 256, 0, s>>>(cases, list);
    k_spread_scatter_batch<<<dim3(nc, (unsigned)n), 256, 0, s>>>(cases, list);
    k_spread_reduce_batch<<<dim3((unsigned)((np + 127) / 128), (unsigned)n), 128, 0, s>>>(cases, list);
}

void launch_markers_in_batch(const CaseDev* cases, const int* list, int n, int max_markers, const double* stage,
                             hipStream_t s) {
    if (n <= 0 || max_markers <= 0) return;
    k_markers_in_batch<<<dim3((unsigned)((max_markers + 127) / 128), (unsigned)n), 128, 0, s>>>(cases, list, stage);
}

void launch_markers_out_batch(const CaseDev* cases, const int* list, int n, int max_markers, double* stage,
                              hipStream_t s) {
    if (n <= 0 || max_markers <= 0) return;
    k_markers_out_batch<<<dim3((unsigned)((max_markers + 127) / 128), (unsigned)n), 128, 0, s>>>(cases, list, stage);
}

}  // namespace life
