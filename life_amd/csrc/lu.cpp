#include "lu.h"

#include <emmintrin.h>

#include <cmath>
#include <cstring>

namespace life {

namespace {

// The elimination on the m rows in w (rows B, their non-zero patterns bits,
// right-hand sides y), into x[0..m).  Rows stay where they are: row[p] is the
// row at position p of the canonical algorithm, pos its inverse.
//
// A row takes part from the column of its first non-zero on (before that its
// entries in the pivot column are zero), so a step looks at the active rows
// only, and at the pattern of the pivot row instead of all columns.
int eliminate(LuWork& w, int m, double* x) {
    const int words = (m + 63) / 64;
    double* const B = w.B.data();
    double* const y = w.y.data();
    uint64_t* const bits = w.bits.data();
    auto row = [&](int r) { return B + (size_t)r * m; };
    auto pat = [&](int r) { return bits + (size_t)r * words; };
    w.row.resize(m);
    w.pos.resize(m);
    w.head.assign(m + 1, -1);
    w.next.resize(m);
    w.cols.resize(m);
    w.act.clear();
    for (int r = 0; r < m; r++) {
        w.row[r] = w.pos[r] = r;
        int f = m;  // first non-zero column
        for (int q = 0; q < words && f == m; q++)
            if (pat(r)[q]) f = q * 64 + __builtin_ctzll(pat(r)[q]);
        w.next[r] = w.head[f];
        w.head[f] = r;
    }
    int info = 0;
    int* const cols = w.cols.data();
    for (int k = 0; k < m; k++) {
        for (int r = w.head[k]; r >= 0; r = w.next[r])
            if (w.pos[r] >= k) w.act.push_back(r);  // (else U's row of a column without a pivot)
        // first row of maximum magnitude, by position
        int p = k;
        double best = std::fabs(row(w.row[k])[k]);
        for (int r : w.act) {
            const double a = std::fabs(row(r)[k]);
            if (a > best || (a == best && w.pos[r] < p)) {
                best = a;
                p = w.pos[r];
            }
        }
        if (best == 0.0) {
            if (!info) info = k + 1;
            // the row at position k keeps its place, as U's row k
            for (size_t q = 0; q < w.act.size(); q++)
                if (w.pos[w.act[q]] == k) {
                    w.act[q] = w.act.back();
                    w.act.pop_back();
                    break;
                }
            continue;
        }
        const int rp = w.row[p], rq = w.row[k];
        w.row[p] = rq;
        w.pos[rq] = p;
        w.row[k] = rp;
        w.pos[rp] = k;
        const double* const rk = row(rp);
        const uint64_t* const pk = pat(rp);
        const double piv = rk[k];
        int nc = 0;
        const int w0 = (k + 1) / 64;
        for (int q = w0; q < words; q++) {
            uint64_t b = pk[q];
            if (q == w0) b &= ~uint64_t(0) << ((k + 1) % 64);
            for (; b; b &= b - 1) {
                const int j = q * 64 + __builtin_ctzll(b);
                if (rk[j] != 0.0) cols[nc++] = j;
            }
        }
        size_t keep = 0;
        for (int r : w.act) {
            if (r == rp) continue;
            w.act[keep++] = r;
            double* const ri = row(r);
            if (ri[k] == 0.0) continue;
            const double l = ri[k] / piv;
            ri[k] = l;
            for (int q = 0; q < nc; q++) {
                const int j = cols[q];
                ri[j] = ri[j] - l * rk[j];
            }
            uint64_t* const pi = pat(r);
            for (int q = w0; q < words; q++) pi[q] |= pk[q];
            y[r] = y[r] - l * y[rp];
        }
        w.act.resize(keep);
    }
    for (int i = m - 1; i >= 0; i--) {
        const int r = w.row[i];
        const double* const ri = row(r);
        const uint64_t* const pi = pat(r);
        double s = y[r];
        const int w0 = (i + 1) / 64;
        for (int q = w0; q < words; q++) {
            uint64_t b = pi[q];
            if (q == w0) b &= ~uint64_t(0) << ((i + 1) % 64);
            for (; b; b &= b - 1) {
                const int j = q * 64 + __builtin_ctzll(b);
                if (ri[j] != 0.0) s = s - ri[j] * x[j];
            }
        }
        x[i] = s / ri[i];
    }
    return info;
}

}  // namespace

int lu_solve_sparse(int n, int bc, const double* A, const double* b, double* x, LuWork& w) {
    const int m = n - bc, words = (m + 63) / 64;
    w.rows_m = 0;  // B is overwritten as a whole
    w.B.resize((size_t)m * m);
    w.y.resize(m);
    w.bits.assign((size_t)m * words, 0);
    for (int i = 0; i < m; i++) {
        const double* a = A + (size_t)(i + bc) * n + bc;
        std::memcpy(&w.B[(size_t)i * m], a, sizeof(double) * m);
        uint64_t* p = &w.bits[(size_t)i * words];
        int j = 0;
        for (; j + 2 <= m; j += 2)
            p[j / 64] |= (uint64_t)_mm_movemask_pd(_mm_cmpneq_pd(_mm_loadu_pd(a + j), _mm_setzero_pd())) << (j % 64);
        for (; j < m; j++) p[j / 64] |= (uint64_t)(a[j] != 0.0) << (j % 64);
        w.y[i] = b[i + bc];
    }
    const int info = eliminate(w, m, x + bc);
    for (int i = 0; i < bc; i++) x[i] = 0.0;
    return info;
}

int lu_solve_rows(int n, int cap, const int* count, const int* col, const double* val, const double* b, double* x,
                  LuWork& w) {
    const int words = (n + 63) / 64;
    const bool fits = w.rows_m == n;
    w.rows_m = 0;  // until B is zero again (memory may run out on the way)
    if (!fits) {
        w.B.assign((size_t)n * n, 0.0);
        w.bits.assign((size_t)n * words, 0);
        w.y.resize(n);
    }
    for (int r = 0; r < n; r++) {
        double* const ri = &w.B[(size_t)r * n];
        uint64_t* const p = &w.bits[(size_t)r * words];
        for (int q = 0; q < count[r]; q++) {
            const int j = col[(size_t)r * cap + q];
            ri[j] = val[(size_t)r * cap + q];
            p[j / 64] |= uint64_t(1) << (j % 64);
        }
        w.y[r] = b[r];
    }
    const int info = eliminate(w, n, x);
    // zero again for the next system: only what the patterns name was written
    for (int r = 0; r < n; r++) {
        double* const ri = &w.B[(size_t)r * n];
        uint64_t* const p = &w.bits[(size_t)r * words];
        for (int q = 0; q < words; q++) {
            for (uint64_t v = p[q]; v; v &= v - 1) ri[q * 64 + __builtin_ctzll(v)] = 0.0;
            p[q] = 0;
        }
    }
    w.rows_m = n;
    return info;
}

void BandMatrix::resize(int n_, int kl_, int ku_) {
    n = n_;
    kl = kl_;
    ku = ku_;
    w = 2 * kl + ku + 1;
    data.assign((size_t)n * w, 0.0);
}

void BandMatrix::zero() { std::memset(data.data(), 0, sizeof(double) * data.size()); }

namespace {
// row_i[j] -= l * row_k[j] for j in [lo, hi] (rows k != i: no aliasing)
inline void axpy_row(double* __restrict ri, const double* __restrict rk, double l, int lo, int hi) {
    for (int j = lo; j <= hi; j++) ri[j] = ri[j] - l * rk[j];
}
}  // namespace

// Row operations touch only the columns a row can hold non-zeros in:
// last[r] is the last such column of row r (its band, widened by the fill
// of row swaps and updates).  Entries past it are exact zeros, so the
// skipped operations (a - l * 0, s - 0 * x) would leave every value as it
// is.  Without row swaps (the diagonally dominant FEM and epsilon systems)
// each update covers ku columns instead of kl + ku.
int lu_solve_band(const BandMatrix& A, int bc, const double* b, double* x, BandMatrix& W, std::vector<double>& y) {
    const int n = A.n, kl = A.kl, ku = A.ku;
    const int m = n - bc;
    if (W.n != m || W.kl != kl || W.ku != ku) W.resize(m, kl, ku);
    // row(r)[c] is entry (r, c) for c in [r - kl, r + kl + ku]
    const int w = W.w;
    double* const base = W.data.data();
    auto row = [&](int r) { return base + (ptrdiff_t)r * w + kl - r; };
    const double* const abase = A.data.data();
    auto arow = [&](int r) { return abase + (ptrdiff_t)r * A.w + kl - r; };
    y.resize(2 * (size_t)m);
    double* const yv = y.data();
    int* const last = reinterpret_cast<int*>(yv + m);  // m ints in the second half
    const int kext = kl + ku;
    // copy the trailing block; the fill columns past the original upper band start at zero
    for (int r = 0; r < m; r++) {
        const int lo = r - kl < 0 ? 0 : r - kl;
        const int hi = r + ku > m - 1 ? m - 1 : r + ku;
        const int top = r + kext > m - 1 ? m - 1 : r + kext;
        double* wr = row(r);
        const double* ar = arow(r + bc) + bc;
        for (int c = lo; c <= hi; c++) wr[c] = ar[c];
        for (int c = hi + 1; c <= top; c++) wr[c] = 0.0;
        last[r] = hi;
        yv[r] = b[r + bc];
    }
    int info = 0;
    for (int k = 0; k < m; k++) {
        const int ilast = k + kl > m - 1 ? m - 1 : k + kl;
        int p = k;
        double best = std::fabs(row(k)[k]);
        for (int i = k + 1; i <= ilast; i++) {
            const double a = std::fabs(row(i)[k]);
            if (a > best) {
                best = a;
                p = i;
            }
        }
        if (best == 0.0) {
            if (!info) info = k + 1;
            continue;
        }
        double* rk = row(k);
        if (p != k) {
            double* rp = row(p);
            const int jl = last[k] > last[p] ? last[k] : last[p];
            for (int j = k; j <= jl; j++) {
                const double t = rk[j];
                rk[j] = rp[j];
                rp[j] = t;
            }
            const int tl = last[k];
            last[k] = last[p];
            last[p] = tl;
            const double t = yv[k];
            yv[k] = yv[p];
            yv[p] = t;
        }
        const double piv = rk[k];
        const int jlast = last[k];
        for (int i = k + 1; i <= ilast; i++) {
            double* ri = row(i);
            const double l = ri[k] / piv;
            ri[k] = l;
            axpy_row(ri, rk, l, k + 1, jlast);
            if (last[i] < jlast) last[i] = jlast;
            yv[i] = yv[i] - l * yv[k];
        }
    }
    for (int i = m - 1; i >= 0; i--) {
        const double* ri = row(i);
        double s = yv[i];
        const int jlast = last[i];
        for (int j = i + 1; j <= jlast; j++) s = s - ri[j] * x[j + bc];
        x[i + bc] = s / ri[i];
    }
    for (int i = 0; i < bc; i++) x[i] = 0.0;
    return info;
}

}  // namespace life
