"""lu_solve_rows on the CPU with an allocator that fails at a given call: the
work space that a failed solve leaves behind gives the next system its own
solution, that of a fresh work space."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>
#include "lu.h"

static long left = -1;  // allocations until one fails, -1: none
void* operator new(size_t n) {
    if (left == 0) {
        left = -1;
        throw std::bad_alloc();
    }
    if (left > 0) left--;
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// a band of half-bandwidth bw, entries by seed
struct System {
    static constexpr int cap = 32;
    std::vector<int> count, col;
    std::vector<double> val, b;
    System(int n, int bw, unsigned seed) : count(n, 0), col((size_t)n * cap), val((size_t)n * cap), b(n, 1.0) {
        for (int r = 0; r < n; r++)
            for (int c = r > bw ? r - bw : 0; c < n && c <= r + bw; c++) {
                seed = seed * 1664525u + 1013904223u;
                col[(size_t)r * cap + count[r]] = c;
                val[(size_t)r * cap + count[r]++] = 0.1 + (seed >> 8) / 16777216.0;
            }
    }
    int solve(std::vector<double>& x, life::LuWork& w) const {
        return life::lu_solve_rows((int)b.size(), cap, count.data(), col.data(), val.data(), b.data(), x.data(), w);
    }
};

int main() {
    const int n = 70;
    const System first(n, 6, 1), next(n, 2, 2);
    std::vector<double> x(n), want(n);
    {
        life::LuWork w;
        next.solve(want, w);
    }
    int failures = 0;
    for (long k = 0; k < 200; k++) {
        life::LuWork w;
        bool threw = false;
        left = k;
        try {
            first.solve(x, w);
        } catch (const std::bad_alloc&) {
            threw = true;
        }
        left = -1;
        failures += threw;
        next.solve(x, w);
        if (std::memcmp(x.data(), want.data(), sizeof(double) * n)) {
            std::printf("allocation %ld failed: the next solution differs\n", k);
            return 1;
        }
        if (!threw) break;
    }
    std::printf("%d failed allocations\n", failures);
    return failures < 5;
}
"""


def test_work_space_after_a_failed_solve(tmp_path):
    src, exe = tmp_path / "lu_rows.cpp", tmp_path / "lu_rows"
    src.write_text(SOURCE)
    csrc = os.path.join(ROOT, "life_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-I", csrc, "-o", str(exe), str(src),
                           os.path.join(csrc, "lu.cpp")])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
