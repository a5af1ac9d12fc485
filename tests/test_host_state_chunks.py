"""The buffers of a state transfer on the CPU, with the page-locked pool and the
events replaced by ones that fail at a given call: every buffer that was taken
is given back once, and a transfer that gets at least one buffer is done with
those it has."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>
#include "state_chunks.h"

static int takes_left, events_left;
static std::map<void*, size_t> held;
static bool bad = false;

namespace life {
void* pinned_take(size_t n) {
    if (takes_left-- <= 0) throw std::bad_alloc();
    void* p = std::malloc(n);
    held[p] = n;
    return p;
}
void pinned_give(void* p, size_t n) {
    if (!p) return;
    if (!held.count(p) || held[p] != n) bad = true;
    held.erase(p);
    std::free(p);
}
}  // namespace life

extern "C" {
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (events_left-- <= 0) return hipErrorOutOfMemory;
    *e = (hipEvent_t)(size_t)1;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
}

int main() {
    using life::StateChunks;
    const size_t N = 2500000;  // six chunks of rho, u and force
    std::vector<double> rho(N), u(2 * N), b(2 * N);
    for (int takes = 0; takes <= 5; takes++)
        for (int events = 0; events <= 5; events++) {
            takes_left = takes;
            events_left = events;
            life_grid g;
            g.g.N = (long long)N;
            bool threw = false;
            size_t depth = 0;
            try {
                StateChunks ch(&g, nullptr, rho.data(), u.data(), b.data());
                depth = ch.depth();
                for (size_t k = 0; k < ch.count() + ch.depth(); k++) {
                    if (k >= ch.depth()) {
                        ch.wait(k - ch.depth());
                        ch.copy(k - ch.depth(), true);
                    }
                    if (k >= ch.count()) continue;
                    const StateChunks::Part p = ch.part(k);
                    for (long long q = 0; q < p.n; q++) {
                        p.rho[q] = (double)(p.first + q);
                        p.u[2 * q] = p.u[2 * q + 1] = p.fibm[2 * q] = p.fibm[2 * q + 1] = 1.0;
                    }
                    ch.record(k);
                }
            } catch (const std::bad_alloc&) {
                threw = true;
            } catch (const life::HipError&) {
                threw = true;
            }
            bool whole = true;
            for (size_t q = 0; q < N && whole; q++) whole = rho[q] == (double)q;
            if (!held.empty() || bad || (!threw && !whole)) {
                std::printf("takes %d events %d: %zu buffers held, depth %zu, threw %d, whole %d\n", takes, events,
                            held.size(), depth, (int)threw, (int)whole);
                return 1;
            }
            // an event for each buffer, and one ahead of the buffer that could not be had
            const bool enough = takes > 0 && events >= (takes < 4 ? takes + 1 : 4);
            if (threw == enough) {
                std::printf("takes %d events %d: threw %d\n", takes, events, (int)threw);
                return 1;
            }
            std::fill(rho.begin(), rho.end(), -1.0);
        }
    std::puts("ok");
}
"""


def test_buffers_are_given_back(tmp_path):
    src, exe = tmp_path / "chunks.cpp", tmp_path / "chunks"
    src.write_text(SOURCE)
    csrc = os.path.join(ROOT, "life_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fopenmp", "-D__HIP_PLATFORM_AMD__", "-I", csrc,
                           "-I", "/opt/rocm/include", "-o", str(exe), str(src)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
