// A grid's state between the device and the caller's arrays.
#pragma once

#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

#include "runtime.h"

namespace life {

// One transfer of a grid's state in the reference layout, in chunks of sites
// through page-locked buffers: the device reads or writes a buffer over the
// link (launch_materialise, launch_upload) while the host's threads copy
// others from or to the caller's arrays.  A copy straight to pageable memory
// runs at 18 GB/s, this at the link's rate (57 GB/s) as far as the host's
// threads keep up, and needs no device memory: 4096 x 2048, rho and u
// (201 MB) 12.0 -> 4.2 ms, 8192 x 4096 47 -> 15.  The buffers come from the pool
// of page-locked blocks and go back to it.
class StateChunks {
  public:
    struct Part {
        long long first, n;
        double *f, *rho, *u, *fibm;
    };
    StateChunks(life_grid* g, double* f, double* rho, double* u, double* fibm) : g_(g), user_{f, rho, u, fibm} {
        size_t per = 0;  // doubles per site
        for (int a = 0; a < 4; a++)
            if (user_[a]) per += kWidth[a];
        const size_t N = (size_t)g->g.N;
        if (per == 0) return;
        // buffers of a power of two, so that lattices of many sizes share them
        bytes_ = kMinBytes;
        while (bytes_ < kMaxBytes && bytes_ < N * per * sizeof(double)) bytes_ *= 2;
        sites_ = bytes_ / (per * sizeof(double));
        if (sites_ > 64) sites_ = sites_ / 64 * 64;
        count_ = (N + sites_ - 1) / sites_;
        depth_ = count_ < kDepth ? count_ : kDepth;
        for (size_t b = 0; b < depth_; b++) {
            if (!g->ev_state[b]) LIFE_HIP(hipEventCreateWithFlags(&g->ev_state[b], hipEventDisableTiming));
            try {
                buf_[b].take(bytes_);
            } catch (const std::bad_alloc&) {
                if (b == 0) throw;
                depth_ = b;  // one buffer is enough
            }
        }
    }
    StateChunks(const StateChunks&) = delete;
    StateChunks& operator=(const StateChunks&) = delete;
    ~StateChunks() {
        // the device is done with the buffers (an error may have come between)
        if (open_) (void)hipStreamSynchronize(g_->stream);
    }
    size_t count() const { return count_; }
    size_t depth() const { return depth_; }
    Part part(size_t k) const {
        Part p{(long long)(k * sites_), 0, nullptr, nullptr, nullptr, nullptr};
        p.n = (long long)std::min(sites_, (size_t)g_->g.N - k * sites_);
        double* at = buf_[k % depth_].p;
        double** out[4] = {&p.f, &p.rho, &p.u, &p.fibm};
        for (int a = 0; a < 4; a++) {
            if (!user_[a]) continue;
            *out[a] = at;
            at += kWidth[a] * sites_;
        }
        return p;
    }
    // Chunk k's launch is queued.
    void record(size_t k) {
        open_ = true;
        LIFE_HIP(hipGetLastError());
        LIFE_HIP(hipEventRecord(g_->ev_state[k % depth_], g_->stream));
    }
    void wait(size_t k) {
        LIFE_HIP(hipEventSynchronize(g_->ev_state[k % depth_]));
        if (k + 1 == count_) open_ = false;
    }
    // Chunk k between its buffer and the caller's arrays.
    void copy(size_t k, bool to_user) const {
        const Part p = part(k);
        double* buf[4] = {p.f, p.rho, p.u, p.fibm};
        struct Piece {
            double *dst, *src;
            size_t n;
        };
        std::vector<Piece> pieces;
        constexpr size_t kPiece = 1 << 15;  // doubles a thread takes at a time
        for (int a = 0; a < 4; a++) {
            if (!user_[a]) continue;
            const size_t n = kWidth[a] * (size_t)p.n;
            double* user = user_[a] + kWidth[a] * (size_t)p.first;
            for (size_t o = 0; o < n; o += kPiece) {
                const size_t m = std::min(kPiece, n - o);
                if (to_user) pieces.push_back({user + o, buf[a] + o, m});
                else pieces.push_back({buf[a] + o, user + o, m});
            }
        }
        const int np = (int)pieces.size();
#pragma omp parallel for schedule(dynamic, 1) if (np > 4)
        for (int q = 0; q < np; q++) std::memcpy(pieces[q].dst, pieces[q].src, pieces[q].n * sizeof(double));
    }

  private:
    static constexpr size_t kWidth[4] = {9, 1, 2, 2};  // doubles per site of f, rho, u, force_ibm
    static constexpr size_t kMinBytes = size_t(64) << 10, kMaxBytes = size_t(16) << 20;
    static constexpr size_t kDepth = life_grid::kStateDepth;
    life_grid* g_;
    double* user_[4];
    // a member each, so that an error in the constructor gives back those
    // already taken
    struct Buffer {
        double* p = nullptr;
        size_t bytes = 0;
        void take(size_t n) {
            p = static_cast<double*>(pinned_take(n));
            bytes = n;
        }
        ~Buffer() { pinned_give(p, bytes); }
    };
    Buffer buf_[kDepth];
    size_t bytes_ = 0, sites_ = 1, count_ = 0, depth_ = 0;
    bool open_ = false;
};

}  // namespace life
