// ql_state_out.hpp -- results on their way to the caller's memory.
//
// States, gradients and the small per-run records leave the device through
// pinned host memory that a kernel writes, in the caller's layout (HD_fullU's
// two fields without the two it does not have), and that host threads copy out
// of while the next piece is on its way.  Pageable copies take a staging round
// trip for each array (35 us for a few KB) and one thread's copy, which also
// meets the page faults of memory touched for the first time (17 GB/s of a
// warm array, 10 of a fresh one; the link does 50).
// Measured, pageable copies -> this: a state of 89 MB into fresh memory 8.5 -> 2.2
// ms, 22 MB 1.66 -> 0.88, 11 MB of HD_fullU 2.3 -> 0.47, 0.2 MB 113 -> 26 us.
#pragma once
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>

#include "ql_runtime.hpp"

namespace qlk {

struct StateOut {
    const double2 *u;  // rows of rowlen values, rowstride apart
    int rows, rowlen, rowstride;
    double2 *dst;
    const double2 *mf;
    int nmf;
    double2 *dst_mf;
    const double *k;  // a last array of doubles
    int nk;
    double *dst_k;
};

// Writes over the link are 16 bytes per lane, whole wavefronts consecutive
[[maybe_unused]] static __global__ __launch_bounds__(NT) void k_state_out(StateOut a)
{
    const int id = blockIdx.x * NT + threadIdx.x, step = gridDim.x * NT;
    const int n = a.rows * a.rowlen;
    for (int k = id; k < n; k += step)
        a.dst[k] = a.u[a.rowlen == a.rowstride ? (size_t)k : (size_t)(k / a.rowlen) * a.rowstride + k % a.rowlen];
    for (int k = id; k < a.nmf; k += step) a.dst_mf[k] = a.mf[k];
    for (int k = id; k < a.nk; k += step) a.dst_k[k] = a.k[k];
}

}  // namespace qlk

namespace qlh {

// Pieces of at most OUT_SLOT bytes, OUT_SLOTS of them in flight; from
// OUT_THREADED pieces on, copied by up to OUT_SLOTS threads, whose start takes
// as long as half a piece's copy (pieces of 1 MiB, 16 of them, measured the same)
constexpr size_t OUT_SLOT = (size_t)2 << 20;
constexpr int OUT_SLOTS = 8, OUT_THREADED = 3;

// One context's pinned memory: the slots, then a tail for everything but the
// fluctuations, allocated with the first result that leaves through it.  Where
// none can be had, host stays null and results take the runtime's own copies.
struct Staging {
    std::mutex mu;  // calls of several threads on one context take turns
    bool tried = false;
    char *host = nullptr;
    size_t slot = 0, tail = 0;
    int n = 0;
    hipEvent_t ev[OUT_SLOTS] = {};
    char *tail_ptr() const { return host + slot * n; }
    ~Staging()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (host) (void)hipHostFree(host);
    }
};

// sized for the largest run's fluctuations (lin bytes) and tail
inline void staging_create(Staging **out, size_t lin, size_t tail)
{
    std::unique_ptr<Staging> s(new Staging);
    s->slot = std::min((lin + 255) / 256 * 256, OUT_SLOT);
    s->n = (int)std::min<size_t>((lin + s->slot - 1) / s->slot, OUT_SLOTS);
    s->tail = (tail + 255) / 256 * 256;
    *out = s.release();
}

// the memory, and the events of several slots (with mu held)
inline int staging_get(Staging &s)
{
    if (s.tried) return QL_OK;
    for (int k = 0; s.n > 1 && k < s.n; ++k)
        if (!s.ev[k]) QL_HIP(hipEventCreateWithFlags(&s.ev[k], hipEventDisableTiming));
    if (hipHostMalloc((void **)&s.host, s.slot * s.n + s.tail, hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        s.host = nullptr;
    }
    s.tried = true;
    return QL_OK;
}

// rows of rowlen values, rowstride apart from u on, to lin; nmf values to mf and
// nk doubles to k (each left out where its destination is null), in stream
// order on st; returns when all are there
inline int state_out(Staging &sg, hipStream_t st, const double2 *u, int rows, int rowlen, int rowstride, void *lin,
                     const double2 *mf_src, int nmf, void *mf, const double *k_src, int nk, void *k)
{
    if (!lin) rows = 0;
    if (!mf) nmf = 0;
    if (!k) nk = 0;
    const size_t row_bytes = sizeof(double2) * rowlen, mf_bytes = sizeof(double2) * nmf, k_bytes = sizeof(double) * nk;
    std::lock_guard<std::mutex> lock(sg.mu);
    QL_RC(staging_get(sg));
    if (!sg.host || mf_bytes + k_bytes > sg.tail || (rows && row_bytes > sg.slot)) {
        if (rows)
            QL_HIP(hipMemcpy2DAsync(lin, row_bytes, u, sizeof(double2) * rowstride, row_bytes, rows,
                                    hipMemcpyDeviceToHost, st));
        if (nmf) QL_HIP(hipMemcpyAsync(mf, mf_src, mf_bytes, hipMemcpyDeviceToHost, st));
        if (nk) QL_HIP(hipMemcpyAsync(k, k_src, k_bytes, hipMemcpyDeviceToHost, st));
        QL_HIP(hipStreamSynchronize(st));
        return QL_OK;
    }
    const int per = rows ? (int)std::min<size_t>(sg.slot / row_bytes, rows) : 0;
    const int np = rows ? (rows + per - 1) / per : 0;  // pieces
    auto issue = [&](int c) -> int {
        qlk::StateOut a{};
        a.u = u + (size_t)c * per * rowstride;
        a.rows = rows ? std::min(per, rows - c * per) : 0;
        a.rowlen = rowlen;
        a.rowstride = rowstride;
        a.dst = reinterpret_cast<double2 *>(sg.host + sg.slot * (c % sg.n));
        if (c == 0) {
            a.mf = mf_src;
            a.nmf = nmf;
            a.dst_mf = reinterpret_cast<double2 *>(sg.tail_ptr());
            a.k = k_src;
            a.nk = nk;
            a.dst_k = reinterpret_cast<double *>(sg.tail_ptr() + mf_bytes);
        }
        const int work = std::max(std::max(a.rows * rowlen, a.nmf), a.nk);
        qlk::k_state_out<<<std::max(1, std::min((work + qlk::NT - 1) / qlk::NT, 512)), qlk::NT, 0, st>>>(a);
        QL_HIP(hipGetLastError());
        if (np > 1) QL_HIP(hipEventRecord(sg.ev[c % sg.n], st));
        return QL_OK;
    };
    auto copy = [&](int c) {
        std::memcpy(static_cast<char *>(lin) + (size_t)c * per * row_bytes, sg.host + sg.slot * (c % sg.n),
                    row_bytes * std::min(per, rows - c * per));
    };
    if (np <= 1) {
        QL_RC(issue(0));
        QL_HIP(hipStreamSynchronize(st));
        if (np) copy(0);
    } else {
        std::atomic<int> ready{0}, next{0};
        std::atomic<bool> stop{false};
        // per slot, one past the last piece copied out of it (nothing here takes
        // memory but the threads, which are done without where there is none: no
        // exception may leave a call)
        std::atomic<int> copied[OUT_SLOTS];
        for (auto &d : copied) d.store(0, std::memory_order_relaxed);
        // a worker takes the next piece, waits until it has arrived and copies it
        auto work = [&]() {
            for (int c; (c = next.fetch_add(1)) < np;) {
                while (ready.load(std::memory_order_acquire) <= c) {
                    if (stop.load()) return;
                    std::this_thread::yield();
                }
                copy(c);
                copied[c % sg.n].store(c + 1, std::memory_order_release);
            }
        };
        std::thread pool[OUT_SLOTS];
        int workers = 0, issued = 0;
        auto run = [&]() -> int {
            for (int c = 0; c < np; ++c) {
                // slots are filled again once they have been copied out
                while (issued < np && issued < c + sg.n) {
                    if (issued >= sg.n &&
                        copied[issued % sg.n].load(std::memory_order_acquire) != issued - sg.n + 1) {
                        if (issued > c) break;
                        std::this_thread::yield();
                        continue;
                    }
                    QL_RC(issue(issued));
                    ++issued;
                    if (c == 0 && np >= OUT_THREADED && issued == std::min(np, sg.n)) {
                        // the first pieces are on their way: start the workers
                        const unsigned cpus = std::max(1u, std::thread::hardware_concurrency());
                        try {
                            for (; workers < std::min<int>(std::min(np, OUT_SLOTS), cpus); ++workers)
                                pool[workers] = std::thread(work);
                        } catch (...) {  // no more threads: those there are, or none, do it
                        }
                    }
                }
                QL_HIP(hipEventSynchronize(sg.ev[c % sg.n]));
                if (!workers) {
                    copy(c);
                    copied[c % sg.n].store(c + 1, std::memory_order_release);
                } else {
                    ready.store(c + 1, std::memory_order_release);
                }
            }
            return QL_OK;
        };
        const int rc = run();
        if (rc != QL_OK) stop.store(true);
        for (int k = 0; k < workers; ++k) pool[k].join();
        if (rc != QL_OK) return rc;
    }
    if (nmf) std::memcpy(mf, sg.tail_ptr(), mf_bytes);
    if (nk) std::memcpy(k, sg.tail_ptr() + mf_bytes, k_bytes);
    return QL_OK;
}

}  // namespace qlh
