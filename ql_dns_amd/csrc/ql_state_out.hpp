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
// as long as half a piece's copy (a state of 89 MB 2.2 ms; eight pieces of 1 MiB 2.8,
// of 512 KiB 4.0, sixteen of 512 KiB 3.0)
constexpr size_t OUT_SLOT = (size_t)2 << 20;
constexpr int OUT_SLOTS = 8, OUT_THREADED = 3;

// Pinned memory for results on their way: lent to one download at a time and kept
// for the next one of any handle, since new pinned pages cost more than a download
// where they are first touched.  First state of a handle, us, with memory of its
// own -> lent (pageable copies): 36x60x64 1350 -> 200 (1370), 64x64x128 1740 -> 550
// (2840), 64x128x128 2290 -> 1030 (1850), 128x128x256 3840 -> 2520 (8900).  At most
// PINNED_KEPT buffers wait here, and with the last handle they go.  Two sizes:
// records and small states take the small one.
constexpr int PINNED_KEPT = 4;
constexpr size_t PINNED_SMALL = (size_t)512 << 10, PINNED_LARGE = OUT_SLOT * OUT_SLOTS + ((size_t)1 << 20);

struct PinnedPool {
    struct Buffer {
        char *host = nullptr;
        size_t size = 0;
    };
    std::mutex mu;
    int handles = 0, kept = 0;
    Buffer buf[PINNED_KEPT];

    void open()
    {
        std::lock_guard<std::mutex> lock(mu);
        ++handles;
    }
    void close()
    {
        std::lock_guard<std::mutex> lock(mu);
        if (--handles > 0) return;
        for (; kept > 0; --kept) (void)hipHostFree(buf[kept - 1].host);
    }
    // the smallest kept buffer of at least size bytes, or a new one (host null:
    // none can be had)
    Buffer take(size_t size)
    {
        size = size <= PINNED_SMALL ? PINNED_SMALL : std::max(size, PINNED_LARGE);
        {
            std::lock_guard<std::mutex> lock(mu);
            int best = -1;
            for (int k = 0; k < kept; ++k)
                if (buf[k].size >= size && (best < 0 || buf[k].size < buf[best].size)) best = k;
            if (best >= 0) {
                const Buffer b = buf[best];
                buf[best] = buf[--kept];
                return b;
            }
        }
        Buffer b;
        b.size = size;
        if (hipHostMalloc((void **)&b.host, size, hipHostMallocCoherent | hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            b.host = nullptr;
        }
        return b;
    }
    void give(const Buffer &b)
    {
        if (!b.host) return;
        {
            std::lock_guard<std::mutex> lock(mu);
            if (kept < PINNED_KEPT && handles > 0 && b.size <= PINNED_LARGE) {
                buf[kept++] = b;
                return;
            }
        }
        (void)hipHostFree(b.host);
    }
};
// one per process, never destroyed: handles may be released while it ends
inline PinnedPool &pinned_pool()
{
    static PinnedPool *const p = new PinnedPool;
    return *p;
}

// One handle's part in it
struct Staging {
    std::mutex mu;  // calls of several threads on one handle take turns
    hipEvent_t ev[OUT_SLOTS] = {};  // with the first result of several pieces
    Staging() { pinned_pool().open(); }
    ~Staging()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        pinned_pool().close();
    }
};

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
    const int per = rows ? (int)std::min<size_t>(OUT_SLOT / row_bytes, rows) : 0;
    const int np = rows ? (rows + per - 1) / per : 0;  // pieces
    const int n = std::max(1, std::min(np, OUT_SLOTS));  // slots
    const size_t slot = (per * row_bytes + 255) / 256 * 256;
    std::lock_guard<std::mutex> lock(sg.mu);
    for (int k = 0; np > 1 && k < n; ++k)
        if (!sg.ev[k]) QL_HIP(hipEventCreateWithFlags(&sg.ev[k], hipEventDisableTiming));
    // the slots, then everything but the fluctuations
    struct Lent {
        PinnedPool::Buffer b;
        hipStream_t st;
        bool whole = false;  // nothing queued writes it any more
        ~Lent()
        {
            if (!whole) (void)hipStreamSynchronize(st);
            pinned_pool().give(b);
        }
    } lent{pinned_pool().take(slot * n + mf_bytes + k_bytes), st};
    char *const host = lent.b.host, *const tail = host + slot * n;
    if (!host) {
        lent.whole = true;
        if (rows)
            QL_HIP(hipMemcpy2DAsync(lin, row_bytes, u, sizeof(double2) * rowstride, row_bytes, rows,
                                    hipMemcpyDeviceToHost, st));
        if (nmf) QL_HIP(hipMemcpyAsync(mf, mf_src, mf_bytes, hipMemcpyDeviceToHost, st));
        if (nk) QL_HIP(hipMemcpyAsync(k, k_src, k_bytes, hipMemcpyDeviceToHost, st));
        QL_HIP(hipStreamSynchronize(st));
        return QL_OK;
    }
    auto issue = [&](int c) -> int {
        qlk::StateOut a{};
        a.u = u + (size_t)c * per * rowstride;
        a.rows = rows ? std::min(per, rows - c * per) : 0;
        a.rowlen = rowlen;
        a.rowstride = rowstride;
        a.dst = reinterpret_cast<double2 *>(host + slot * (c % n));
        if (c == 0) {
            a.mf = mf_src;
            a.nmf = nmf;
            a.dst_mf = reinterpret_cast<double2 *>(tail);
            a.k = k_src;
            a.nk = nk;
            a.dst_k = reinterpret_cast<double *>(tail + mf_bytes);
        }
        const int work = std::max(std::max(a.rows * rowlen, a.nmf), a.nk);
        qlk::k_state_out<<<std::max(1, std::min((work + qlk::NT - 1) / qlk::NT, 512)), qlk::NT, 0, st>>>(a);
        QL_HIP(hipGetLastError());
        if (np > 1) QL_HIP(hipEventRecord(sg.ev[c % n], st));
        return QL_OK;
    };
    auto copy = [&](int c) {
        std::memcpy(static_cast<char *>(lin) + (size_t)c * per * row_bytes, host + slot * (c % n),
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
                copied[c % n].store(c + 1, std::memory_order_release);
            }
        };
        std::thread pool[OUT_SLOTS];
        int workers = 0, issued = 0;
        auto run = [&]() -> int {
            for (int c = 0; c < np; ++c) {
                // slots are filled again once they have been copied out
                while (issued < np && issued < c + n) {
                    if (issued >= n &&
                        copied[issued % n].load(std::memory_order_acquire) != issued - n + 1) {
                        if (issued > c) break;
                        std::this_thread::yield();
                        continue;
                    }
                    QL_RC(issue(issued));
                    ++issued;
                    if (c == 0 && np >= OUT_THREADED && issued == std::min(np, n)) {
                        // the first pieces are on their way: start the workers
                        const unsigned cpus = std::max(1u, std::thread::hardware_concurrency());
                        try {
                            for (; workers < std::min<int>(std::min(np, OUT_SLOTS), cpus); ++workers)
                                pool[workers] = std::thread(work);
                        } catch (...) {  // no more threads: those there are, or none, do it
                        }
                    }
                }
                QL_HIP(hipEventSynchronize(sg.ev[c % n]));
                if (!workers) {
                    copy(c);
                    copied[c % n].store(c + 1, std::memory_order_release);
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
    lent.whole = true;
    if (nmf) std::memcpy(mf, tail, mf_bytes);
    if (nk) std::memcpy(k, tail + mf_bytes, k_bytes);
    return QL_OK;
}

}  // namespace qlh
