// hip_on_host.cpp -- the HIP runtime calls libql_dns.so makes, on host memory,
// for tests of what the host code does when a call fails.  Preloaded
// (LD_PRELOAD) ahead of the real runtime; needs no GPU.
//
// Allocations are tracked and filled with a pattern; any of them, or any
// operator new, can be made to fail once, and device memory can be limited.
// A failed call leaves its error for hipGetLastError until that is read, as
// the runtime does.  hipMemset runs on the null stream, which the library's
// non-blocking streams do not wait for: it is held back until the null stream
// is waited for, and a copy or launch on another stream before that is counted
// as a race.  Copies are made, and their device ranges checked, at once.
// Kernels do nothing, except k_state_out, which copies.
#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace {

constexpr int OK = 0, OUT_OF_MEMORY = 2, INVALID = 1;

struct Fill {
    char *p;
    size_t n;
    int v;
};
struct World {
    std::recursive_mutex mu;
    std::map<char *, size_t> dev, host;  // live allocations
    std::map<const void *, std::string> kernels;
    std::vector<Fill> held;  // hipMemset on the null stream, not yet run
    size_t limit = SIZE_MAX, live = 0;
    long fail_malloc = 0, fail_host = 0;  // 1: the next one fails, 2: the one after it, ...
    long races = 0, bad = 0, null_waits = 0, mallocs = 0;
    int last = OK;
    bool capturing = false;
    std::vector<char> symbol;
};
World &w()
{
    static World *x = new World;
    return *x;
}
thread_local long fail_new = 0;

int err(int e)
{
    if (e != OK) w().last = e;
    return e;
}
void run_held()
{
    for (const Fill &f : w().held) std::memset(f.p, f.v, f.n);
    w().held.clear();
}
// whether [p, p + n) lies in one live device allocation
bool on_device(const void *p, size_t n)
{
    char *c = (char *)p;
    auto it = w().dev.upper_bound(c);
    if (it == w().dev.begin()) return false;
    --it;
    return c >= it->first && c + n <= it->first + it->second;
}
void touch(const void *stream)
{
    if (stream && !w().held.empty()) ++w().races;
}
// kind: 1 host to device, 2 device to host, 3 device to device
bool ranges_ok(void *d, const void *s, size_t n, int kind)
{
    const bool ok = d && s && (kind == 2 || on_device(d, n)) && (kind == 1 || on_device(s, n));
    if (!ok) ++w().bad;
    return ok;
}
typedef std::lock_guard<std::recursive_mutex> Lock;

struct StateOut {  // qlk::StateOut
    const double *u;
    int rows, rowlen, rowstride;
    double *dst;
    const double *mf;
    int nmf;
    double *dst_mf;
    const double *k;
    int nk;
    double *dst_k;
};
void state_out(const StateOut &a)
{
    for (int r = 0; r < a.rows; ++r)
        std::memcpy(a.dst + (size_t)2 * r * a.rowlen, a.u + (size_t)2 * r * a.rowstride, 16 * (size_t)a.rowlen);
    if (a.nmf) std::memcpy(a.dst_mf, a.mf, 16 * (size_t)a.nmf);
    if (a.nk) std::memcpy(a.dst_k, a.k, 8 * (size_t)a.nk);
}
int launch(const void *f, void **args, void *stream)
{
    Lock l(w().mu);
    touch(stream);
    if (w().capturing) return OK;
    const std::string &name = w().kernels[f];
    if (name.find("k_state_out") != std::string::npos) state_out(*(const StateOut *)args[0]);
    return OK;
}

struct dim3_t {
    unsigned x, y, z;
};
struct Call {
    dim3_t g, b;
    size_t shared;
    void *stream;
};
thread_local std::vector<Call> pushed;

}  // namespace

// what the tests set and read
extern "C" {
void hoh_fail_malloc(long k) { w().fail_malloc = k; }
void hoh_fail_host(long k) { w().fail_host = k; }
void hoh_fail_new(long k) { fail_new = k; }
void hoh_limit(size_t n) { w().limit = n; }
long hoh_races(void) { return w().races; }
long hoh_bad(void) { return w().bad; }
long hoh_null_waits(void) { return w().null_waits; }
long hoh_mallocs(void) { return w().mallocs; }
size_t hoh_live(void) { return w().live; }
long hoh_host_live(void) { return (long)w().host.size(); }
// the sizes of the live device allocations, in order; returns how many
long hoh_sizes(size_t *out, long n)
{
    std::vector<size_t> s;
    for (auto &e : w().dev) s.push_back(e.second);
    std::sort(s.begin(), s.end());
    for (size_t k = 0; k < s.size() && (long)k < n; ++k) out[k] = s[k];
    return (long)s.size();
}
}

void *operator new(size_t n)
{
    if (fail_new > 0 && --fail_new == 0) throw std::bad_alloc();
    void *p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {

void **__hipRegisterFatBinary(const void *)
{
    static void *h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *)
{
    w().kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t shared, void *stream)
{
    pushed.push_back(Call{g, b, shared, stream});
    return OK;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *shared, void **stream)
{
    const Call c = pushed.back();
    pushed.pop_back();
    *g = c.g, *b = c.b, *shared = c.shared, *stream = c.stream;
    return OK;
}
int hipLaunchKernel(const void *f, dim3_t, dim3_t, void **args, size_t, void *stream) { return launch(f, args, stream); }
int hipExtLaunchKernel(const void *f, dim3_t, dim3_t, void **args, size_t, void *stream, void *, void *, int)
{
    return launch(f, args, stream);
}

int hipGetLastError(void)
{
    Lock l(w().mu);
    const int e = w().last;
    w().last = OK;
    return e;
}
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : e ? "error" : "no error"; }
int hipGetDeviceCount(int *n)
{
    *n = 1;
    return OK;
}
int hipSetDevice(int) { return OK; }

int hipMalloc(void **p, size_t n)
{
    Lock l(w().mu);
    ++w().mallocs;
    *p = nullptr;
    if ((w().fail_malloc > 0 && --w().fail_malloc == 0) || n > w().limit - std::min(w().limit, w().live))
        return err(OUT_OF_MEMORY);
    char *c = (char *)std::malloc(n);
    if (!c) return err(OUT_OF_MEMORY);
    std::memset(c, 0xA5, n);
    w().dev[c] = n;
    w().live += n;
    *p = c;
    return OK;
}
int hipFree(void *p)
{
    Lock l(w().mu);
    run_held();  // waits for the device
    if (!p) return OK;
    auto it = w().dev.find((char *)p);
    if (it == w().dev.end()) {
        ++w().bad;
        return err(INVALID);
    }
    w().live -= it->second;
    w().dev.erase(it);
    std::free(p);
    return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned)
{
    Lock l(w().mu);
    *p = nullptr;
    if (w().fail_host > 0 && --w().fail_host == 0) return err(OUT_OF_MEMORY);
    *p = std::malloc(n);
    w().host[(char *)*p] = n;
    return OK;
}
int hipHostFree(void *p)
{
    Lock l(w().mu);
    if (w().host.erase((char *)p) != 1) ++w().bad;
    std::free(p);
    return OK;
}
int hipMemset(void *p, int v, size_t n)
{
    Lock l(w().mu);
    if (!on_device(p, n)) {
        ++w().bad;
        return err(INVALID);
    }
    w().held.push_back(Fill{(char *)p, n, v});
    return OK;
}
int hipMemsetAsync(void *p, int v, size_t n, void *stream)
{
    Lock l(w().mu);
    touch(stream);
    if (!on_device(p, n)) {
        ++w().bad;
        return err(INVALID);
    }
    std::memset(p, v, n);
    return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind)
{
    Lock l(w().mu);
    run_held();
    if (!ranges_ok(d, s, n, kind)) return err(INVALID);
    std::memcpy(d, s, n);
    return OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream)
{
    Lock l(w().mu);
    touch(stream);
    if (!ranges_ok(d, s, n, kind)) return err(INVALID);
    std::memcpy(d, s, n);
    return OK;
}
int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t width, size_t rows, int kind, void *stream)
{
    Lock l(w().mu);
    touch(stream);
    for (size_t r = 0; r < rows; ++r) {
        if (!ranges_ok((char *)d + r * dp, (const char *)s + r * sp, width, kind)) return err(INVALID);
        std::memcpy((char *)d + r * dp, (const char *)s + r * sp, width);
    }
    return OK;
}
int hipGetSymbolAddress(void **p, const void *)
{
    w().symbol.resize((size_t)8 << 20);
    *p = w().symbol.data();
    return OK;
}

int hipStreamCreateWithFlags(void **s, unsigned)
{
    *s = std::malloc(1);
    return OK;
}
int hipStreamDestroy(void *s)
{
    std::free(s);
    return OK;
}
int hipStreamSynchronize(void *s)
{
    Lock l(w().mu);
    if (!s) {
        ++w().null_waits;
        run_held();
    }
    return OK;
}
int hipStreamWaitEvent(void *, void *, unsigned) { return OK; }
int hipEventCreate(void **e)
{
    *e = std::malloc(1);
    return OK;
}
int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void *e)
{
    std::free(e);
    return OK;
}
int hipEventRecord(void *, void *) { return OK; }
int hipEventSynchronize(void *) { return OK; }
int hipEventElapsedTime(float *ms, void *, void *)
{
    *ms = 1.0f;
    return OK;
}
int hipStreamBeginCapture(void *, int)
{
    w().capturing = true;
    return OK;
}
int hipStreamEndCapture(void *, void **g)
{
    w().capturing = false;
    *g = std::malloc(1);
    return OK;
}
int hipGraphDestroy(void *g)
{
    std::free(g);
    return OK;
}
int hipGraphInstantiate(void **x, void *, void **, char *, size_t)
{
    *x = std::malloc(1);
    return OK;
}
int hipGraphExecDestroy(void *x)
{
    std::free(x);
    return OK;
}
int hipGraphLaunch(void *, void *) { return OK; }

}  // extern "C"
