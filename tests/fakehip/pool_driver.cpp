// The library's buffer pool under host-pointer calls, and the device that the native
// server's thread works on, without a GPU: the HIP calls
// that librlgpu makes are defined here (device memory is host memory, kernels do
// nothing, copies are immediate) and checked (test infrastructure).
//
//   pool_driver SCENARIO
//
// Prints "ok" and exits 0, or prints what went wrong and exits 1.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "../../include/rlgpu.h"

namespace {

std::mutex g_mu;
std::map<void *, size_t> g_mem;      // device allocations
size_t g_held = 0, g_limit = SIZE_MAX;
std::set<void *> g_freed;
bool g_busy = false;                 // work recorded now does not end until it is cleared
std::atomic<int> g_stalls{0};        // waits for such work
std::atomic<int> g_locked_frees{0};  // frees during which the pool could not be used
std::atomic<bool> g_probe{false};
bool g_fail_launch = false;
std::atomic<int> g_wrong_device{0};  // work for a stream or memory of another device than the thread's
int g_want_device = -1;              // the device that allocations are to be on (-1: any)
thread_local int t_device = 0;
int g_copies = 0;                    // asynchronous copies that read or write host memory, not yet waited for
thread_local hipError_t g_last = hipSuccess;

hipError_t ret(hipError_t e) {
    if (e != hipSuccess && e != hipErrorNotReady) g_last = e;
    return e;
}

struct Event {
    bool pending = false;
};

// A call that takes and returns pooled buffers, from a thread of its own.
bool pool_is_usable() {
    auto done = std::make_shared<std::atomic<bool>>(false);
    std::thread([done] {
        double m[4] = {1, 2, 3, 4}, v[2] = {1, 1}, y[2];
        rlg_matvec_f64(2, 2, m, 2, 2, v, y);
        *done = true;
    }).detach();
    for (int i = 0; i < 200 && !*done; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    return *done;
}

}  // namespace

extern "C" {

hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = t_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 << 10;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipMalloc(void **p, size_t n) {
    if (g_want_device >= 0 && t_device != g_want_device) ++g_wrong_device;
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_held + n > g_limit) return ret(hipErrorOutOfMemory);
    *p = std::malloc(n);
    g_mem[*p] = n;
    g_held += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    if (g_probe.exchange(false) && !pool_is_usable()) ++g_locked_frees;
    std::lock_guard<std::mutex> lk(g_mu);
    g_copies = 0;  // waits for the device
    g_held -= g_mem.at(p);
    g_mem.erase(p);
    g_freed.insert(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(new int(t_device)); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { g_copies = 0; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { g_copies = 0; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = reinterpret_cast<hipEvent_t>(new Event()); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { reinterpret_cast<Event *>(e)->pending = g_busy; return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { return ret(reinterpret_cast<Event *>(e)->pending && g_busy ? hipErrorNotReady : hipSuccess); }
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (reinterpret_cast<Event *>(e)->pending && g_busy) ++g_stalls;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
    std::memcpy(d, s, n);
    if (k != hipMemcpyDeviceToDevice) ++g_copies;
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    for (size_t i = 0; i < h; ++i) std::memcpy(static_cast<char *>(d) + i * dp, static_cast<const char *>(s) + i * sp, w);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s) {
    if (t_device != *reinterpret_cast<int *>(s)) ++g_wrong_device;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
    return ret(g_fail_launch ? hipErrorInvalidConfiguration : hipSuccess);
}

}  // extern "C"

namespace {

constexpr size_t MB = 1 << 20;
std::vector<double> g_a(90 * MB / 8, 1.0), g_v(8192, 1.0), g_y(1 << 17);

int fail(const char *what, double v = 0) {
    std::printf("%s (%g)\n", what, v);
    return 1;
}
// A product with one operand of `mb` megabytes.
int product(size_t mb) {
    const size_t n = 1024, m = mb * MB / 8 / n;
    const int st = rlg_matvec_f64(m, n, g_a.data(), n, n, g_v.data(), g_y.data());
    if (st != RLG_OK) std::printf("product of %zu MB: %s\n", mb, rlg_last_error_message());
    return st;
}
// Host products of growing size, none of whose operands fits a buffer kept before.
int products(size_t from, size_t to) {
    for (size_t mb = from; mb <= to; ++mb)
        if (product(mb) != RLG_OK) return 1;
    return 0;
}
// Another user's pooled buffers (a permutation's), as large as the products'.
std::set<void *> others() {
    std::vector<size_t> p(1024);
    for (size_t i = 0; i < p.size(); ++i) p[i] = p.size() - 1 - i;
    std::vector<double> a(1024 * 1024), o(1024 * 1024);
    if (rlg_permute_rows_f64(p.size(), p.data(), 1024, 1024, a.data(), 1024, o.data(), 1024) != RLG_OK) std::abort();
    std::set<void *> kept;
    for (auto &e : g_mem) kept.insert(e.first);
    return kept;
}

// The kept operands are bounded, and giving them back takes nothing of others.
int bounded() {
    const std::set<void *> kept = others();
    size_t base = g_held;
    if (product(2) != RLG_OK || products(8, 64)) return 1;
    for (void *p : kept)
        if (!g_mem.count(p)) return fail("a buffer of another user was freed");
    if (g_held - base > (1024 + 64) * MB) return fail("megabytes held beyond the bound", (double)(g_held - base) / MB);
    return 0;
}
// Giving back waits for nobody's work and leaves the pool usable meanwhile.
int unblocked() {
    if (products(16, 40)) return 1;
    g_busy = true;
    others();
    for (size_t mb = 41; mb <= 64; ++mb) {
        g_probe = true;
        if (product(mb) != RLG_OK) return 1;
    }
    if (g_stalls) return fail("waits for unrelated work", g_stalls);
    if (g_locked_frees) return fail("frees with the pool locked", g_locked_frees);
    return 0;
}
// Kept operands are given back where memory is short: for a large operand of a
// host call and for the caller's own allocation.
int shortage() {
    if (products(32, 60)) return 1;
    g_limit = g_held + MB;
    if (product(80) != RLG_OK) return 1;
    g_limit = SIZE_MAX;
    if (products(32, 60)) return 1;
    g_limit = g_held + MB;
    void *p = nullptr;
    if (rlg_dev_alloc(100 * MB, &p) != RLG_OK) return fail("rlg_dev_alloc");
    if (hipGetLastError() != hipSuccess) return fail("an error that was dealt with is left behind");
    return rlg_dev_free(p);
}

// A call that fails leaves no copy from the caller's memory under way.
int drained() {
    rlg_mixed_opts o;
    rlg_mixed_opts_default(&o);
    o.factor_prec = 99;
    const size_t n = 256;
    if (rlg_solve_mixed_f64(n, g_a.data(), n, 1, g_v.data(), n, g_y.data(), n, &o, nullptr) != RLG_E_INVALID_ARG)
        return fail("an unknown precision was accepted");
    if (g_copies) return fail("copies under way after an invalid option", g_copies);
    g_fail_launch = true;
    if (rlg_gemm_f64(n, n, g_a.data(), n, n, n, g_a.data(), n, g_y.data(), n) == RLG_OK) return fail("launch");
    if (g_copies) return fail("copies under way after a failed product", g_copies);
    if (rlg_matvec_f64(n, n, g_a.data(), n, n, g_v.data(), g_y.data()) == RLG_OK) return fail("launch");
    if (g_copies) return fail("copies under way after a failed matrix-vector product", g_copies);
    g_fail_launch = false;
    const int st = product(4);
    return g_copies ? fail("copies under way after a call", g_copies) : st;
}

// The server's own thread stays on the device that the server was created on.
int server() {
    setenv("RLG_ENABLE_SERVER", "1", 1);
    if (rlg_set_device(1) != RLG_OK) return fail("rlg_set_device");
    rlg_server *s = nullptr;
    if (rlg_server_create(nullptr, &s) != RLG_OK) return fail(rlg_last_error_message());
    g_want_device = 1;
    for (int i = 0; i < 4; ++i) {
        rlg_request q{};
        rlg_result r{};
        int64_t t = 0;
        q.kind = i % 2 ? RLG_KIND_LU : RLG_KIND_CHOL;
        q.n = 150 + i;
        q.nrhs = 2;
        q.a = g_a.data();
        q.b = g_v.data();
        // (the kernels do nothing, so a request may well fail)
        if (rlg_server_submit(s, &q, &t) != RLG_OK || rlg_server_wait(s, t, &r) != RLG_OK) return fail("request");
        rlg_server_release(s, t);
    }
    rlg_server_destroy(s);
    return g_wrong_device ? fail("launches or allocations on another device", g_wrong_device) : 0;
}

}  // namespace

int main(int argc, char **argv) {
    const std::string s = argc > 1 ? argv[1] : "";
    const int st = s == "bounded" ? bounded() : s == "unblocked" ? unblocked() : s == "shortage" ? shortage()
                   : s == "drained" ? drained() : s == "server" ? server() : 2;
    if (st == 0) std::printf("ok\n");
    std::fflush(stdout);
    std::_Exit(st);
}
