// Runs the library's host code without a GPU: this program defines the HIP functions that the
// library calls, and the loader binds the library to them.  Device memory is a range of addresses
// that nothing may touch, allocations are counted and may be refused, launches are printed with
// the kernel's name and grid.  Copies to the host deliver zeros.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "gemm.hpp"
#include "moao_hip.h"
#include "recon.hpp"
#include "stages.hpp"

namespace {

std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> k;
    return k;
}
std::mutex mu;
bool show = true;          // print launches
std::set<std::string> launched;
size_t limit = SIZE_MAX;   // bytes a single stream-ordered allocation may ask for
struct Pool {
    size_t live = 0, peak = 0;
    std::map<void*, size_t> blocks;
};
Pool pool, heap;           // stream-ordered, hipMalloc
char* next_address = reinterpret_cast<char*>(1L << 44);

hipError_t take(Pool& p, void** ptr, size_t bytes) {
    std::lock_guard<std::mutex> g(mu);
    *ptr = next_address;
    next_address += (bytes + 4095) & ~size_t(4095);
    p.blocks[*ptr] = bytes;
    p.live += bytes;
    p.peak = std::max(p.peak, p.live);
    return hipSuccess;
}
hipError_t give(Pool& p, void* ptr) {
    std::lock_guard<std::mutex> g(mu);
    auto it = p.blocks.find(ptr);
    if (ptr && it == p.blocks.end()) {
        std::printf("free of an unknown block\n");
        std::exit(3);
    }
    if (ptr) {
        p.live -= it->second;
        p.blocks.erase(it);
    }
    return hipSuccess;
}

// bytes of the C++ heap in use by what runs between the two readings of heap_peak
std::atomic<long> cpp_live{0}, cpp_peak{0};

}  // namespace

void* operator new(size_t n) {
    void* p = std::malloc(n + 16);
    if (!p) throw std::bad_alloc();
    *static_cast<size_t*>(p) = n;
    const long live = cpp_live += (long)n;
    long peak = cpp_peak;
    while (live > peak && !cpp_peak.compare_exchange_weak(peak, live)) {
    }
    return static_cast<char*>(p) + 16;
}
void operator delete(void* q) noexcept {
    if (!q) return;
    char* p = static_cast<char*>(q) - 16;
    cpp_live -= (long)*reinterpret_cast<size_t*>(p);
    std::free(p);
}
void operator delete(void* q, size_t) noexcept { operator delete(q); }

extern "C" {

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
    int rc = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &rc);
    std::string s = rc == 0 ? d : name;
    std::free(d);
    // "void moao::(anonymous namespace)::kernel<args>(parameters)" -> "kernel<args>"
    if (s.compare(0, 5, "void ") == 0) s.erase(0, 5);
    const std::string ns = "moao::(anonymous namespace)::";
    if (s.compare(0, ns.size(), ns) == 0) s.erase(0, ns.size());
    int depth = 0;
    for (size_t k = 0; k < s.size(); ++k) {
        if (s[k] == '<') ++depth;
        if (s[k] == '>') --depth;
        if (s[k] == '(' && depth == 0) {
            s.resize(k);
            break;
        }
    }
    kernels()[host] = s;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t);
static thread_local dim3 cfg_grid, cfg_block;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
    cfg_grid = grid;
    cfg_block = block;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
    *grid = cfg_grid;
    *block = cfg_block;
    *shared = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t) {
    std::lock_guard<std::mutex> l(mu);
    launched.insert(kernels()[f]);
    if (!g.x || !g.y || !g.z || g.y > 65535 || g.z > 65535 || b.x * b.y * b.z > 1024) {
        std::printf("impossible launch of %s\n", kernels()[f].c_str());
        std::exit(3);
    }
    if (show) std::printf("launch %s %u %u %u\n", kernels()[f].c_str(), g.x, g.y, g.z);
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return take(heap, p, n); }
hipError_t hipFree(void* p) { return give(heap, p); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) {
    const bool ok = n <= limit;
    if (show) std::printf("async %zu %s\n", n, ok ? "given" : "refused");
    return ok ? take(pool, p, n) : hipErrorOutOfMemory;
}
hipError_t hipFreeAsync(void* p, hipStream_t) { return give(pool, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void*, size_t n, hipMemcpyKind k) {
    if (k == hipMemcpyDeviceToHost) std::memset(d, 0, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind,
                            hipStream_t) {
    return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = reinterpret_cast<void*>(1L << 43);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    static std::atomic<long> k{1};
    *s = reinterpret_cast<hipStream_t>(k++ << 8);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) {
    *c = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = size_t(256) << 30;
    return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) {
    *p = nullptr;
    return hipSuccess;
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }

}  // extern "C"

namespace {

double* at(long k) { return reinterpret_cast<double*>((1L << 42) + (k << 36)); }

// <f64|f32> transb M N K lda ldb
int run_gemm(char** a) {
    const int tb = std::atoi(a[1]), M = std::atoi(a[2]), N = std::atoi(a[3]), K = std::atoi(a[4]);
    const long lda = std::atol(a[5]), ldb = std::atol(a[6]);
    if (std::string(a[0]) == "f64")
        return moao_hip_dgemm_dev(tb, M, N, K, 1.0, at(1), lda, at(2), ldb, 1.0, at(3), M, nullptr);
    return moao_hip_sgemm_dev(tb, M, N, K, 1.0f, (float*)at(1), lda, (float*)at(2), ldb, 1.0f,
                              (float*)at(3), M, nullptr);
}

// n m <1 FP32 | 2 BF16>: a mixed solve in the least and in the best workspace; launches of both
int run_mixed(char** a) {
    const long n = std::atol(a[0]), m = std::atol(a[1]);
    const int mode = std::atoi(a[2]);
    const size_t least = moao::mixed_workspace_bytes(n, m, nullptr, mode);
    std::printf("least %zu spare %zu\n", least, moao::mixed_spare_bytes(n, m));
    for (const size_t ws : {least, least + moao::mixed_spare_bytes(n, m)}) {
        std::printf("workspace %zu\n", ws);
        if (int rc = moao::reconstructor_mixed_dev(n, m, at(1), n, at(2), m, nullptr, mode, 1e-11, 5,
                                                   nullptr, nullptr, at(3), ws, nullptr))
            return rc;
    }
    return moao_hip_reconstructor_mixed_dev(n, m, at(1), n, at(2), m, nullptr, mode, 1e-11, 5,
                                            nullptr, nullptr, nullptr);
}

// sys atm type [field index value]...: matcov of a whole matrix, with values of the system replaced
int run_matcov(char** a, int n) {
    moao_tomo* t = nullptr;
    if (int rc = moao_tomo_create(a[0], a[1], &t)) return rc;
    moao_tomo_set_target(t, 0);
    moao_tomo_view v;
    moao_tomo_get_view(t, &v);
    const int type = std::atoi(a[2]);
    for (int k = 3; k + 2 < n; k += 3) {
        const std::string f = a[k];
        const double* p = f == "X" ? v.X : f == "Y" ? v.Y : f == "u" ? v.u : f == "v" ? v.v
                        : f == "sspSizeL" ? v.sspSizeL : f == "L0" ? v.L0 : nullptr;
        const_cast<double*>(p)[std::atol(a[k + 1])] = std::atof(a[k + 2]);
    }
    const int cols = (int)moao_tomo_nmeas(t), rows = type == 1 ? cols : (int)moao_tomo_nmeasts(t);
    const int rc = moao_hip_matcov_tile_dev(at(1), rows, cols, 0, 0, rows, &v, type, nullptr);
    moao_tomo_destroy(t);
    return rc;
}

// sys atm mode slots budget requests: what the requests were said to hold and what they took
int run_serve(char** a) {
    show = false;
    moao_serve_config cfg{std::atoi(a[3]), std::strtoull(a[4], nullptr, 10), 0};
    moao_server* srv = nullptr;
    if (int rc = moao_serve_create(&cfg, &srv)) return rc;
    moao_serve_request q{};
    q.sys_file = a[0];
    q.atm_file = a[1];
    q.mode = std::atoi(a[2]);
    std::vector<long> tickets(std::atoi(a[5]));
    for (long& t : tickets)
        if (int rc = moao_serve_submit(srv, &q, &t)) return rc;
    for (long t : tickets) {
        moao_serve_result r{};
        const int rc = moao_serve_wait(srv, t, &r);
        std::printf("request status %d n %ld m %ld footprint %zu\n", rc, r.n, r.m, r.footprint);
    }
    moao_serve_counters c{};
    moao_serve_stats(srv, &c);
    std::printf("peak %zu taken %zu left %zu kept %zu\n", c.peak_bytes, pool.peak, pool.live,
                heap.live);
    for (auto& k : launched) std::printf("launched %s\n", k.c_str());
    moao_serve_destroy(srv);
    return 0;
}

// np N <0 in order | 1 shuffled>: the plan of a PSF whose index lists every pair of np x np actuators
int run_create(char** a) {
    const long np = std::atol(a[0]), N = std::atol(a[1]), nact = np * np, ncov = 2 * np - 1;
    std::vector<long> idx(nact * nact);
    for (long i = 0; i < nact; ++i)
        for (long j = 0; j < nact; ++j)
            idx[i * nact + j] = (i / np - j / np + np - 1) * ncov + i % np - j % np + np;
    if (std::atoi(a[2])) {
        unsigned long x = 88172645463325252ul;
        for (size_t k = idx.size() - 1; k > 0; --k) {
            x ^= x << 13, x ^= x >> 7, x ^= x << 17;
            std::swap(idx[k], idx[x % (k + 1)]);
        }
    }
    const std::vector<double> w(N * N, 1.0);
    cpp_peak = cpp_live.load();
    const long before = cpp_live;
    const auto t = std::chrono::steady_clock::now();
    moao_isample* S = nullptr;
    const int rc = moao_hip_intersample_create(idx.size(), np, N, idx.data(), w.data(), w.data(), 1, &S);
    const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count();
    std::printf("plan entries %zu heap %ld device %zu us %.0f\n", idx.size(), cpp_peak - before,
                heap.live, s * 1e6);
    moao_hip_intersample_destroy(S);
    return rc;
}

}  // namespace

int main(int argc, char** argv) {
    const std::string cmd = argc > 1 ? argv[1] : "";
    int rc = 2;
    if (const char* l = std::getenv("ASYNC_LIMIT")) limit = std::strtoull(l, nullptr, 10);
    if (cmd == "gemm" && argc == 9) rc = run_gemm(argv + 2);
    if (cmd == "mixed" && argc == 5) rc = run_mixed(argv + 2);
    if (cmd == "matcov" && argc >= 5) rc = run_matcov(argv + 2, argc - 2);
    if (cmd == "plan" && argc == 5) rc = run_create(argv + 2);
    if (cmd == "serve" && argc == 8) rc = run_serve(argv + 2);
    std::printf("rc %d\n", rc);
    return rc == 2;
}
