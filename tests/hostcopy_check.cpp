// Host check of HostCopy (fenice_amd/csrc/fvg_transfer.hip) where its helper threads cannot be started: the HIP calls it
// makes are defined here over host memory (the conversion kernels run at once, on the caller's thread), and
// pthread_create or the allocation of a thread's state fails from the k-th thread on. Every transfer must still move
// every value, on the threads that are there.
#include <dlfcn.h>
#include <hip/hip_runtime.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>
#include <vector>

#include "../fenice_amd/csrc/fvg_transfer.hpp"

static int g_threads = 0, g_started = 0;   // threads allowed, threads asked for
static bool g_no_memory = false;           // fail by the allocation instead of pthread_create
static thread_local bool g_in_copy = false;

void* operator new(size_t n) {
    if (g_in_copy && g_no_memory && g_started++ >= g_threads) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// the one that std::thread finds first
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
    using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Create next = (Create)dlsym(RTLD_NEXT, "pthread_create");
    if (g_in_copy && !g_no_memory && g_started++ >= g_threads) return EAGAIN;
    return next(t, a, f, x);
}

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
// the conversion kernels: (slot, n, planes, stride, c0, map), five components per cell
static bool g_up;
hipError_t hipLaunchKernel(const void*, dim3, dim3, void** a, size_t, hipStream_t) {
    double* slot = *(double**)a[0];
    const unsigned n = *(unsigned*)a[1], map = *(unsigned*)a[5];
    double* planes = *(double**)a[2];
    const long long stride = *(long long*)a[3], c0 = *(long long*)a[4];
    for (unsigned e = 0; e < n; ++e) {
        double& p = planes[(map >> 4 * (e % 5) & 15) * stride + c0 + e / 5];
        if (g_up) p = slot[e];
        else slot[e] = p;
    }
    return hipSuccess;
}
}

int main() {
    std::setvbuf(stdout, nullptr, _IONBF, 0);
    const long long n = 1000003;   // 40 MB: six lanes
    const unsigned map = fvg::plane_map(0, 1, 2, 3, 4);
    std::vector<double> U(5 * n), V(5 * n), planes(5 * n);
    for (long long k = 0; k < 5 * n; ++k) U[k] = (double)k;
    int bad = 0;
    for (int memory = 0; memory < 2; ++memory)
        for (int k = 0; k < 6; ++k) {
            g_no_memory = memory != 0;
            std::fill(planes.begin(), planes.end(), -1.0);
            std::fill(V.begin(), V.end(), -1.0);
            fvg::HostCopy copy;
            std::string what;
            hipError_t e[2];
            for (int down = 0; down < 2; ++down) {
                g_up = !down;
                g_threads = k;
                g_started = 0;
                g_in_copy = true;
                e[down] = down ? copy.to_host(0, nullptr, planes.data(), n, V.data(), n, 5, map, what)
                               : copy.to_device(0, nullptr, U.data(), n, 5, planes.data(), n, map, what);
                g_in_copy = false;
            }
            copy.release();
            const bool ok = e[0] == hipSuccess && e[1] == hipSuccess && U == V;
            bad += !ok;
            std::printf("%s after %d threads: %s\n", memory ? "no memory" : "no thread", k, ok ? "ok" : "WRONG");
        }
    return bad != 0;
}
