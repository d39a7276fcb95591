// Uploads and downloads of a state: the array of cells on the host against structure-of-arrays planes on the device.
//
// What bounds it is the bus (57 GB/s pinned, each way) and the host's memory. The chunks of the array go through
// pinned slots that the conversion kernels read or write directly over the bus, so there is no device staging and no
// separate copy; host threads fill or drain the slots (one thread copies 12-30 GB/s, and 5-14 GB/s into pages that a
// caller has just allocated, so large arrays take several). Measured (up / down): 256^3 Taylor-Green, 671 MB,
// 18 / 15 ms (36 / 44 GB/s), 206 / 216 ms with the conversion on one host thread through a pageable vector; 2048^2
// Kelvin-Helmholtz, 134 MB, 3.9 / 4.3 ms against 42 / 43; 101 x 75 x 52, 15.8 MB, 0.5 / 0.5 ms against 2.4 / 4.4. A
// single chunk is latency: it waits for the stream itself, without an event (164 KB 19 / 20 us, 24-28 / 21-24 with one,
// 21-30 / 20-22 by pageable copies; 40 KB 16 / 16, 16-20 / 16-19, 14-15 / 13).
#include "fvg_transfer.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <thread>

namespace fvg {

namespace {

// n elements of an array of cells from cell c0 on, in element order: consecutive lanes take consecutive elements, two
// each, so that the bus side is coalesced (64 lanes: 1 KiB); the planes' side is NC runs of consecutive cells.
template <int NC>
__device__ __forceinline__ double* plane_of(double* planes, long long stride, unsigned map, long long c0, unsigned e) {
    const unsigned c = e / NC, q = (map >> 4 * (e - c * NC)) & 15u;
    return q == kNoPlane ? nullptr : planes + (long long)q * stride + c0 + c;
}
template <int NC>
__global__ __launch_bounds__(256) void k_cells_up(const double2* __restrict__ src, unsigned n, double* __restrict__ planes, long long stride,
                                                  long long c0, unsigned map) {
    const unsigned e = 2 * (blockIdx.x * 256 + threadIdx.x);
    if (e >= n) return;
    const double2 v = src[e / 2];   // the slot is padded to a multiple of two elements
    if (double* p = plane_of<NC>(planes, stride, map, c0, e)) *p = v.x;
    if (e + 1 < n)
        if (double* p = plane_of<NC>(planes, stride, map, c0, e + 1)) *p = v.y;
}
template <int NC>
__global__ __launch_bounds__(256) void k_cells_down(double2* __restrict__ dst, unsigned n, double* __restrict__ planes, long long stride,
                                                    long long c0, unsigned map) {
    const unsigned e = 2 * (blockIdx.x * 256 + threadIdx.x);
    if (e >= n) return;
    double2 v = {0.0, 0.0};
    if (const double* p = plane_of<NC>(planes, stride, map, c0, e)) v.x = *p;
    if (e + 1 < n)
        if (const double* p = plane_of<NC>(planes, stride, map, c0, e + 1)) v.y = *p;
    dst[e / 2] = v;
}

template <int NC>
void convert(hipStream_t s, bool up, double* slot, unsigned n, double* planes, long long stride, long long c0, unsigned map) {
    const dim3 g((n + 511) / 512), b(256);
    if (up) hipLaunchKernelGGL((k_cells_up<NC>), g, b, 0, s, (const double2*)slot, n, planes, stride, c0, map);
    else hipLaunchKernelGGL((k_cells_down<NC>), g, b, 0, s, (double2*)slot, n, planes, stride, c0, map);
}

}   // namespace

// Chunks j, j + nlanes, ... of the array through this lane's two slots.
hipError_t HostCopy::lane(int j, int nlanes, hipStream_t stream, double* host, long long ncells, int ncomp, double* planes,
                          long long stride, unsigned map, bool up, long long chunk) {
    const long long nchunks = (ncells + chunk - 1) / chunk;
    auto first = [&](long long c) { return c * chunk; };
    auto cells = [&](long long c) { return std::min(chunk, ncells - c * chunk); };
    auto launch = [&](long long c, int s) {
        const unsigned n = (unsigned)(cells(c) * ncomp);
        if (ncomp == 5) convert<5>(stream, up, slot[s], n, planes, stride, first(c), map);
        else if (ncomp == 4) convert<4>(stream, up, slot[s], n, planes, stride, first(c), map);
        else convert<3>(stream, up, slot[s], n, planes, stride, first(c), map);
        const hipError_t e = hipGetLastError();
        return e != hipSuccess || nchunks == 1 ? e : hipEventRecord(done[s], stream);
    };
    hipError_t e = hipSuccess;
    if (up) {
        int k = 0;
        for (long long c = j; c < nchunks && e == hipSuccess; c += nlanes, ++k) {
            const int s = kSlotsPerThread * j + k % kSlotsPerThread;
            if (k >= kSlotsPerThread) e = hipEventSynchronize(done[s]);   // its previous chunk has been read
            if (e != hipSuccess) break;
            std::memcpy(slot[s], host + first(c) * ncomp, (size_t)cells(c) * ncomp * sizeof(double));
            e = launch(c, s);
        }
    } else {
        for (int k = 0; k < kSlotsPerThread && e == hipSuccess; ++k)
            if (const long long c = j + (long long)k * nlanes; c < nchunks) e = launch(c, kSlotsPerThread * j + k);
        int k = 0;
        for (long long c = j; c < nchunks && e == hipSuccess; c += nlanes, ++k) {
            const int s = kSlotsPerThread * j + k % kSlotsPerThread;
            e = nchunks == 1 ? hipStreamSynchronize(stream) : hipEventSynchronize(done[s]);
            if (e != hipSuccess) break;
            std::memcpy(host + first(c) * ncomp, slot[s], (size_t)cells(c) * ncomp * sizeof(double));
            if (const long long next = c + (long long)kSlotsPerThread * nlanes; next < nchunks) e = launch(next, s);
        }
    }
    return e;
}

hipError_t HostCopy::run(int device, hipStream_t stream, double* host, long long ncells, int ncomp, double* planes, long long stride,
                         unsigned map, bool up, std::string& what) {
    if (ncells <= 0) return hipSuccess;
    // Chunks: a whole slot of a large array; a small array is cut in four so that the host's copy of one chunk runs
    // beside the conversion of the one before, down to 256 KiB, below which launches cost more than they hide.
    // Lanes: one per 6 MiB, since starting a thread takes about 30 us, in which one lane moves 1 MB.
    const size_t cell = (size_t)ncomp * sizeof(double), bytes = (size_t)ncells * cell;
    const size_t per = std::min(kSlotBytes, std::max(bytes / 4, size_t(256) << 10));
    const long long chunk = (long long)std::max<size_t>(1, per / cell);
    const long long nchunks = (ncells + chunk - 1) / chunk;
    int nlanes = (int)std::min<long long>({(long long)kThreads, nchunks, std::max<long long>(1, (long long)(bytes / (size_t(6) << 20)))});
    const int used = (int)std::min<long long>((long long)nlanes * kSlotsPerThread, nchunks);
    const size_t need = (std::min<size_t>(chunk, ncells) * cell + 15) / 16 * 16;
    hipError_t e = hipSuccess;
    for (int s = 0; s < nlanes * kSlotsPerThread && e == hipSuccess; ++s) {
        if (nlanes == 1 && s >= used) break;
        if (!done[s]) e = hipEventCreateWithFlags(&done[s], hipEventDisableTiming);
        if (e == hipSuccess && slot_bytes[s] < need) {
            if (slot[s]) hipHostFree(slot[s]);
            slot[s] = nullptr;
            slot_bytes[s] = 0;
            e = hipHostMalloc((void**)&slot[s], need);
            if (e == hipSuccess) slot_bytes[s] = need;
        }
    }
    if (e != hipSuccess) {
        what = "pinned staging of a host copy";
        return e;
    }
    hipError_t err[kThreads];
    std::thread th[kThreads];
    int started = 1;
    err[0] = hipSuccess;
    for (; started < nlanes; ++started) {
        const int j = started;
        err[j] = hipSuccess;
        try {
            th[j] = std::thread([&, j] {
                err[j] = hipSetDevice(device);
                if (err[j] == hipSuccess) err[j] = lane(j, nlanes, stream, host, ncells, ncomp, planes, stride, map, up, chunk);
            });
        } catch (const std::exception&) {   // no more threads, or no memory for one: this one takes the other lanes
            break;
        }
    }
    err[0] = lane(0, nlanes, stream, host, ncells, ncomp, planes, stride, map, up, chunk);
    for (int j = started; j < nlanes; ++j) err[j] = lane(j, nlanes, stream, host, ncells, ncomp, planes, stride, map, up, chunk);
    for (int j = 1; j < started; ++j) th[j].join();
    for (int j = 0; j < nlanes; ++j)
        if (err[j] != hipSuccess && e == hipSuccess) e = err[j];
    // also after a failed lane: no kernel may outlive the call
    const hipError_t es = nchunks == 1 && !up && e == hipSuccess ? hipSuccess : hipStreamSynchronize(stream);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) what = "host copy of a state";
    return e;
}

hipError_t HostCopy::to_device(int device, hipStream_t stream, const double* src, long long ncells, int ncomp, double* planes,
                               long long stride, unsigned map, std::string& what) {
    return run(device, stream, const_cast<double*>(src), ncells, ncomp, planes, stride, map, true, what);
}
hipError_t HostCopy::to_host(int device, hipStream_t stream, const double* planes, long long stride, double* dst, long long ncells,
                             int ncomp, unsigned map, std::string& what) {
    return run(device, stream, dst, ncells, ncomp, const_cast<double*>(planes), stride, map, false, what);
}

void HostCopy::release() {
    for (int s = 0; s < kSlots; ++s) {
        if (done[s]) hipEventDestroy(done[s]);
        if (slot[s]) hipHostFree(slot[s]);
        done[s] = nullptr;
        slot[s] = nullptr;
        slot_bytes[s] = 0;
    }
}

}   // namespace fvg
