// Host array of cells (ncomp doubles per cell) <-> structure-of-arrays planes on the device (fvg_transfer.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <string>

namespace fvg {

// The plane that holds each host component, 4 bits each from component 0; kNoPlane: none (skipped on the way up,
// written as +0 on the way down).
constexpr unsigned kNoPlane = 15;
constexpr unsigned plane_map(unsigned a, unsigned b, unsigned c, unsigned d = kNoPlane, unsigned e = kNoPlane) {
    return a | b << 4 | c << 8 | d << 12 | e << 16;
}

// Pinned staging slots of one context, allocated at its first transfers and kept until release(): at most kSlots of
// kSlotBytes. Not thread-safe, like the context it belongs to.
struct HostCopy {
    static constexpr int kThreads = 6, kSlotsPerThread = 2, kSlots = kThreads * kSlotsPerThread;
    static constexpr size_t kSlotBytes = size_t(2) << 20;
    double* slot[kSlots] = {};
    size_t slot_bytes[kSlots] = {};
    hipEvent_t done[kSlots] = {};

    // ncells cells of ncomp doubles into / out of planes (plane q at planes + q * stride); the copy is complete on
    // return, after what was enqueued on the stream before it. ncomp 3, 4 or 5. Returns hipSuccess, or the error with
    // its place in what.
    hipError_t to_device(int device, hipStream_t stream, const double* src, long long ncells, int ncomp, double* planes, long long stride,
                         unsigned map, std::string& what);
    hipError_t to_host(int device, hipStream_t stream, const double* planes, long long stride, double* dst, long long ncells, int ncomp,
                       unsigned map, std::string& what);
    void release();

private:
    hipError_t run(int device, hipStream_t stream, double* host, long long ncells, int ncomp, double* planes, long long stride,
                   unsigned map, bool up, std::string& what);
    hipError_t lane(int j, int nlanes, hipStream_t stream, double* host, long long ncells, int ncomp, double* planes, long long stride,
                    unsigned map, bool up, long long chunk);
};

}   // namespace fvg
