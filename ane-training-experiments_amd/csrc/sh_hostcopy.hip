// sh_hostcopy.hip — the large copies declared in sh_hostcopy.hpp.
#include "sh_hostcopy.hpp"

#include <stdint.h>

#include <algorithm>
#include <exception>
#include <thread>

#include "sh_copypool.hpp"

namespace sh {
namespace {

// Smaller copies take the runtime's own path. Into warm pages, called every 2 ms (the helpers asleep):
// 1 MiB 63 us by the runtime and 80 through the ring, 2 MiB 122 and 129, 3 MiB 185 and 131, 32 MiB
// 1878 and 707; into fresh pages 2 MiB 480 and 362. (The other way the runtime is as fast up to 16
// MiB: 2 MiB in 80 us against 201 through the ring.)
constexpr size_t kMin = 2u << 20;
constexpr int kOutBlocks = 128, kOutThreads = 256;
constexpr size_t kSlot = 2u << 20;
constexpr int kSlots = 4;
constexpr int kMaxHelpers = 5;

// n16 16-byte words to pinned host memory: a launch starts sooner than a transfer of the copy
// engines, whose first use by a process costs about 1.5 ms.
__global__ __launch_bounds__(kOutThreads) void k_copy_out(const uint4 *src, uint4 *dst, size_t n16) {
    for (size_t i = (size_t)blockIdx.x * kOutThreads + threadIdx.x; i < n16; i += (size_t)kOutBlocks * kOutThreads)
        dst[i] = src[i];
}

}  // namespace

struct HostCopier::State {
    uint8_t *ring = nullptr;
    hipEvent_t ev[kSlots] = {};
    CopyPool pool{std::max(1, std::min(kMaxHelpers, (int)std::thread::hardware_concurrency() / 2 - 1))};
};

bool HostCopier::ready() {
    if (st_ || refused_) return st_ != nullptr;
    try {
        st_ = new State;
    } catch (const std::exception &) {
        refused_ = true;
        return false;
    }
    bool ok = hipHostMalloc((void **)&st_->ring, kSlots * kSlot, hipHostMallocDefault) == hipSuccess;
    for (int i = 0; ok && i < kSlots; i++)
        ok = hipEventCreateWithFlags(&st_->ev[i], hipEventDisableTiming) == hipSuccess;
    if (ok) return true;
    (void)hipGetLastError();
    release();
    refused_ = true;
    return false;
}

void HostCopier::release() {
    if (!st_) return;
    st_->pool.finish();
    for (hipEvent_t e : st_->ev)
        if (e) (void)hipEventDestroy(e);
    if (st_->ring) (void)hipHostFree(st_->ring);
    delete st_;
    st_ = nullptr;
}

HostCopier::Prefault::Prefault(HostCopier &c, void *dst, size_t n) : c_(c) {
    if (n >= kMin && c.ready()) c.st_->pool.start(dst, nullptr, n);
}
HostCopier::Prefault::~Prefault() {
    if (c_.st_) c_.st_->pool.finish();
}

// Eight chunks or more, so that the DMA of one runs beside the host copies of others.
static size_t chunk_of(size_t n) { return std::min(kSlot, std::max<size_t>(256u << 10, (n / 8 + 65535) & ~(size_t)65535)); }

hipError_t HostCopier::to_host(void *dst, const void *src, size_t n, hipStream_t s) {
    if (n < kMin || n % 16 || (uintptr_t)src % 16 || !ready()) {
        const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    uint8_t *ring = st_->ring;
    CopyPool &pool = st_->pool;
    const size_t chunk = chunk_of(n);
    const int nc = (int)((n + chunk - 1) / chunk);
    hipError_t e = hipSuccess;
    const auto fetch = [&](int i) {
        const size_t o = i * chunk, m = std::min(chunk, n - o);
        hipLaunchKernelGGL(k_copy_out, dim3(kOutBlocks), dim3(kOutThreads), 0, s, (const uint4 *)((const uint8_t *)src + o),
                           (uint4 *)(ring + (i % kSlots) * kSlot), m / 16);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(st_->ev[i % kSlots], s);
    };
    for (int i = 0; e == hipSuccess && i < std::min(nc, kSlots - 1); i++) fetch(i);
    for (int i = 0; e == hipSuccess && i < nc; i++) {
        e = hipEventSynchronize(st_->ev[i % kSlots]);
        if (e != hipSuccess) break;
        const size_t o = i * chunk;
        pool.start((uint8_t *)dst + o, ring + (i % kSlots) * kSlot, std::min(chunk, n - o));
        // starting chunk i finished chunk i - 1's copy, whose slot is the next one to fill
        if (i + kSlots - 1 < nc) fetch(i + kSlots - 1);
    }
    pool.finish();
    if (e != hipSuccess) (void)hipStreamSynchronize(s);   // nothing may still write the ring
    return e;
}

}  // namespace sh
