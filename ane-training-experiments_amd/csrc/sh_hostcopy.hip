// sh_hostcopy.hip — the large copies declared in sh_hostcopy.hpp.
#include "sh_hostcopy.hpp"

#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <utility>

#include "sh_copypool.hpp"

namespace sh {
namespace {

// Smaller copies take the runtime's own path: 0.25 MiB alone 22 us against 47 through the ring with the
// helpers asleep. Whole calls, three models in turn, by the runtime and through the ring: a layer over
// 180 rows (0.55 MB) 167 us and 139, over 640 (2 MB) 350 and 287; logits of 5 rows (0.64 MB) 231 us
// and 226, of 20 (2.6 MB) 346 and 284. (The other way the runtime is as fast up to 16 MiB: 2 MiB in 80
// us against 201 through the ring.)
constexpr size_t kMin = 512u << 10;
// The ring and the threads are set up once a process has copied this much without them: it takes 0.5
// to 2 ms, mostly of pinning, against about 1 ms that they save per 32 MiB.
constexpr size_t kSetUp = 32u << 20;
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

// One for all copiers of the process: whoever holds `use` may use it.
struct Ring {
    std::mutex use;
    uint8_t *mem = nullptr;
    CopyPool pool{std::max(1, std::min(kMaxHelpers, (int)std::thread::hardware_concurrency() / 2 - 1))};
    ~Ring() {
        if (mem) (void)hipHostFree(mem);
    }
};

std::mutex g_ring_mu;
std::weak_ptr<Ring> g_ring;
std::atomic<size_t> g_copied{0};   // bytes of large copies made without the ring

// The process's ring, made if none of its copiers holds one; null where it can't be made.
std::shared_ptr<Ring> shared_ring() {
    try {
        std::lock_guard<std::mutex> lk(g_ring_mu);
        std::shared_ptr<Ring> r = g_ring.lock();
        if (r) return r;
        r = std::make_shared<Ring>();
        if (hipHostMalloc((void **)&r->mem, kSlots * kSlot, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        g_ring = r;
        return r;
    } catch (const std::exception &) {
        return nullptr;
    }
}

}  // namespace

struct HostCopier::State {
    std::shared_ptr<Ring> ring;
    hipEvent_t ev[kSlots] = {};
    bool held = false;   // ring->use
};

bool HostCopier::hold(size_t n) {
    if (n < kMin || refused_) return false;
    if (!st_) {
        if (g_copied.load() < kSetUp) return false;
        std::shared_ptr<Ring> r = shared_ring();
        st_ = r ? new (std::nothrow) State : nullptr;
        refused_ = !st_;
        if (refused_) return false;
        st_->ring = std::move(r);
        for (hipEvent_t &e : st_->ev)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                release();
                refused_ = true;
                return false;
            }
    }
    return st_->held = st_->ring->use.try_lock();   // another thread's copy has it: the runtime's copy is used
}

void HostCopier::let_go() {
    st_->held = false;
    st_->ring->use.unlock();
}

void HostCopier::release() {
    if (!st_) return;
    for (hipEvent_t e : st_->ev)
        if (e) (void)hipEventDestroy(e);
    delete st_;
    st_ = nullptr;
}

HostCopier::Prefault::Prefault(HostCopier &c, void *dst, size_t n) : c_(c), on_(c.hold(n)) {
    if (on_) c.st_->ring->pool.start(dst, nullptr, n);
}
HostCopier::Prefault::~Prefault() {
    if (!on_) return;
    c_.st_->ring->pool.finish();
    c_.let_go();
}

// Eight chunks or more, so that the DMA of one runs beside the host copies of others.
static size_t chunk_of(size_t n) { return std::min(kSlot, std::max<size_t>(256u << 10, (n / 8 + 65535) & ~(size_t)65535)); }

hipError_t HostCopier::to_host(void *dst, const void *src, size_t n, hipStream_t s) {
    const bool prefaulted = st_ && st_->held;
    if (n < kMin || n % 16 || (uintptr_t)src % 16 || (!prefaulted && !hold(n))) {
        if (n >= kMin) g_copied += n;
        const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    uint8_t *ring = st_->ring->mem;
    CopyPool &pool = st_->ring->pool;
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
    if (!prefaulted) let_go();
    return e;
}

}  // namespace sh
