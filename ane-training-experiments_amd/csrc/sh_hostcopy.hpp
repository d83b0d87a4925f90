// sh_hostcopy.hpp — large results copied into a caller's ordinary (pageable) memory.
//
// The entry points return host arrays, so a full-sequence forward's logits (32.8 MB for Stories110M
// at 256 positions) cross PCIe into pages the caller has often just mapped. The runtime's own copy
// moves 17 GB/s into warm pages and, faulting them on its one thread, 4 to 9 into fresh ones, against
// 56 GB/s of PCIe into pinned memory. Here the transfer runs through a small pinned ring, a few
// threads move the other half of the way, and the result's pages are faulted in while the GPU still
// computes it.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace sh {

// Owned by one model or trainer and used, like it, by one thread at a time, always with the
// owner's stream. The copiers of a process share one pinned ring (8 MiB) and its threads, one copy
// at a time: they come once the process has copied 32 MiB of large results without them, and go
// with the last object that used them. Without them (not set up yet, another thread's copy has
// them, allocation refused) the runtime's copy is used.
class HostCopier {
  public:
    HostCopier() = default;
    HostCopier(const HostCopier &) = delete;
    HostCopier &operator=(const HostCopier &) = delete;
    ~HostCopier() { release(); }
    // Faults in dst[0, n) beside whatever the caller does while the object lives; the contents
    // do not change.
    class Prefault {
      public:
        Prefault(HostCopier &c, void *dst, size_t n);
        ~Prefault();

      private:
        HostCopier &c_;
        const bool on_;
    };
    // Copies n device bytes to dst after the stream's earlier work; dst is complete on return.
    hipError_t to_host(void *dst, const void *src, size_t n, hipStream_t s);

  private:
    struct State;
    bool hold(size_t n);   // true: the ring is this copier's until let_go()
    void let_go();
    void release();
    State *st_ = nullptr;
    bool refused_ = false;
};

}  // namespace sh
