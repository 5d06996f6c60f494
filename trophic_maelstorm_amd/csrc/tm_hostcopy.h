// tm_hostcopy.h -- device-to-host copies into pageable memory through pinned staging.
//
// hipMemcpy into pageable memory reaches 17 GB/s here, and widening FP32 fields to FP64
// in one thread 16, where the link carries 56 GB/s into pinned memory.  A HostCopier
// holds two pinned halves and a few threads: a kernel writes the source into a half,
// one workgroup per piece, and raises the piece's flag in pinned memory when it has
// landed (DMA copies with an event per slot cost 15 us a slot); the threads, the calling
// one among them, copy (or widen) the landed pieces out.  Halves of 2 MiB stay in the
// host's caches: 8 MiB of FP64 in 213 us (480 before; 267 with halves of 8 MiB), 4 MiB of
// FP32 widened in 129 (514), 256 KiB in 18 (25).
// One HostCopier per device is shared by the contexts that made a large download and
// released with the last of them.  Making and releasing it takes 0.8 ms, what it saves on
// 7 MiB into fresh memory (whose page faults its threads share) or 24 MiB into memory in use,
// so it is made with the download that brings those without one to 8 MiB, each counted as
// 1 MiB at least (a plain copy of 256 KiB takes up to 115 us, a staged one 18): a context
// that downloads 2 MiB once took 0.6 ms longer for it.
#pragma once
#include <cstddef>
#include <memory>

namespace tmk {

class HostCopier {
public:
    static constexpr int kThreads = 8;        // the calling thread and seven of its own
    static constexpr size_t kHalf = (size_t)2 << 20, kPiece = (size_t)32 << 10;
    static constexpr size_t kMakeAfter = (size_t)8 << 20, kCountedMin = (size_t)1 << 20;
    // The device's copier for a download of so many bytes of doubles.  Null where there is
    // none and the downloads since the last come to less than kMakeAfter with this one, and
    // where threads, streams or pinned memory are refused (tried again after kRefused more).
    static std::shared_ptr<HostCopier> get(int device, size_t bytes) noexcept;
    ~HostCopier();
    enum Result { kOk, kBusy, kFailed };
    // n elements at src (device, complete: the caller has waited for its writers) to dst
    // (host): floats widened to doubles, or doubles as they are.  kBusy, with nothing
    // done, while another thread's copy runs; kFailed on a HIP error, of the device's copy
    // too.  The caller's current device stays what it is.
    Result copy(double* dst, const void* src, size_t n, bool widen);

private:
    static constexpr size_t kRefused = (size_t)1 << 30;
    HostCopier() = default;
    struct Impl;
    Impl* impl_ = nullptr;
};

}  // namespace tmk
