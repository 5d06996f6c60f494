// tm_hostcopy.hip -- see tm_hostcopy.h.
#include "tm_hostcopy.h"
#include "tm_ondevice.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>

namespace tmk {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_4 __attribute__((ext_vector_type(4), aligned(4)));   // loads need dword alignment only

// Workgroup b copies piece b of `bytes` bytes (a multiple of 4; src 4-byte aligned: an
// instance of odd side starts anywhere) into pinned memory and stores `mark` in its
// flag once every thread's writes are visible to the host.
__global__ __launch_bounds__(256) void to_pinned_kernel(const char* __restrict__ src, char* __restrict__ dst,
                                                        size_t bytes, uint64_t* flags, uint64_t mark)
{
    const size_t b0 = (size_t)blockIdx.x * HostCopier::kPiece;
    const size_t m = bytes - b0 < HostCopier::kPiece ? bytes - b0 : HostCopier::kPiece;
    for (size_t i = (size_t)threadIdx.x * 16; i + 16 <= m; i += 256 * 16)
        *(u32x4*)(dst + b0 + i) = *(const u32x4_4*)(src + b0 + i);
    const size_t t = (m & ~(size_t)15) + (size_t)threadIdx.x * 4;   // the last words of a ragged piece
    if (t < m) *(uint32_t*)(dst + b0 + t) = *(const uint32_t*)(src + b0 + t);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flags + blockIdx.x, mark, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

struct HostCopier::Impl {
    static constexpr size_t kPer = kHalf / kPiece;   // pieces of a half
    int device = 0;
    hipStream_t stream = nullptr;
    char* half[2] = {nullptr, nullptr};       // pinned
    uint64_t* flags = nullptr;                // pinned, kPer per half
    uint64_t mark = 0;                        // of the last segment queued; flags start at 0
    std::thread threads[kThreads - 1];

    // the copy in hand, set before `job` is raised: segment g (kHalf bytes of the source)
    // passes through half g % 2 in pieces of kPiece, marked mark0 + g
    double* dst = nullptr;
    size_t bytes = 0, pieces = 0, queued = 0;        // queued: segments, the calling thread's
    uint64_t mark0 = 0;
    bool widen = false;
    std::atomic<size_t> next{0};              // piece to take
    std::atomic<size_t> out[2];               // pieces copied out of each half
    std::atomic<bool> failed{false};
    std::atomic<int> busy{0};                 // threads still in the copy

    std::mutex use;                           // held by the thread whose copy runs
    std::mutex mu;
    std::condition_variable cv;
    std::atomic<uint64_t> job{0};
    std::atomic<bool> stop{false};

    // The calling thread, now and then while it waits: a stream that failed, or is done
    // and left a flag as it was, ends the copy for all threads.
    void look()
    {
        const hipError_t e = hipStreamQuery(stream);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();
            return;
        }
        bool all = e == hipSuccess;
        for (size_t g = queued < 2 ? 0 : queued - 2; g < queued; ++g)   // the segments in the halves
            for (size_t i = 0; i < kPer && g * kPer + i < pieces; ++i)
                all = all && __atomic_load_n(flags + (g & 1) * kPer + i, __ATOMIC_ACQUIRE) == mark0 + g;
        if (!all) failed = true;
    }
    static constexpr unsigned kLookEvery = 4096;     // waits; a wait is a yield, under a microsecond
    void wait(unsigned& waits, bool caller)
    {
        if (caller && ++waits % kLookEvery == 0) look();
        std::this_thread::yield();
    }

    // One piece below `limit` off the common counter, once it has landed; false when none
    // is left.
    bool piece(size_t limit, bool caller)
    {
        size_t p = next.load();
        do {
            if (p >= limit) return false;
        } while (!next.compare_exchange_weak(p, p + 1));
        const size_t g = p / kPer, i = p % kPer;
        const uint64_t* f = flags + (g & 1) * kPer + i;
        const uint64_t want = mark0 + g;
        unsigned waits = 0;
        while (__atomic_load_n(f, __ATOMIC_ACQUIRE) != want) {
            if (failed.load()) return false;
            wait(waits, caller);
        }
        const size_t b0 = p * kPiece, m = std::min(kPiece, bytes - b0);
        const char* from = half[g & 1] + i * kPiece;
        if (widen) {
            const float* s = (const float*)from;
            double* d = dst + b0 / sizeof(float);
            for (size_t k = 0; k < m / sizeof(float); ++k) d[k] = s[k];
        } else {
            std::memcpy((char*)dst + b0, from, m);
        }
        out[g & 1].fetch_add(1, std::memory_order_release);
        return true;
    }
    void loop()
    {
        uint64_t seen = 0;
        for (;;) {
            // copies come in runs (one call per instance): look for the next one for a
            // moment before sleeping (10 times as long took as long a copy, and the CPUs)
            const auto t0 = std::chrono::steady_clock::now();
            while (job.load(std::memory_order_acquire) == seen && !stop.load() &&
                   std::chrono::steady_clock::now() - t0 < std::chrono::microseconds(20))
                std::this_thread::yield();
            if (job.load(std::memory_order_acquire) == seen && !stop.load()) {
                std::unique_lock<std::mutex> lock(mu);
                cv.wait(lock, [&] { return job.load() != seen || stop.load(); });
            }
            if (stop.load()) return;
            seen = job.load(std::memory_order_acquire);
            while (piece(pieces, false)) {}
            busy.fetch_sub(1, std::memory_order_release);
        }
    }
    ~Impl()
    {
        {
            std::lock_guard<std::mutex> lock(mu);
            stop = true;
        }
        cv.notify_all();
        for (std::thread& t : threads)
            if (t.joinable()) t.join();
        if (stream) {
            (void)hipStreamSynchronize(stream);
            (void)hipStreamDestroy(stream);
        }
        for (char* h : half)
            if (h) (void)hipHostFree(h);
        if (flags) (void)hipHostFree(flags);
    }
};

std::shared_ptr<HostCopier> HostCopier::get(int device, size_t bytes) noexcept
{
    static std::mutex mu;
    static std::weak_ptr<HostCopier> of[64];
    static size_t plain[64], after[64];   // bytes downloaded without one since; how many it takes
    if (device < 0 || device >= 64) return nullptr;
    try {
        std::lock_guard<std::mutex> lock(mu);
        if (std::shared_ptr<HostCopier> c = of[device].lock()) return c;
        plain[device] += std::max(bytes, kCountedMin);
        if (plain[device] < std::max(after[device], kMakeAfter)) return nullptr;
        plain[device] = 0;
        after[device] = kRefused;
        std::shared_ptr<HostCopier> c(new HostCopier());
        Impl* m = c->impl_ = new Impl();
        m->device = device;
        const OnDevice on(device);
        const bool ok = on.ok() &&
                        hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) == hipSuccess &&
                        hipHostMalloc((void**)&m->half[0], kHalf, hipHostMallocDefault) == hipSuccess &&
                        hipHostMalloc((void**)&m->half[1], kHalf, hipHostMallocDefault) == hipSuccess &&
                        hipHostMalloc((void**)&m->flags, sizeof(uint64_t) * 2 * Impl::kPer, hipHostMallocDefault) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            return nullptr;
        }
        std::memset(m->flags, 0, sizeof(uint64_t) * 2 * Impl::kPer);
        for (std::thread& t : m->threads) t = std::thread([m] { m->loop(); });
        of[device] = c;
        after[device] = kMakeAfter;
        return c;
    } catch (...) {   // no thread, no memory: the caller copies without staging
        return nullptr;
    }
}

HostCopier::~HostCopier() { delete impl_; }

HostCopier::Result HostCopier::copy(double* dst, const void* src, size_t n, bool widen)
{
    Impl& m = *impl_;
    std::unique_lock<std::mutex> use(m.use, std::try_to_lock);
    if (!use.owns_lock()) return kBusy;
    const OnDevice on(m.device);
    if (!on.ok()) return kFailed;
    m.dst = dst;
    m.bytes = n * (widen ? sizeof(float) : sizeof(double));
    m.pieces = (m.bytes + kPiece - 1) / kPiece;
    m.widen = widen;
    const size_t segs = (m.bytes + kHalf - 1) / kHalf;
    m.mark0 = m.mark + 1;
    m.mark += segs;
    m.next = 0;
    m.out[0] = m.out[1] = 0;
    m.failed = false;
    m.busy = kThreads - 1;
    m.queued = 0;
    size_t& queued = m.queued;
    unsigned waits = 0;
    auto queue = [&]() {
        const size_t b0 = queued * kHalf, b = std::min(kHalf, m.bytes - b0);
        hipLaunchKernelGGL(to_pinned_kernel, dim3((unsigned)((b + kPiece - 1) / kPiece)), dim3(256), 0, m.stream,
                           (const char*)src + b0, m.half[queued & 1], b, m.flags + (queued & 1) * Impl::kPer,
                           m.mark0 + queued);
        if (hipGetLastError() != hipSuccess) m.failed = true;
        ++queued;
    };
    queue();
    {
        std::lock_guard<std::mutex> lock(m.mu);
        m.job.fetch_add(1, std::memory_order_release);
    }
    m.cv.notify_all();
    // Segment g takes its half once the g / 2 segments before it there are out.  Until then
    // this thread copies pieces of the queued segments only: a later one would wait for it.
    while (queued < segs && !m.failed) {
        if (m.out[queued & 1].load(std::memory_order_acquire) >= queued / 2 * Impl::kPer) queue();
        else if (!m.piece(queued * Impl::kPer, true)) m.wait(waits, true);
    }
    while (m.piece(m.pieces, true)) {}
    while (m.busy.load(std::memory_order_acquire) != 0) m.wait(waits, true);
    if (m.failed) (void)hipStreamSynchronize(m.stream);
    return m.failed ? kFailed : kOk;
}

}  // namespace tmk
