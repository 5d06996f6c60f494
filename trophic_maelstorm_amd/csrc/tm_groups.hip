// tm_groups.hip -- see tm_groups.h.
#include "tm_groups.h"
#include "tm_ondevice.h"

#include <algorithm>
#include <cstdint>

namespace tmk {

namespace {

constexpr int kLinks = 4;          // launches of a measured chain
constexpr int kLinkMicros = 20;

// One link: its first and last clock into t[0], t[1].
__global__ __launch_bounds__(64) void link_kernel(int64_t* t, int64_t ticks)
{
    if (threadIdx.x != 0) return;
    const int64_t t0 = (int64_t)wall_clock64();
    int64_t t1 = t0;
    for (int n = 0; n < 1 << 16 && t1 - t0 < ticks; ++n) {   // the clock ends it; the count if it stood still
        __builtin_amdgcn_s_sleep(2);
        t1 = (int64_t)wall_clock64();
    }
    t[0] = t0;
    t[1] = t1;
}

struct DevMem {
    void* p = nullptr;
    ~DevMem() { if (p) (void)hipFree(p); }
};

}  // namespace

std::shared_ptr<RunLanes> RunLanes::get(int device) noexcept
{
    static std::mutex mu;
    static RunLanes* of[64];   // never destroyed: a process ends with them
    if (device < 0 || device >= 64) return nullptr;
    try {
        RunLanes* l;
        {
            std::lock_guard<std::mutex> lock(mu);
            if (!of[device]) of[device] = new RunLanes(device);
            l = of[device];
        }
        {
            std::lock_guard<std::mutex> lock(l->mu_);
            ++l->contexts_;
        }
        return std::shared_ptr<RunLanes>(l, [](RunLanes* r) { r->leave(); });
    } catch (...) {   // no memory: runs stay on their contexts' streams
        return nullptr;
    }
}

void RunLanes::leave()
{
    std::lock_guard<std::mutex> lock(mu_);
    if (--contexts_ > 0) return;
    if (!wanted_) release();
    wanted_ = false;
}

void RunLanes::release()
{
    for (hipStream_t& s : s_)
        if (s) {
            (void)hipStreamSynchronize(s);
            (void)hipStreamDestroy(s);
            s = nullptr;
        }
    for (hipEvent_t& e : ev_)
        if (e) {
            (void)hipEventDestroy(e);
            e = nullptr;
        }
    n_ = attempts_ = 0;
}

// Whether chains of dependent short launches on streams 0 .. n, queued in turn, take less
// than 1.5 times one chain alone (on queues that take turns: twice).
bool RunLanes::side_by_side(int n)
{
    int dev = 0, khz = 0;
    DevMem mem;
    int64_t t[kLanes][kLinks][2];
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0 ||
        hipMalloc(&mem.p, sizeof(t)) != hipSuccess)
        return false;
    const int64_t ticks = (int64_t)khz * kLinkMicros / 1000;
    auto link = [&](int s, int k) {
        hipLaunchKernelGGL(link_kernel, dim3(1), dim3(64), 0, s_[s], (int64_t*)mem.p + 2 * (s * kLinks + k), ticks);
    };
    auto wait = [&]() {
        for (int s = 0; s <= n; ++s)
            if (hipStreamSynchronize(s_[s]) != hipSuccess) return false;
        return hipGetLastError() == hipSuccess;
    };
    for (int s = 0; s <= n; ++s) link(s, 0);   // the first launch on a stream may set up its queue
    int64_t span[2];
    for (int all = 0; all < 2; ++all) {
        if (!wait()) return false;
        for (int k = 0; k < kLinks; ++k)
            for (int s = 0; s <= (all ? n : 0); ++s) link(s, k);
        if (!wait() || hipMemcpy(t, mem.p, sizeof(t), hipMemcpyDeviceToHost) != hipSuccess) return false;
        int64_t first = t[0][0][0], last = t[0][kLinks - 1][1];
        for (int s = 1; s <= (all ? n : 0); ++s) {
            first = std::min(first, t[s][0][0]);
            last = std::max(last, t[s][kLinks - 1][1]);
        }
        span[all] = last - first;
    }
    return span[0] > 0 && 2 * span[1] < 3 * span[0];
}

bool RunLanes::prepare()
{
    std::lock_guard<std::mutex> lock(mu_);
    wanted_ = true;
    if (n_ < 2 && attempts_ < kAttempts) {
        ++attempts_;
        make();
    }
    return n_ >= 2;
}

void RunLanes::make()
{
    const OnDevice on(device_);
    if (!on.ok()) return;
    // New streams take the least used queues, so those passed over are kept meanwhile.
    hipStream_t passed_over[kTries];
    int np = 0;
    for (int k = 0; k < kTries && n_ < kLanes; ++k) {
        if (!ev_[n_] && hipEventCreateWithFlags(&ev_[n_], hipEventDisableTiming) != hipSuccess) {
            ev_[n_] = nullptr;
            break;
        }
        if (hipStreamCreateWithFlags(&s_[n_], hipStreamNonBlocking) != hipSuccess) {
            s_[n_] = nullptr;
            break;
        }
        if (n_ == 0 || side_by_side(n_)) {
            ++n_;
        } else {
            passed_over[np++] = s_[n_];
            s_[n_] = nullptr;
        }
    }
    for (int k = 0; k < np; ++k) (void)hipStreamDestroy(passed_over[k]);
    (void)hipGetLastError();
}

int RunLanes::take()
{
    std::lock_guard<std::mutex> lock(mu_);
    if (n_ < 2) return -1;
    for (int k = 0; k < n_; ++k)
        if (!taken_[k]) {
            taken_[k] = true;
            return k;
        }
    return -1;
}

void RunLanes::give(int lane)
{
    std::lock_guard<std::mutex> lock(mu_);
    taken_[lane] = false;
}

}  // namespace tmk
