// tm_groups.h -- the streams that runs of large batches take.
//
// A step is a chain of launches, and between two of them the GPU drains: the last wave
// of workgroups of one runs alone, and the next starts some microseconds later.  Two
// halves of a batch as two chains on two streams fill each other's gaps: 1024^2 x 4 of
// FP32 DP 38.6 -> 27.3 us a step, 256^2 x 16 of two-species DP consumers 110.6 -> 88.5,
// 512^2 x 16 of FP64 Rietkerk 165.5 -> 152.4 (three or four chains are no faster).
// That holds while the streams have hardware queues that run side by side.  HIP lays
// streams onto a few queues (four by default, whichever are least used when a stream is
// made) and queues onto pipes, and two chains that share one take turns: 143 us for the
// consumer batch above.  So the streams of runs, lanes, are made and measured once per
// device, and a run takes the free ones whatever the context's own stream shares.  Making
// them takes 2 to 8 ms (a hardware queue's first stream 2.8), so they are kept from one
// context to the next: released with the last of them, they took 10 of the 12 ms of a
// context that made one short run.  A
// batch is grouped only while its run is the device's only one in the process: runs of
// several contexts already overlap (two of half the consumer batch each 92 us a step; four
// of a quarter 126 on the contexts' streams, 92 to 126 on lanes).  Other processes on the
// card are not seen: two with the consumer batch each 157 us a step, grouped 192.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <memory>
#include <mutex>

namespace tmk {

class RunLanes {
public:
    // A context's share of the device's lanes.  The last one's end gives the streams back
    // if no context has prepared them since there last was none.
    static std::shared_ptr<RunLanes> get(int device) noexcept;
    // Makes and measures the lanes at the first call; false where fewer than two ran side
    // by side.  Work of others on the GPU can make two queues look like one, so up to
    // kAttempts calls measure until two are found.
    bool prepare();
    // A free lane of its own, or -1; to be given back when what it was given is done.
    int take();
    void give(int lane);
    hipStream_t stream(int lane) const { return s_[lane]; }
    // `after` goes on once what is on `before` now is done (the lane's event: one of the
    // two is this lane's).
    bool order(int lane, hipStream_t before, hipStream_t after)
    {
        return hipEventRecord(ev_[lane], before) == hipSuccess && hipStreamWaitEvent(after, ev_[lane], 0) == hipSuccess;
    }
    // Runs of the device's contexts between their first launch and their last wait.
    void begin() { runs_.fetch_add(1); }
    void end() { runs_.fetch_sub(1); }
    bool alone() const { return runs_.load() == 1; }

private:
    static constexpr int kLanes = 4, kTries = 8, kAttempts = 4;
    explicit RunLanes(int device) : device_(device) {}
    void leave();
    void make();
    void release();
    bool side_by_side(int n);   // streams 0 .. n
    const int device_;
    std::mutex mu_;
    std::atomic<int> runs_{0};
    int contexts_ = 0;
    bool wanted_ = false;       // since there last was no context
    int attempts_ = 0;
    int n_ = 0;
    hipStream_t s_[kLanes] = {};
    hipEvent_t ev_[kLanes] = {};
    bool taken_[kLanes] = {};
};

}  // namespace tmk
