// On which streams the runs of a large batch launch, through the C interface: short runs on
// the context's own, long ones as two groups on two others.  Kernels do not run, but for
// those that measure the streams.
#include <map>
#include <set>

#include <hip/hip_runtime.h>

#include "tm/tm.h"

static std::set<void*> streams;   // of the step launches since it was cleared
static std::map<void*, uint64_t> clocks;
static uint64_t now = 0;
static int bad = 0;

static void check(bool ok, const char* what)
{
    if (ok) return;
    fprintf(stderr, "%s\n", what);
    ++bad;
}

int main()
{
    cpu_hip::on_launch = [](const cpu_hip::Launch& l) {
        if (strstr(l.name, "link_kernel")) {   // the clocks of streams that run side by side
            uint64_t& c = clocks[l.stream];
            cpu_hip_clock = max(c, now);
            l.run();
            c = cpu_hip_clock;
        } else if (strstr(l.name, "step")) {
            streams.insert(l.stream);
        }
    };
    cpu_hip::on_query = [](hipStream_t) {
        for (const auto& c : clocks) now = max(now, c.second);
        return hipSuccess;
    };
    tm_rietkerk_params p{};
    p.dt = 0.001;
    p.dx = p.sigma = p.D[0] = 1;
    tm_instance_desc inst[4] = {};
    for (int k = 0; k < 4; ++k) inst[k] = tm_instance_desc{256, 0, 1, (uint32_t)k, 0};
    tm_ctx* c = nullptr;
    if (tm_create(&c, 0) != TM_OK || tm_configure(c, TM_MODEL_RIETKERK, TM_F64, &p, 1, inst, 4) != TM_OK) {
        fprintf(stderr, "%s\n", tm_last_error(c));
        return 2;
    }
    void* own = tm_stream(c);
    auto run = [&](int64_t steps) {
        streams.clear();
        if (tm_run(c, steps, nullptr) < 0) {   // (a fault of fields that nothing steps)
            fprintf(stderr, "%s\n", tm_last_error(c));
            exit(2);
        }
    };
    // 4 x 256^2: 11 million cell steps are 42 steps
    for (int64_t n : {1, 8, 41}) {
        run(n);
        check(streams.size() == 1 && streams.count(own) == 1, "a short run left its context's stream");
    }
    for (int64_t n : {42, 1000}) {
        run(n);
        check(streams.size() == 2 && streams.count(own) == 0, "a long run is not in two lanes");
    }
    double ms = 0;
    streams.clear();
    (void)tm_time_steps(c, 1000, &ms, nullptr);   // its capture is refused here
    check(streams.empty() || (streams.size() == 1 && streams.count(own) == 1), "timed steps left the context's stream");
    tm_destroy(c);
    if (bad) return 1;
    puts("ok");
    return 0;
}
