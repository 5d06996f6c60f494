// The lanes of runs where the device is busy when they are first measured: a later
// measurement finds them, a device that has none is not measured for ever.  And how long
// they are kept.
#include <map>

#include "tm_groups.hip"

using namespace tmk;

static bool together;   // streams that run side by side
static int launches, streams;

int main()
{
    std::map<void*, uint64_t> clock;   // of each stream, or of all that take turns
    uint64_t now = 0;                  // at the last wait of the host
    cpu_hip::on_launch = [&](const cpu_hip::Launch& l) {
        ++launches;
        uint64_t& c = clock[together ? l.stream : nullptr];
        cpu_hip_clock = max(c, now);
        l.run();
        c = cpu_hip_clock;
    };
    cpu_hip::on_query = [&](hipStream_t) {
        for (const auto& c : clock) now = max(now, c.second);
        return hipSuccess;
    };
    cpu_hip::on_call = [](const char* f, const void*) {
        if (!strcmp(f, "hipStreamCreate")) ++streams;
        if (!strcmp(f, "hipStreamDestroy")) --streams;
    };
    int bad = 0;
    auto check = [&](bool ok, const char* what) {
        if (!ok) fprintf(stderr, "%s\n", what), ++bad;
    };
    {
        std::shared_ptr<RunLanes> g = RunLanes::get(0);
        check(!g->prepare(), "lanes on a busy device");
        check(g->take() < 0, "a lane without a second");
        together = true;
        check(g->prepare(), "no lanes once the device is idle");
        const int a = g->take(), b = g->take();
        check(a >= 0 && b >= 0 && a != b, "two lanes");
        if (a >= 0) g->give(a);
        if (b >= 0) g->give(b);
        const int n = launches;
        check(g->prepare() && launches == n, "measured again once made");
    }
    {
        // kept for the next context that wants them, whether its runs take them or not ...
        for (int life = 0; life < 3; ++life) {
            std::shared_ptr<RunLanes> g = RunLanes::get(0), h = RunLanes::get(0);
            const int n = launches;
            check(g->prepare() && launches == n, "made again for the next context");
        }
        // ... and given back at the end of one that does not
        { std::shared_ptr<RunLanes> g = RunLanes::get(0); }
        std::shared_ptr<RunLanes> g = RunLanes::get(0);
        const int n = launches;
        check(g->prepare() && launches > n, "lanes that nobody wanted were kept");
    }
    {
        { std::shared_ptr<RunLanes> g = RunLanes::get(0); }
        together = false;
        std::shared_ptr<RunLanes> g = RunLanes::get(0);
        int measured = 0;
        for (int k = 0; k < 20; ++k) {
            const int n = launches;
            check(!g->prepare(), "lanes that take turns");
            measured += launches != n;
        }
        check(measured >= 2 && measured <= 4, "measurements of a device without lanes");
    }
    { std::shared_ptr<RunLanes> g = RunLanes::get(0); }   // (an unwanted set of lanes)
    check(streams == 0, "streams left over");
    if (bad) return 1;
    puts("ok");
    return 0;
}
