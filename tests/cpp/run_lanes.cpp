// The lanes of runs where the device is busy when they are first measured: a later
// measurement finds them, a device that has none is not measured for ever.
#include <map>

#include "tm_groups.hip"

using namespace tmk;

static bool together;   // streams that run side by side
static int launches;

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
    if (bad) return 1;
    puts("ok");
    return 0;
}
