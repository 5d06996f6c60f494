// The staged download on the CPU: what it copies, what it returns where the device's copy
// never lands, and the calling thread's current device.
#include <sys/time.h>
#include <unistd.h>

#include "tm_hostcopy.hip"

using namespace tmk;

static int bad = 0;
static void check(bool ok, const char* what)
{
    if (ok) return;
    fprintf(stderr, "%s\n", what);
    ++bad;
}

static bool copies(HostCopier& c, size_t n, bool widen)
{
    std::vector<double> src64(widen ? 0 : n), dst(n, -1.0);
    std::vector<float> src32(widen ? n : 0);
    for (size_t i = 0; i < n; ++i) {
        if (widen) src32[i] = (float)i * 0.25f;
        else src64[i] = (double)i * 0.25;
    }
    const void* src = widen ? (const void*)src32.data() : (const void*)src64.data();
    if (c.copy(dst.data(), src, n, widen) != HostCopier::kOk) return false;
    for (size_t i = 0; i < n; ++i)
        if (dst[i] != (double)i * 0.25) return false;
    return true;
}

int main()
{
    alarm(100);   // a copy that waits for good ends here
    cpu_hip::device = 3;
    // made once the downloads come to 8 MiB, and again after the last user's end
    std::shared_ptr<HostCopier> c;
    for (int life = 0; life < 3; ++life) {
        c.reset();
        check(HostCopier::get(1, 5 << 20) == nullptr, "a copier for a first download");
        check(HostCopier::get(4 + life, 5 << 20) == nullptr, "another device's downloads counted");
        check(HostCopier::get(1, 2 << 20) == nullptr, "a copier for 7 MiB");
        c = HostCopier::get(1, 1 << 20);
        check(c != nullptr, "no copier for 8 MiB");
        check(HostCopier::get(1, 1 << 18) == c, "not the device's copier");
        cpu_hip::device = 3;
    }
    check(cpu_hip::device == 3, "making the copier changed the current device");
    c.reset();
    for (int k = 0; k < 8; ++k) {
        check(c == nullptr, "a copier for a few small downloads");
        c = HostCopier::get(1, 1 << 18);
    }
    check(c != nullptr, "no copier for many small downloads");
    cpu_hip::device = 3;
    int on = -1;
    auto run = [&](const cpu_hip::Launch& l) {
        on = cpu_hip::device;
        l.run();
    };
    cpu_hip::on_launch = run;
    // pieces of 32 KiB, halves of 2 MiB
    for (size_t n : {1u, 4095u, 4096u, 4097u, 262143u, 262144u, 262145u, 700001u}) {
        check(copies(*c, n, false), "doubles");
        check(copies(*c, n, true), "floats");
    }
    check(on == 1, "launched with another device current");
    check(cpu_hip::device == 3, "a copy changed the current device");

    // the device fails after the launch: nothing lands, and the stream says so
    std::vector<double> buf(700001);
    int launches = 0;
    for (int healthy : {0, 2}) {                        // launches that land before that
        for (hipError_t says : {hipErrorUnknown, hipSuccess}) {   // an error, or done without the flags
            launches = 0;
            cpu_hip::on_launch = [&](const cpu_hip::Launch& l) {
                if (launches++ < healthy) l.run();
            };
            int asked = 0;
            cpu_hip::on_query = [&](hipStream_t) { return ++asked < 3 ? hipErrorNotReady : says; };
            check(c->copy(buf.data(), buf.data(), buf.size(), false) == HostCopier::kFailed, "a failed copy returned kOk");
        }
    }
    // the next one is served
    cpu_hip::on_launch = run;
    cpu_hip::on_query = nullptr;
    check(copies(*c, 700001, false), "doubles after a failure");
    check(cpu_hip::device == 3, "a failed copy changed the current device");
    c.reset();
    if (bad) return 1;
    puts("ok");
    return 0;
}
