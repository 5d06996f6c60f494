// The operators' kept scratch: a context's end gives back its own device's blocks only.
#include <map>

#include "tm_movement.hip"

namespace {
thread_local double s_move[1];   // of kernels that do not run here
}
namespace tmk { namespace {
thread_local double s_move[1];
} }
extern "C" int tm_perception_offsets(int, int32_t*, int) { return 0; }

int main()
{
    std::map<const void*, int> blocks;   // kept allocations and their devices
    cpu_hip::on_call = [&](const char* f, const void* p) {
        if (!strcmp(f, "hipMalloc")) blocks[p] = cpu_hip::device;
        if (!strcmp(f, "hipFree")) blocks.erase(p);
    };
    auto count = [&](int dev) {
        int n = 0;
        for (const auto& b : blocks) n += b.second == dev;
        return n;
    };
    tm_fke_rk_params p{};
    p.dt = p.dt_rk = 0.01;
    p.dx = 1;
    p.K[1] = p.K[2] = 5;
    std::vector<double> fields(4 * 9 * 9, 1.0);
    for (int dev : {0, 1, 0}) {
        cpu_hip::device = dev;
        if (tm_fke_rk4(1, 9, &p, fields.data(), nullptr, nullptr) != TM_OK) return 2;
    }
    if (count(0) != 1 || count(1) != 1) return 3;   // one block a device, used again
    tmk::workspace_give_back(0);
    if (count(0) != 0 || count(1) != 1) {
        fprintf(stderr, "blocks kept: device 0 %d, device 1 %d\n", count(0), count(1));
        return 1;
    }
    tmk::workspace_give_back(1);
    if (!blocks.empty()) return 4;
    puts("ok");
    return 0;
}
