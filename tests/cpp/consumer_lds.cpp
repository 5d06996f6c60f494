// Opt-in of the consumers' step kernels to more LDS than a launch may take by default
// (64 KiB, static and dynamic together), for every variant and every accepted perception
// radius, on small and large batches.
#include <map>

#include "tm_consumers.hip"

namespace tmk {
namespace {
thread_local double s_lds[1];   // the kernels do not run here
}
}  // namespace tmk

using namespace tmk;

int main()
{
    // the static LDS of the kernels with a thread per cell, three species; the others have less
    constexpr size_t kStatic = 23 << 10, kDefault = 64 << 10;
    std::map<const void*, size_t> granted;
    cpu_hip::static_lds = [&](const void*) { return kStatic; };
    cpu_hip::on_opt_in = [&](const void* f, int bytes) {
        granted[f] = (size_t)bytes;
        return hipSuccess;
    };
    size_t seen = 0;
    int bad = 0;
    cpu_hip::on_launch = [&](const cpu_hip::Launch& l) {
        if (l.lds == 0) return;
        ++seen;
        if (l.lds + kStatic > kDefault && granted[l.kernel] < l.lds) {
            fprintf(stderr, "%zu bytes of LDS in a workgroup of %u threads without an opt-in\n", l.lds + kStatic, l.block.x);
            ++bad;
        }
    };
    for (int ns = 2; ns <= 3; ++ns) {
        int n = 0;
        const Variant* v = ns == 2 ? dpc2_variants_f64(&n) : dpc3_variants_f64(&n);
        for (int halo = TM_DPC_MAX_RADIUS; halo >= 1; --halo) {   // a later context's need is smaller
            if (!dpc_lds_ready(ns, halo)) return 2;
            for (int tiles : {2, 100000})
                for (int k = 0; k < n; ++k) {
                    ConsumerArgs a{};
                    a.ntiles = a.ptiles = tiles;
                    a.halo = halo;
                    v[k].fn(a, tiles, nullptr);
                }
        }
    }
    // a refusal is the caller's to know
    cpu_hip::on_opt_in = [](const void*, int) { return hipErrorUnknown; };
    if (dpc_lds_ready(3, TM_DPC_MAX_RADIUS)) {
        fprintf(stderr, "a refused opt-in went unnoticed\n");
        ++bad;
    }
    if (bad || seen == 0) return 1;
    puts("ok");
    return 0;
}
