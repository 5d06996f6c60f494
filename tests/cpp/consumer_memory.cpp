// A DP consumer batch whose allocations are refused one after another: configuring it is an
// error, or the fields it steps are those of a batch that got everything.
#include <hip/hip_runtime.h>

#include "tm/tm.h"

static int at, refused;   // allocations of a batch so far; the one that is refused, or -1

static tm_status step(int model, std::vector<double>& out)
{
    const int nf = model == TM_MODEL_DP3 ? 5 : 3, L = 33;
    tm_dpc_params p{};
    p.a = p.b = 0.5;
    p.dt = p.dx = 0.1;
    for (int s = 0; s < 3; ++s) {
        p.D[s] = 0.001 * (s + 1);
        p.sigma[s] = 0.5 + 0.2 * s;
        p.v[s] = 0.3 * (s > 0);
        p.M[s] = 0.1 * s;
        p.E[s] = 0.6;
        p.pR[s] = s > 0 ? 0.25 : 0.0;
    }
    p.A[0][1] = p.A[1][0] = p.A[1][2] = p.A[2][1] = 0.7;
    p.H[0][1] = p.H[1][0] = p.H[1][2] = p.H[2][1] = 0.5;
    p.flush_eps = 1e-12;
    p.flush_neg = -1e-80;
    tm_instance_desc inst[2] = {{L, 0, 7, 1, 0}, {L, 0, 7, 2, 0}};
    tm_ctx* c = nullptr;
    at = -1000;   // the context's own are all served
    if (tm_create(&c, 0) != TM_OK) return TM_ERR_HIP;
    at = 0;
    tm_status s = tm_configure(c, model, TM_F64, &p, 1, inst, 2);
    const int configured = at;
    if (s == TM_OK) {
        at = 1000;   // and the run's
        const double lo[8] = {}, hi[8] = {20.0, 2.0, 0.5, 0.0, 0.0};
        s = tm_init_uniform(c, lo, hi);
        if (s == TM_OK) s = tm_run(c, 4, nullptr);
        out.assign((size_t)(nf * L * L), 0.0);
        if (s == TM_OK) s = tm_download_fields(c, 1, out.data());
    }
    tm_destroy(c);
    at = configured;
    return s;
}

int main()
{
    cpu_hip::refuse = [](size_t) { return at++ == refused; };
    for (int model : {TM_MODEL_DP2, TM_MODEL_DP3}) {
        std::vector<double> want, got;
        refused = -1;
        if (step(model, want) != TM_OK) return 2;
        int served = 0, denied = 0;
        for (int k = 0;; ++k) {
            refused = k;
            const tm_status s = step(model, got);
            if (s != TM_OK) {
                ++denied;
                continue;
            }
            if (got != want) {
                fprintf(stderr, "model %d: other fields without allocation %d\n", model, k);
                return 1;
            }
            if (at <= k) break;   // there was none to refuse
            ++served;
        }
        if (served < 1 || denied < 1) {
            fprintf(stderr, "model %d: %d allocations can be done without, %d cannot\n", model, served, denied);
            return 1;
        }
    }
    puts("ok");
    return 0;
}
