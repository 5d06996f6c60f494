// tm_consumers.hip -- the vegetation + consumer step (multiSPDP.cpp built with
// SPB = 2: vegetation and grazer; SPB = 3: and predator), FP64, performing the
// CPU restatement's operations in its order with contraction off.
//
// Fields per instance: rho_0 .. rho_{NS-1}, then the perception fields
// gamma_1 .. gamma_{NS-1} (NF = 2 NS - 1), species-major [NF][L*L].
//
// A step is three launches:
//   dpc_head_kernel   the vegetation's Dornic step P* (:2901-2945), and beside it one
//                     workgroup per 4096-cell chunk: the chunk's sums of every
//                     density and the occupied count of the vegetation, in a
//                     fixed order (lane strides, then a pairwise fold);
//   dpc_state_kernel  one thread per instance: the chunk sums in chunk order ->
//                     spatial means, the cover factor and the number of
//                     perception neighbours each consumer uses this step
//                     (multiSPDP.cpp:2962-2975, :1705-1730);
//   dpc_step_kernel   one workgroup per tile: the tile and a halo of the
//                     perception radius of every density in LDS, then each
//                     consumer's perception gamma (:1699-1786, :2166-2284) and
//                     its Dornic step with upwind advection in a random direction
//                     (:3041-3190), and per cell the RK4 of the trophic terms from
//                     P* (:1821-1898), checks and flush (:3228-3262), and rho(t)
//                     partials.
// The means steer the step (they scale gamma and switch consumers off), so they
// come from the fixed-order reduction rather than from the compensated rho(t)
// rows; the rows stay the reporting path.
#include <hip/hip_runtime.h>
#include "tm_launch.h"
#include "tm_veg.h"

namespace tmk {

namespace {

constexpr int kChunk = kDpcChunkCells;
constexpr double kGammaEps = 1.0e-12;   // calc_gamma's eps (multiSPDP.cpp:1715, :2182)

template <int NS>
__device__ __forceinline__ void dpc_chunk(const ConsumerArgs& a, const DPCWork* w, int block, double (&red)[NS + 1][256])
{
#pragma clang fp contract(off)
    constexpr int NF = 2 * NS - 1;
    const int2 ch = w->chunks[block];
    const DevInst di = a.inst[ch.x];
    const int64_t N = (int64_t)di.L * di.L;
    const double* f0 = (const double*)a.in + (int64_t)NF * di.cell_off;
    const int64_t base = (int64_t)ch.y * kChunk;
    const int t = threadIdx.x;
    double s[NS + 1];
#pragma unroll
    for (int f = 0; f <= NS; ++f) s[f] = 0.0;
    for (int64_t i = base + t; i < base + kChunk && i < N; i += 256) {
#pragma unroll
        for (int f = 0; f < NS; ++f) s[f] += f0[f * N + i];
        s[NS] += f0[i] > 0.0 ? 1.0 : 0.0;
    }
#pragma unroll
    for (int f = 0; f <= NS; ++f) red[f][t] = s[f];
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (t < o) {
#pragma unroll
            for (int f = 0; f <= NS; ++f) red[f][t] += red[f][t + o];
        }
        __syncthreads();
    }
    if (t == 0) {
#pragma unroll
        for (int f = 0; f <= NS; ++f) w->chunk[(int64_t)block * 4 + f] = red[f][0];
    }
}

// The vegetation's Dornic step (workgroups 0 .. nvtiles - 1) and the chunk sums (the
// rest): both read the old fields only, so the short sums run beside the samplers.
template <int NS>
__global__ __launch_bounds__(256, 5) void dpc_head_kernel(ConsumerArgs a)
{
    constexpr int NF = 2 * NS - 1;
    __shared__ union {
        VegLds veg;
        double red[NS + 1][256];
    } sm;
    const DPCWork* w = (const DPCWork*)a.work;
    if ((int)blockIdx.x >= a.nvtiles) {
        dpc_chunk<NS>(a, w, a.chunk0 + (int)blockIdx.x - a.nvtiles, sm.red);
        return;
    }
    const int4 tl = w->vtiles[a.vtile0 + blockIdx.x];   // (instance, x0, y0)
    const DevInst di = a.inst[tl.x];
    const DPCConst c = ((const DPCConst*)a.consts)[(int64_t)a.k * a.n_inst + tl.x];
    const VegConst vc = {c.k, di.seed, di.inst_id, c.compat, c.step};
    const double* P = (const double*)a.in + (int64_t)NF * di.cell_off;
    double* pstar = (double*)a.out + (int64_t)NF * di.cell_off;   // field 0, where the step takes it from
    if (a.vdirect) {   // 64 x 4 tiles, one cell a thread
        const int y = tl.z + (int)(threadIdx.x >> 6), x = tl.y + (int)(threadIdx.x & 63);
        if (y < di.L && x < di.L) veg_cell(vc, di.L, y, x, P, pstar);
    } else {
        veg_tile(vc, di.L, tl.y, tl.z, P, pstar, sm.veg);
    }
}

// The per-instance numbers of the perception step, a wave per instance.
template <int NS>
__global__ __launch_bounds__(64) void dpc_state_kernel(ConsumerArgs a)
{
#pragma clang fp contract(off)
    __shared__ double s_sum[64 * (NS + 1)];
    const int i = a.inst0 + blockIdx.x, f = threadIdx.x;
    const DPCWork* w = (const DPCWork*)a.work;
    const DPCInstInfo& in = w->info[i];
    const DevInst di = a.inst[i];
    const double N = (double)((int64_t)di.L * di.L);
    const double tot = chunk_totals<NS + 1, 4>(w->chunk + (int64_t)in.chunk0 * 4, in.nchunks, s_sum);
    if (f >= NS) return;
    const double fr = in.fr[f];
    double nfac = 1 - s_sum[NS] / N;                 // multiSPDP.cpp:2972-2974
    if (nfac < 0.35) nfac = 0.35;
    const int new_len = (int)(nfac * nfac * (double)in.disk_len);
    const double mean = tot / N;
    int e = (int)(fr * fr * (double)new_len);
    if (NS == 3 && e < 1 && fr > 0) e = 1;     // multiSPDP.cpp:2215-2216
    DPCStepState& st = w->st[i];
    st.mean[f] = mean;
    st.inv[f] = mean >= kGammaEps ? 1 / mean : 1 / kGammaEps;
    st.eff[f] = e;
}

// f_DP_Dor_2Sp / f_DP_Dor_3Sp (multiSPDP.cpp:1670-1697, :1789-1819) at one cell.
template <int NS>
__device__ __forceinline__ void dpc_f(const tm_dpc_params& p, const double* y, double* f)
{
#pragma clang fp contract(off)
    const double A01H01 = p.A[0][1] * p.H[0][1];
    const double EA1 = p.E[1] * p.A[0][1];
    f[0] = -p.b * y[0] * y[0] - (p.A[0][1] * y[0] / (1 + A01H01 * y[0])) * y[1];
    if constexpr (NS == 2) {
        f[1] = (EA1 * y[0] / (1 + A01H01 * y[0])) * y[1];
    } else {
        const double A12H12 = p.A[1][2] * p.H[1][2];
        const double EA2 = p.E[2] * p.A[1][2];
        f[1] = (EA1 * y[0] / (1 + A01H01 * y[0])) * y[1] - p.A[1][2] * y[1] / (1 + A12H12 * y[1]) * y[2];
        f[2] = (EA2 * y[1] / (1 + A12H12 * y[1])) * y[2];
    }
}

// RK4_Integrate_Stochastic_MultiSp (multiSPDP.cpp:1821-1898): pointwise.
template <int NS>
__device__ __forceinline__ void dpc_rk4(const tm_dpc_params& p, double* y)
{
#pragma clang fp contract(off)
    const double dt = p.dt, dt2 = dt / 2.0, dt6 = dt / 6.0;
    double k1[NS], k2[NS], k3[NS], k4[NS], ys[NS];
    dpc_f<NS>(p, y, k1);
#pragma unroll
    for (int s = 0; s < NS; ++s) ys[s] = y[s] + (dt2) * k1[s];
    dpc_f<NS>(p, ys, k2);
#pragma unroll
    for (int s = 0; s < NS; ++s) ys[s] = y[s] + (dt2) * k2[s];
    dpc_f<NS>(p, ys, k3);
#pragma unroll
    for (int s = 0; s < NS; ++s) ys[s] = y[s] + (dt) * k3[s];
    dpc_f<NS>(p, ys, k4);
#pragma unroll
    for (int s = 0; s < NS; ++s) y[s] += (dt6) * (k1[s] + 2.0 * k2[s] + 2.0 * k3[s] + k4[s]);
}

// One consumer's Dornic transition with upwind advection in a random direction
// (multiSPDP.cpp:3041-3190) at image index r of its density is, from its perception
// gamma.  FIRST: as dornic_cell_d's first pass; lambda and words (of the direction and
// the count) are for its kDornicGamma.
template <bool FIRST>
__device__ __forceinline__ int dpc_consumer(const tm_dpc_params& p, int s, const DevInst& di, uint32_t cell,
                                            int64_t step, bool compat, double gam, const double* is, int r, int RW,
                                            double& y, double& lambda, int& words)
{
#pragma clang fp contract(off)
    const double dx = p.dx, dt = p.dt;
    const double dx2 = dx * dx, dx1 = 1 / dx, dx1_2 = 1 / (dx2), dxb2 = dx / 2.0;
    const double Dc0 = p.D[0] / (dx2);
    y = is[r];
    Stream sc(di.seed, di.inst_id, cell, step);
    sc.blk = (uint32_t)s << 24;
    double sn, cs;
    dsincos2pi(sc.u64(), sn, cs);
    const double vx = p.v[s] * cs, vy = p.v[s] * sn;
    const double vxa = vx * (double)((0 < vx) - (vx < 0));
    const double vya = vy * (double)((0 < vy) - (vy < 0));
    const double gp = (1 - gam);
    double Dx = (p.D[s] - (dxb2) * (gp * vxa * (1 - dt * dx1 * gp * vxa))) * dx1_2;
    double Dy = (p.D[s] - (dxb2) * (gp * vya * (1 - dt * dx1 * gp * vya))) * dx1_2;
    if (Dx < Dc0) Dx = Dc0;
    if (Dy < Dc0) Dy = Dc0;
    const double ux = vx > 0 ? is[r - 1] : is[r + 1];
    const double uy = vy > 0 ? is[r - RW] : is[r + RW];
    const double alpha = gam * (Dy * (is[r - RW] + is[r + RW]) + Dx * (is[r - 1] + is[r + 1]))
                         + dx1 * (gp) * (vxa * ux + vya * uy);
    if (alpha == 0 && is[r] == 0) return kDornicDone;
    const double beta = -p.M[s] - 2 * gam * (Dx + Dy) - (1 - gam) * (vxa + vya) * dx1;
    const double lexp = dexp((beta) * dt);
    const double sig2_1 = 1 / (p.sigma[s] * p.sigma[s]);
    const double lam = 2 * (beta) * (sig2_1) / (lexp - 1.0);
    DornicConst k{};
    k.lambda = lam;
    k.ll = lam * lexp;
    k.sigma2_1 = sig2_1;
    double n;
    const int st = dornic_cell_d<FIRST, Stream>(sc, alpha, is[r], k, compat, n, y);
    lambda = lam;
    words = 1 + dornic_words(k.ll * is[r], compat);
    return st;
}

// One tile, in phases with a barrier between them: the consumers' perception gamma and
// first trials per cell (the vegetation's P* is in its output field), the transitions
// those leave open from two queues per consumer, densely packed, then the RK4, checks,
// flush and partials per cell.  Between phases a cell's new densities and gamma wait in
// the output fields.  In one pass every wave ran every sampler path of its 64 cells and
// held the samplers', the perception's and the RK4's registers at once (146 VGPRs): 16 x
// 256^2, two species, 139 us for the step kernel alone, 32 + 77 here.
template <int NS, int TX, int TY, int NT, int MINW>
__global__ __launch_bounds__(NT, MINW) void dpc_step_kernel(ConsumerArgs a)
{
#pragma clang fp contract(off)
    constexpr int NF = 2 * NS - 1, NC = TX * TY;
    static_assert(NC <= 512, "a queue entry holds a cell in 9 bits, then its words");
    static_assert(NT == 256 || (NT == 512 && NC == 512), "one or two cells a thread");
    extern __shared__ __align__(16) double s_lds[];
    __shared__ double s_red[2 * NF * (NT / 64)];
    __shared__ uint16_t s_q[NS - 1][NC];        // restarts from the front, Gamma deviates from the back
    __shared__ uint32_t s_n[NS - 1][2];

    const int64_t counter = a.state->counter + a.k;
    const int64_t slot = counter & (int64_t)(a.nslots - 1);
    const int tile = blockIdx.x;
    if (tile >= a.ntiles) return;
    const DevTile tl = a.tiles[tile];
    const DevInst di = a.inst[tl.inst];
    const DPCConst c = ((const DPCConst*)a.consts)[(int64_t)a.k * a.n_inst + tl.inst];
    const DPCWork* w = (const DPCWork*)a.work;
    const tm_dpc_params p = w->params[di.pidx];
    const DPCInstInfo info = w->info[tl.inst];
    const DPCStepState st = w->st[tl.inst];
    const int H = a.halo;
    const int RW = TX + 2 * H, RH = TY + 2 * H, IMG = RW * RH;
    double* img = s_lds;                        // [NS][RH][RW]
    int* offs = (int*)(s_lds + NS * IMG);       // perception offsets as LDS strides
    const int L = tl.L;
    const int64_t N = (int64_t)L * L;
    const double* fin = (const double*)a.in + (int64_t)NF * tl.cell_off;
    double* fout = (double*)a.out + (int64_t)NF * tl.cell_off;
    double* const lambdas = w->lambda;

    // 32 lanes along a row, NT / 32 rows at a time: no index division
    for (int ry = threadIdx.x >> 5; ry < RH; ry += NT / 32) {
        const int64_t row = (int64_t)wrap(tl.y0 + ry - H, L) * L;
        for (int rx = threadIdx.x & 31; rx < RW; rx += 32) {
            const int64_t g = row + wrap(tl.x0 + rx - H, L);
#pragma unroll
            for (int s = 0; s < NS; ++s) img[s * IMG + ry * RW + rx] = fin[s * N + g];
        }
    }
    for (int k = threadIdx.x; k < info.disk_len; k += NT) {
        const int2 o = w->disk[info.disk_off + k];
        offs[k] = o.x * RW + o.y;
    }
    if (threadIdx.x < 2 * (NS - 1)) (&s_n[0][0])[threadIdx.x] = 0u;
    __syncthreads();

    // perception gamma of each consumer from the old fields, and its first trials
#pragma unroll
    for (int s = 1; s < NS; ++s) {
        const bool live = !(st.mean[s] == 0.0);
        const double* is = img + s * IMG;
        const int eff = st.eff[s];
#pragma unroll 1
        for (int e = threadIdx.x; e < NC; e += NT) {
            const int ly = e / TX, lx = e % TX;
            const int gy = tl.y0 + ly, gx = tl.x0 + lx;
            const int r = (ly + H) * RW + (lx + H);
            const double* src = img + (s - 1) * IMG + r;
            int res = kDornicDone, words = 0;
            if (gy < L && gx < L) {
                const uint32_t cell = (uint32_t)gy * (uint32_t)L + (uint32_t)gx;
                double g = fin[(NS + s - 1) * N + cell];
                if (info.fr[s] == 0.0) {
                } else if (st.mean[s] < kGammaEps || st.mean[s - 1] < kGammaEps) {
                    g = 0.0;
                } else {
                    if constexpr (NS == 2) {            // accumulates onto the previous value (:1756-1760)
#pragma unroll 4
                        for (int k = 0; k < eff; ++k) g += src[offs[k]];
                        g = (g * st.inv[s - 1]) / (double)eff;
                    } else if (s == 1) {                // grazers, weighed down by predators (:2228-2249)
                        double acc = 0.0;
                        if (st.mean[2] < kGammaEps) {
#pragma unroll 4
                            for (int k = 0; k < eff; ++k) acc += src[offs[k]];
                        } else {
                            const double* pr = img + 2 * IMG + r;
#pragma unroll 4
                            for (int k = 0; k < eff; ++k) acc += src[offs[k]] * (1 - pr[offs[k]] * st.inv[2]);
                        }
                        g = (acc * st.inv[s - 1]) / (double)eff;
                    } else {                            // predators (:2251-2258)
                        double acc = 0.0;
#pragma unroll 4
                        for (int k = 0; k < eff; ++k) acc += src[offs[k]];
                        g = (acc / (double)eff) * st.inv[s - 1];
                    }
                    if (g > 1) g = 1.0;
                    else if (g < 0) g = 0.0;
                }
                double y = is[r];
                if (live) {
                    if (g > 1) g = 1;
                    double lambda;
                    res = dpc_consumer<true>(p, s, di, cell, c.step, c.compat != 0, g, is, r, RW, y, lambda, words);
                    if (res == kDornicGamma) {
                        if (lambdas) lambdas[(int64_t)(NS - 1) * tl.cell_off + (s - 1) * N + cell] = lambda;
                        else res = kDornicRestart;
                    }
                }
                fout[(NS + s - 1) * N + cell] = g;
                fout[s * N + cell] = y;
            }
            queue_push<false>(res == kDornicRestart, (uint16_t)e, s_q[s - 1], &s_n[s - 1][0]);
            queue_push<true>(res == kDornicGamma, (uint16_t)(e | words << 9), s_q[s - 1] + NC, &s_n[s - 1][1]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 1; s < NS; ++s) {
        // one list, restarts first: its waves run beside each other, nearly each on one kind
        const uint32_t n0 = s_n[s - 1][0], n1 = s_n[s - 1][1];
#pragma unroll 1
        for (uint32_t i = threadIdx.x; i < n0 + n1; i += NT) {
            const int q = i < n0 ? s_q[s - 1][i] : s_q[s - 1][NC - 1 - (i - n0)], e = q & 511;
            const int ly = e / TX, lx = e % TX;
            const uint32_t cell = (uint32_t)(tl.y0 + ly) * (uint32_t)L + (uint32_t)(tl.x0 + lx);
            double y, lambda;
            if (i < n0) {
                int words;
                dpc_consumer<false>(p, s, di, cell, c.step, c.compat != 0, fout[(NS + s - 1) * N + cell],
                                    img + s * IMG, (ly + H) * RW + (lx + H), RW, y, lambda, words);
            } else {
                Stream sc(di.seed, di.inst_id, cell, c.step);
                sc.blk = (uint32_t)s << 24;
                sc.skip(q >> 9);
                lambda = lambdas[(int64_t)(NS - 1) * tl.cell_off + (s - 1) * N + cell];
                y = dornic_gamma_d(sc, fout[s * N + cell], lambda, c.compat != 0);
            }
            fout[s * N + cell] = y;
        }
    }
    __syncthreads();

    double sum[NF], cnt[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) { sum[f] = 0.0; cnt[f] = 0.0; }
    for (int e = threadIdx.x; e < NC; e += NT) {
        const int ly = e / TX, lx = e % TX;
        const int gy = tl.y0 + ly, gx = tl.x0 + lx;
        if (gy >= L || gx >= L) continue;
        const uint32_t cell = (uint32_t)gy * (uint32_t)L + (uint32_t)gx;
        double y[NS];
        y[0] = fout[cell];
#pragma unroll
        for (int s = 1; s < NS; ++s) y[s] = fout[s * N + cell];
        dpc_rk4<NS>(p, y);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double v = y[s];
            if (v < 0 || !__builtin_isfinite(v)) record_fault(a.fault, tl.inst, s * N + cell, counter);
            if (v < c.eps && v >= c.neg) v = 0.0;
            fout[s * N + cell] = v;
            sum[s] += v;
            cnt[s] += v > 0.0 ? 1.0 : 0.0;
        }
#pragma unroll
        for (int s = 1; s < NS; ++s) {
            const double g = fout[(NS + s - 1) * N + cell];
            sum[NS + s - 1] += g;
            cnt[NS + s - 1] += g > 0.0 ? 1.0 : 0.0;
        }
    }
    if constexpr (NT > 256) {   // the sums of 256 threads with two cells each, for the same rows
        __shared__ double s_x[2 * NF][256];
        const int t = threadIdx.x - 256;
        if (t >= 0) {
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                s_x[2 * f][t] = sum[f];
                s_x[2 * f + 1][t] = cnt[f];
            }
        }
        __syncthreads();
        if (t >= 0) return;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            sum[f] += s_x[2 * f][threadIdx.x];
            cnt[f] += s_x[2 * f + 1][threadIdx.x];
        }
    }
    block_partials<256, NF>(sum, cnt, a.partials + (slot * a.ptiles + tile) * NF, s_red);
}

template <int NS, int TX, int TY, int NT, int MINW = 1>
void launch_dpc(const StepArgs& step, int grid, hipStream_t s)
{
    const ConsumerArgs& a = static_cast<const ConsumerArgs&>(step);
    const size_t lds = dpc_lds_bytes(NS, TX, TY, a.halo);   // opted in to by dpc_lds_ready
    hipLaunchKernelGGL(dpc_head_kernel<NS>, dim3(a.nvtiles + a.nchunks), dim3(256), 0, s, a);
    hipLaunchKernelGGL(dpc_state_kernel<NS>, dim3(a.inst1 - a.inst0), dim3(64), 0, s, a);
    hipLaunchKernelGGL((dpc_step_kernel<NS, TX, TY, NT, MINW>), dim3(grid), dim3(NT), lds, s, a);
}

// A workgroup takes 64 KiB of LDS by default, its static arrays among them; CDNA4 has 160.
// The opt-in is always to the widest radius, so that no context lowers another's.
template <int NS, int TX, int TY, int NT, int MINW = 1>
bool dpc_opt_in(int halo)
{
    constexpr size_t kDefaultLds = 64 << 10;
    const void* const f = (const void*)dpc_step_kernel<NS, TX, TY, NT, MINW>;
    hipFuncAttributes at;
    if (hipFuncGetAttributes(&at, f) != hipSuccess) return false;
    return at.sharedSizeBytes + dpc_lds_bytes(NS, TX, TY, halo) <= kDefaultLds ||
           hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)dpc_lds_bytes(NS, TX, TY, TM_DPC_MAX_RADIUS)) == hipSuccess;
}

// The defaults: batches of at most kWideTiles tiles (two and a half a CU) take a thread per
// cell, which halves the chain of each thread's cells; above, 512-thread workgroups leave
// fewer of them in flight.  us a step, 256 / 512 threads: two species 64^2 38.1 / 32.0, 8 x
// 128^2 (256 tiles) 41.7 / 36.0, 512^2 (512) 49.7 / 45.6, 24 x 128^2 (768) 54.2 / 54.3, 1024^2
// 112 / 137; three species 8 x 128^2 55.3 / 46.3, 20 x 128^2 (640) 74.8 / 65.6, 988 tiles of
// odd lattices 82.3 / 87.7.
constexpr int kWideTiles = 640;

template <int NS, int MINW>
void launch_dpc_default(const StepArgs& a, int grid, hipStream_t s)
{
    if (a.ptiles <= kWideTiles) launch_dpc<NS, 32, 16, 512>(a, grid, s);
    else launch_dpc<NS, 32, 16, 256, MINW>(a, grid, s);
}

// _wN: at most 512/N VGPRs, N waves per SIMD.  dpc_lds_ready has these kernels too.
const Variant kDPC2[] = {
    {32, 16, 256, 0, 1, "dpc2_f64_32x16_t256", &launch_dpc<2, 32, 16, 256>, 0, 0, nullptr, 1},
    {64, 8, 256, 0, 1, "dpc2_f64_64x8_t256", &launch_dpc<2, 64, 8, 256>, 0, 0, nullptr, 1},
    {32, 16, 256, 0, 1, "dpc2_f64_32x16_t256_w4", &launch_dpc<2, 32, 16, 256, 4>, 0, 0, nullptr, 1},
    {32, 16, 256, 0, 1, "dpc2_f64_32x16_t256_w5", &launch_dpc_default<2, 5>, 0, 0, nullptr, 1},
    {32, 16, 256, 0, 1, "dpc2_f64_32x16_t256_w6", &launch_dpc<2, 32, 16, 256, 6>, 0, 0, nullptr, 1},
};
const Variant kDPC3[] = {
    {32, 16, 256, 0, 1, "dpc3_f64_32x16_t256", &launch_dpc<3, 32, 16, 256>, 0, 0, nullptr, 1},
    {64, 8, 256, 0, 1, "dpc3_f64_64x8_t256", &launch_dpc<3, 64, 8, 256>, 0, 0, nullptr, 1},
    {32, 16, 256, 0, 1, "dpc3_f64_32x16_t256_w4", &launch_dpc_default<3, 4>, 0, 0, nullptr, 1},
    {32, 16, 256, 0, 1, "dpc3_f64_32x16_t256_w5", &launch_dpc<3, 32, 16, 256, 5>, 0, 0, nullptr, 1},
};

}  // namespace

bool dpc_lds_ready(int ns, int halo)
{
    if (ns == 2)
        return dpc_opt_in<2, 32, 16, 256>(halo) && dpc_opt_in<2, 64, 8, 256>(halo) && dpc_opt_in<2, 32, 16, 256, 4>(halo) &&
               dpc_opt_in<2, 32, 16, 256, 5>(halo) && dpc_opt_in<2, 32, 16, 256, 6>(halo) && dpc_opt_in<2, 32, 16, 512>(halo);
    return dpc_opt_in<3, 32, 16, 256>(halo) && dpc_opt_in<3, 64, 8, 256>(halo) && dpc_opt_in<3, 32, 16, 256, 4>(halo) &&
           dpc_opt_in<3, 32, 16, 256, 5>(halo) && dpc_opt_in<3, 32, 16, 512>(halo);
}

const Variant* dpc2_variants_f64(int* n) { *n = (int)(sizeof(kDPC2) / sizeof(kDPC2[0])); return kDPC2; }
const Variant* dpc3_variants_f64(int* n) { *n = (int)(sizeof(kDPC3) / sizeof(kDPC3[0])); return kDPC3; }

}  // namespace tmk
