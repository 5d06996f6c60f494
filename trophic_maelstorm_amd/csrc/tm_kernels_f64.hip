// tm_kernels_f64.hip -- FP64 instantiations of the step kernels, plus the
// precision-independent rho(t) combine.  Compiled with -ffp-contract=off so
// every FP64 operation rounds exactly as the CPU restatement's does.
#define TM_DEFINE_COMBINE
#include "tm_launch.h"

#include <algorithm>

namespace tmk {

template <typename T, int TX, int TY, int NT, int MODE = 0, int MINW = 1, int Q = 0>
static void launch_dp(const StepArgs& a, int grid, hipStream_t s)
{
    hipLaunchKernelGGL((dp_step_kernel<T, TX, TY, NT, MODE, MINW, Q>), dim3(grid), dim3(NT), 0, s, a);
}

template <typename T, int TX, int TY, int NT, int K, int MINW = 1>
static void launch_dpk(const StepArgs& a, int grid, hipStream_t s)
{
    hipLaunchKernelGGL((dp_stepk_kernel<T, TX, TY, NT, K, MINW>), dim3(grid), dim3(NT), 0, s, a);
}

// The default's single step: a workgroup per part of a tile (dp_part_kernel) for batches of
// up to 1280 tiles, the two-pass tile kernel above.  us a step, parts / tiles: 8.8 / 31.1 at
// 64 tiles (8 x 128^2); as two groups of n x 128^2 24.9 / 35.7 at 512, 46.9 / 47.6 at 1024,
// 54.9 / 56.0 at 1200, 60.0 / 59.7 at 1312, 70.3 / 65.8 at 1536, 93.3 / 86.1 at 2048.  One large
// lattice is one group, and parts hold longer there: 51.8 / 60.3 at 1012 (1408^2), 64.0 / 73.9
// at 1250, 99.6 / 103.8 at 2048.
static void launch_dp_default(const StepArgs& a, int grid, hipStream_t s)
{
    if (a.ptiles <= 1280)
        hipLaunchKernelGGL((dp_part_kernel<double, 64, 32, 1>), dim3(4 * a.ntiles), dim3(512), 0, s, a);
    else
        launch_dp<double, 64, 32, 256, 0, 6, 1>(a, grid, s);
}

template <typename T, int TX, int TY, int NT, bool SPLIT = false>
static void launch_rk(const StepArgs& a, int grid, hipStream_t s)
{
    hipLaunchKernelGGL((rk_step_kernel<T, TX, TY, NT, SPLIT>), dim3(grid), dim3(NT), 0, s, a);
}

static const Variant kDP[] = {
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256", &launch_dp<double, 64, 32, 256>},
    {128, 32, 256, 0, 4, "dp_f64_128x32_t256", &launch_dp<double, 128, 32, 256>},
    {64, 64, 256, 0, 4, "dp_f64_64x64_t256", &launch_dp<double, 64, 64, 256>},
    {256, 32, 256, 0, 4, "dp_f64_256x32_t256", &launch_dp<double, 256, 32, 256>},
    // _xK: K steps per launch (temporal blocking); the single-step kernel of the same
    // tile covers a block's last steps when fewer than K remain
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x2", &launch_dpk<double, 64, 32, 256, 2>, 0, 0, nullptr, 0, 2,
     &launch_dp<double, 64, 32, 256>},
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x4", &launch_dpk<double, 64, 32, 256, 4>, 0, 0, nullptr, 0, 4,
     &launch_dp<double, 64, 32, 256>},
    {64, 16, 256, 0, 4, "dp_f64_64x16_t256_x4", &launch_dpk<double, 64, 16, 256, 4>, 0, 0, nullptr, 0, 4,
     &launch_dp<double, 64, 16, 256>},
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x8", &launch_dpk<double, 64, 32, 256, 8>, 0, 0, nullptr, 0, 8,
     &launch_dp<double, 64, 32, 256>},
    {64, 8, 128, 0, 2, "dp_f64_64x8_t128_x16", &launch_dpk<double, 64, 8, 128, 16>, 0, 0, nullptr, 0, 16,
     &launch_dp<double, 64, 8, 128>},
    // _xKa: adaptive -- single steps while more than the given per-mille of the cells are
    // occupied, K-step launches below
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x4a", &launch_dpk<double, 64, 32, 256, 4>, 0, 0, nullptr, 0, 4,
     &launch_dp<double, 64, 32, 256>, 20},
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x8a", &launch_dpk<double, 64, 32, 256, 8>, 0, 0, nullptr, 0, 8,
     &launch_dp<double, 64, 32, 256>, 20},
    // _q: the single steps defer cells whose Gamma trial is rejected to a second
    // pass over a queue in LDS (dp_tile_deferred)
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x8aq", &launch_dpk<double, 64, 32, 256, 8>, 0, 0, nullptr, 0, 8,
     &launch_dp<double, 64, 32, 256, 0, 1, 1>, 20},
    // _w6 (the default): its single step bounded to 80 VGPRs (six waves per SIMD), and
    // by parts on small batches
    {64, 32, 256, 0, 4, "dp_f64_64x32_t256_x8aq_w6", &launch_dpk<double, 64, 32, 256, 8>, 0, 0, nullptr, 0, 8,
     &launch_dp_default, 20},
};

template <typename T, int FX, int FY, bool SPLIT>
static void launch_frame(const StepArgs& a, int grid, hipStream_t s)
{
    hipLaunchKernelGGL((rk_frame_kernel<T, FX, FY, SPLIT>), dim3(grid), dim3(FX * FY), 0, s, a);
}

static const Variant kRK[] = {
    {16, 16, 256, 0, 1, "rk_f64_16x16_t256", &launch_rk<double, 16, 16, 256>},
    {32, 16, 256, 0, 1, "rk_f64_32x16_t256", &launch_rk<double, 32, 16, 256>},
    {32, 32, 256, 0, 1, "rk_f64_32x32_t256", &launch_rk<double, 32, 32, 256>},
    // split step: Dornic kernel (dp_step_kernel MODE 1) on 64 x 32 tiles, then the RK4 kernel
    {16, 16, 256, 0, 1, "rk_f64_split_16x16_t256", &launch_rk<double, 16, 16, 256, true>, 64, 32,
     &launch_dp<double, 64, 32, 256, 1>},
    {32, 16, 256, 0, 1, "rk_f64_split_32x16_t256", &launch_rk<double, 32, 16, 256, true>, 64, 32,
     &launch_dp<double, 64, 32, 256, 1>},
    {32, 32, 256, 0, 1, "rk_f64_split_32x32_t256", &launch_rk<double, 32, 32, 256, true>, 64, 32,
     &launch_dp<double, 64, 32, 256, 1>},
    // _q16: the Dornic kernel in two passes (dp_tile_deferred) on 64 x 16 tiles at 80
    // VGPRs.  16 x 512^2, Dornic and RK4 together: 163 us a step, one-pass 64 x 32
    // tiles 202; other tiles (64 x 8, 64 x 32, 128 x 16) and bounds 166 to 178.
    {32, 16, 256, 0, 1, "rk_f64_split_32x16_t256_q16", &launch_rk<double, 32, 16, 256, true>, 64, 16,
     &launch_dp<double, 64, 16, 256, 1, 6, 1>},
    // frame_FXxFY: a thread per cell of the frame around a tile 6 narrower and shorter
    // (rk_frame_kernel), fused for small batches, split with the two-pass Dornic kernel
    {26, 26, 1024, 0, 1, "rk_f64_frame_32x32", &launch_frame<double, 32, 32, false>},
    {26, 10, 512, 0, 1, "rk_f64_frame_32x16", &launch_frame<double, 32, 16, false>},
    {26, 10, 512, 0, 1, "rk_f64_split_frame_32x16", &launch_frame<double, 32, 16, true>, 64, 16,
     &launch_dp<double, 64, 16, 256, 1, 6, 1>},
    {10, 10, 256, 0, 1, "rk_f64_frame_16x16", &launch_frame<double, 16, 16, false>},
    {26, 18, 768, 0, 1, "rk_f64_frame_32x24", &launch_frame<double, 32, 24, false>},
};

const Variant* dp_variants_f64(int* n) { *n = (int)(sizeof(kDP) / sizeof(kDP[0])); return kDP; }
const Variant* rk_variants_f64(int* n) { *n = (int)(sizeof(kRK) / sizeof(kRK[0])); return kRK; }

void launch_measure_f64(int nf, const DevInst* inst, const DevTile* tiles, int ntiles, int tx, int ty,
                        const void* fields, double2* partials, hipStream_t s)
{
    if (nf == 1)
        hipLaunchKernelGGL((measure_kernel<double, 1>), dim3(ntiles), dim3(256), 0, s, inst, tiles, ntiles, tx,
                           ty, (const double*)fields, partials);
    else if (nf == 3)
        hipLaunchKernelGGL((measure_kernel<double, 3>), dim3(ntiles), dim3(256), 0, s, inst, tiles, ntiles, tx,
                           ty, (const double*)fields, partials);
    else if (nf == 5)
        hipLaunchKernelGGL((measure_kernel<double, 5>), dim3(ntiles), dim3(256), 0, s, inst, tiles, ntiles, tx,
                           ty, (const double*)fields, partials);
    else
        hipLaunchKernelGGL((measure_kernel<double, 7>), dim3(ntiles), dim3(256), 0, s, inst, tiles, ntiles, tx,
                           ty, (const double*)fields, partials);
}

void launch_combine(const CombineArgs& a, int n_inst, int nsteps, hipStream_t s)
{
    hipLaunchKernelGGL(combine_rows_kernel, dim3(n_inst, nsteps), dim3(256), 0, s, a);
}

void launch_prep(int model, const DevInst* inst, const void* params, const DevState* state, int n_inst,
                 int nsteps, void* table, hipStream_t s)
{
    const int64_t n = (int64_t)n_inst * nsteps;
    const int grid = (int)((n + 255) / 256);
    if (model == TM_MODEL_DP)
        hipLaunchKernelGGL(prep_consts_kernel<TM_MODEL_DP>, dim3(grid), dim3(256), 0, s, inst, params, state,
                           n_inst, nsteps, table);
    else if (model == TM_MODEL_DP2 || model == TM_MODEL_DP3)
        hipLaunchKernelGGL(prep_consts_kernel<TM_MODEL_DP2>, dim3(grid), dim3(256), 0, s, inst, params, state,
                           n_inst, nsteps, table);
    else if (model == TM_MODEL_FKE2 || model == TM_MODEL_FKE3)
        hipLaunchKernelGGL(prep_consts_kernel<TM_MODEL_FKE2>, dim3(grid), dim3(256), 0, s, inst, params, state,
                           n_inst, nsteps, table);
    else
        hipLaunchKernelGGL(prep_consts_kernel<TM_MODEL_RIETKERK>, dim3(grid), dim3(256), 0, s, inst, params,
                           state, n_inst, nsteps, table);
}

void launch_bump(DevState* state, int n, hipStream_t s)
{
    hipLaunchKernelGGL(bump_counter_kernel, dim3(1), dim3(64), 0, s, state, n);
}

void launch_reset(DevState* state, hipStream_t s)
{
    hipLaunchKernelGGL(reset_state_kernel, dim3(1), dim3(64), 0, s, state);
}

void launch_pack_rows(const double* rows, int64_t rows_cap, int w, int64_t n, int n_inst, double* out, hipStream_t s)
{
    const int64_t total = n * w * n_inst;
    hipLaunchKernelGGL(pack_rows_kernel, dim3((unsigned)std::min<int64_t>(256, (total + 255) / 256)), dim3(256), 0, s,
                       rows, rows_cap, w, n, total, out);
}

size_t const_size(int model)
{
    if (model == TM_MODEL_DP) return sizeof(DPConst);
    if (model == TM_MODEL_DP2 || model == TM_MODEL_DP3) return sizeof(DPCConst);
    return sizeof(RKConstD);
}

}  // namespace tmk
