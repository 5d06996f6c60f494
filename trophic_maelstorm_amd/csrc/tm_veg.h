// tm_veg.h -- the vegetation's Dornic sub-step of the consumer models in FP64: P* of
// every cell of a tile from the old vegetation, the single-species transition on the
// single-species stream (rietkerk_bjork_FKE.cpp:4150-4211, multiSPDP.cpp:2901-2945).
#pragma once
#include "tm_kernels.h"

namespace tmk {

struct VegConst {
    const DornicConst& k;
    uint32_t seed, inst;
    int compat;
    int64_t step;
};

// A cell and its four neighbours (value, up, down, left, right), periodic.
__device__ __forceinline__ uint32_t veg_stencil(const double* __restrict__ P, int L, int y, int x, double (&v)[5])
{
    const uint32_t row = (uint32_t)y * (uint32_t)L, cell = row + (uint32_t)x;
    v[0] = P[cell];
    v[1] = P[(uint32_t)(y == 0 ? L - 1 : y - 1) * (uint32_t)L + (uint32_t)x];
    v[2] = P[(uint32_t)(y == L - 1 ? 0 : y + 1) * (uint32_t)L + (uint32_t)x];
    v[3] = P[row + (uint32_t)(x == 0 ? L - 1 : x - 1)];
    v[4] = P[row + (uint32_t)(x == L - 1 ? 0 : x + 1)];
    return cell;
}

// P* of one cell; FIRST: as dornic_cell_d's first pass.
template <bool FIRST>
__device__ __forceinline__ int veg_update(const VegConst& c, uint32_t cell, const double (&v)[5], double& y)
{
    const double alpha = nbr_alpha(c.k.dc, v[1], v[2], v[3], v[4]);
    y = v[0];
    if (alpha == 0.0 && v[0] == 0.0) {   // absorbing: no draw, +0 where the whole stencil is zero
        if (v[1] == 0.0 && v[2] == 0.0 && v[3] == 0.0 && v[4] == 0.0) y = 0.0;
        return kDornicDone;
    }
    double n;
    if constexpr (FIRST) {
        Stream4 s(c.seed, c.inst, cell, c.step);
        return dornic_cell_d<true, Stream4>(s, alpha, v[0], c.k, c.compat != 0, n, y);
    } else {
        Stream s(c.seed, c.inst, cell, c.step);
        return dornic_cell_d<false, Stream>(s, alpha, v[0], c.k, c.compat != 0, n, y);
    }
}

__device__ __forceinline__ void veg_cell(const VegConst& c, int L, int y, int x, const double* __restrict__ P,
                                         double* __restrict__ Pstar)
{
    double v[5], r;
    const uint32_t cell = veg_stencil(P, L, y, x, v);
    veg_update<false>(c, cell, v, r);
    Pstar[cell] = r;
}

// Appends the lanes whose flag is set to a queue in LDS, upwards from q[0] or (DOWN)
// downwards from q[-1] (one counter add a wave; the order of the waves does not matter
// to the callers).  Every lane of the wave calls it.
template <bool DOWN>
__device__ __forceinline__ void queue_push(bool flag, uint16_t e, uint16_t* q, uint32_t* n)
{
    const uint64_t m = __ballot(flag);
    if (m == 0) return;
    const int lane = threadIdx.x & 63;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(n, (uint32_t)__popcll(m));
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    const int i = (int)(base + (uint32_t)__popcll(m & ((1ull << lane) - 1)));
    if (flag) q[DOWN ? -1 - i : i] = e;
}

// One kVegTX x kVegTY tile by 256 threads (a wave per row, four rows each), in two
// passes as dp_tile_deferred: the cells whose first trials do not settle go to LDS queues
// and are finished densely packed -- those that only miss their Gamma deviate (the
// quantile's tails, 5%) from the shape the first pass left in Pstar, the others from
// their first word.  The cells' neighbours come from the caches.  One cell a thread in
// one pass, a wave runs every path its 64 cells take between them: 16 x 256^2 of the
// Rietkerk model in 36 us, with the chunk sums beside it in 30 here.
constexpr int kVegTX = 64, kVegTY = 16;

// Batches of up to this many 64 x 4 tiles run one cell a thread instead.  us a step, direct /
// two passes, n x 256^2 (256 tiles each, two groups) and one lattice:
//   Rietkerk, 3 species  8: 92 / 96   12: 122 / 124   14: 139 / 135   16: 155 / 150   20: 188 / 183
//                        768^2: 119 / 124   896^2 (3136): 148 / 151   1024^2 (4096): 172 / 172
//   Rietkerk, 2 species  8: 66 / 69   12: 87 / 87   14: 98 / 93   16: 106 / 101   20: 126 / 121
//   DP, 2 species        8: 59 / 62   10: 70 / 70   11: 74 / 75   12: 80 / 76   16: 92 / 88
//                        896^2: 100 / 102   1024^2: 114 / 112
//   DP, 3 species        8: 83 / 88   11: 108 / 114   12: 115 / 117   16: 143 / 138
constexpr int kVegDirectTilesFke = 12 * 256, kVegDirectTilesDpc = 11 * 256;

struct VegLds {
    uint32_t n[2];
    uint16_t q[kVegTX * kVegTY];   // restarts from the front, Gamma deviates from the back
};

__device__ __forceinline__ void veg_tile(const VegConst& c, int L, int x0, int y0, const double* __restrict__ P,
                                         double* __restrict__ Pstar, VegLds& sm)
{
    constexpr int NC = kVegTX * kVegTY;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (threadIdx.x < 2) sm.n[threadIdx.x] = 0u;
    __syncthreads();
#pragma unroll 1
    for (int j = 0; j < kVegTY / 4; ++j) {
        const int ly = 4 * j + w, y = y0 + ly, x = x0 + lane;
        int st = kDornicDone;
        if (y < L && x < L) {
            double v[5], r;
            const uint32_t cell = veg_stencil(P, L, y, x, v);
            st = veg_update<true>(c, cell, v, r);
            if (st != kDornicRestart) Pstar[cell] = r;
        }
        const uint16_t e = (uint16_t)(ly * kVegTX + lane);
        queue_push<false>(st == kDornicRestart, e, sm.q, &sm.n[0]);
        queue_push<true>(st == kDornicGamma, e, sm.q + NC, &sm.n[1]);
    }
    __syncthreads();
    // one list, restarts first: its waves run beside each other, nearly each on one kind
    const uint32_t n0 = sm.n[0], n1 = sm.n[1];
#pragma unroll 1
    for (uint32_t i = threadIdx.x; i < n0 + n1; i += 256) {
        const uint32_t e = i < n0 ? sm.q[i] : sm.q[NC - 1 - (i - n0)];
        const int y = y0 + (int)(e / kVegTX), x = x0 + (int)(e % kVegTX);
        if (i < n0) {
            veg_cell(c, L, y, x, P, Pstar);
        } else {
            const uint32_t cell = (uint32_t)y * (uint32_t)L + (uint32_t)x;
            Stream s(c.seed, c.inst, cell, c.step);
            s.skip(dornic_words(c.k.ll * P[cell], c.compat != 0));
            Pstar[cell] = dornic_gamma_d(s, Pstar[cell], c.k.lambda, c.compat != 0);
        }
    }
}

// An instance's sums from its chunks' (NV doubles each, STRIDE apart), by a wave: lanes
// load 64 chunks at a time and lane f adds value f in chunk order; lane f returns total
// f, and s[f] holds it for all.  With a thread to an instance, loading each chunk as it
// came to it, a step of one three-species Rietkerk consumer lattice took 76 us at 512^2
// (64 chunks) and 207 at 1024^2, 69 and 172 here.
template <int NV, int STRIDE>
__device__ __forceinline__ double chunk_totals(const double* chunk, int n, double (&s)[64 * NV])
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x;
    double t = 0.0;
    for (int c0 = 0; c0 < n; c0 += 64) {
        if (c0 + lane < n) {
#pragma unroll
            for (int f = 0; f < NV; ++f) s[lane * NV + f] = chunk[(int64_t)(c0 + lane) * STRIDE + f];
        }
        __syncthreads();
        if (lane < NV) {
            const int m = n - c0 < 64 ? n - c0 : 64;
#pragma unroll 8
            for (int j = 0; j < m; ++j) t += s[j * NV + lane];
        }
        __syncthreads();
    }
    if (lane < NV) s[lane] = t;
    __syncthreads();
    return t;
}

}  // namespace tmk
