// The HIP names that the library's sources use, for a compiler without a GPU: device code
// becomes host code, a workgroup's threads run as fibers of one thread, and the host API
// works on host memory.  For tests of index arithmetic, of samplers and of host logic.
//
// Barriers, wave operations and LDS (static storage) behave as on the GPU.  Launches run
// at once, unless a test takes them over (cpu_hip::on_launch).
#pragma once
#include <sys/mman.h>
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <string>
#include <tuple>
#include <vector>

#define __HIP_DEVICE_COMPILE__ 1
#define __host__
#define __device__
#define __global__
#define __constant__
#define __shared__ thread_local   /* static storage, shared by the fibers; `extern` ones are the test's to define */
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
struct uint4 { unsigned x, y, z, w; };
struct float4 { float x, y, z, w; };
struct alignas(16) double2 { double x, y; };
struct alignas(16) double4 { double x, y, z, w; };
inline int2 make_int2(int x, int y) { return {x, y}; }
inline int4 make_int4(int x, int y, int z, int w) { return {x, y, z, w}; }
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline double2 make_double2(double x, double y) { return {x, y}; }
inline double4 make_double4(double x, double y, double z, double w) { return {x, y, z, w}; }
using std::max;
using std::min;

inline thread_local dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace cpu_hip {

// A workgroup: every fiber runs until it ends or waits.  The wave votes inside samplers
// (__builtin_amdgcn_ballot_w64) are in branches that some lanes do not take: each is done
// first, among the lanes that wait for it.  The other wave operations are where a wave is
// whole again: done once all its lanes that have not ended wait for one.  A barrier is
// done once every lane of the workgroup that has not ended waits for it.
enum Wait { kRun, kBarrier, kVote, kWave, kDone };
struct Lane {
    ucontext_t ctx;
    Wait wait;
    uint64_t in;
};
// What the lanes of a wave brought to its last collective.
struct WaveVals {
    uint64_t mask, v[64];
};
struct Group {
    ucontext_t main;
    std::vector<Lane> lanes;
    std::vector<WaveVals> waves;
    unsigned cur = 0;
    std::function<void()> body;
};
inline thread_local Group* group = nullptr;

inline void yield(Wait w)
{
    Lane& l = group->lanes[group->cur];
    l.wait = w;
    swapcontext(&l.ctx, &group->main);
}
inline void lane_main()
{
    group->body();
    group->lanes[group->cur].wait = kDone;
}
// This lane's value to the wave; what all of them brought.  Valid until the next one.
inline const WaveVals& collective(uint64_t v, Wait kind = kWave)
{
    group->lanes[group->cur].in = v;
    yield(kind);
    return group->waves[group->cur / 64];
}
inline uint64_t votes(bool v, Wait kind)
{
    const WaveVals& w = collective(v ? 1 : 0, kind);
    uint64_t b = 0;
    for (int i = 0; i < 64; ++i) b |= (w.mask >> i & 1 & w.v[i]) << i;
    return b;
}
inline int lane() { return (int)(group->cur % 64); }
// The lane a DPP move reads from, or -1 (quad_perm, row_shl, row_shr, row_ror, mirrors, broadcasts).
inline int dpp_from(int ctrl, int l)
{
    const int row = l & ~15, i = l & 15, n = ctrl & 15;
    if (ctrl < 0x100) return (l & ~3) + (ctrl >> 2 * (l & 3) & 3);
    if (ctrl < 0x110) return i + n < 16 ? l + n : -1;
    if (ctrl < 0x120) return i - n >= 0 ? l - n : -1;
    if (ctrl < 0x130) return row + ((i - n) & 15);
    if (ctrl == 0x140) return row + 15 - i;
    if (ctrl == 0x141) return (l & ~7) + 7 - (l & 7);
    if (ctrl == 0x142) return row - 1;
    if (ctrl == 0x143) return l >= 32 ? 31 : -1;
    fprintf(stderr, "DPP control %#x\n", ctrl);
    abort();
}
inline int update_dpp(int old, int src, int ctrl, int rows, int banks, bool)
{
    const WaveVals& w = collective((uint32_t)src);
    const int l = lane(), from = dpp_from(ctrl, l);
    if (!(rows >> l / 16 & 1) || !(banks >> l % 16 / 4 & 1) || from < 0 || !(w.mask >> from & 1)) return old;
    return (int)(uint32_t)w.v[from];
}
struct Pair {
    uint32_t v[2];
    uint32_t operator[](int i) const { return v[i]; }
};
// Upper n lanes of each 2 n of x against the lower n of y.
inline Pair permlane_swap(int n, uint32_t x, uint32_t y)
{
    const WaveVals& w = collective((uint64_t)y << 32 | x);
    const int l = lane();
    return l & n ? Pair{{(uint32_t)(w.v[l - n] >> 32), y}} : Pair{{x, (uint32_t)w.v[l + n]}};
}

constexpr size_t kStack = 128 << 10;

inline void run_workgroup(dim3 grid, dim3 block, dim3 at, std::function<void()> body)
{
    Group g;
    const unsigned n = block.x;
    g.lanes.resize(n);
    g.waves.resize((n + 63) / 64);
    g.body = std::move(body);
    char* stacks = (char*)mmap(nullptr, kStack * n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (stacks == MAP_FAILED) abort();
    for (unsigned i = 0; i < n; ++i) {
        Lane& l = g.lanes[i];
        l.wait = kRun;
        getcontext(&l.ctx);
        l.ctx.uc_stack.ss_sp = stacks + kStack * i;
        l.ctx.uc_stack.ss_size = kStack;
        l.ctx.uc_link = &g.main;
        makecontext(&l.ctx, lane_main, 0);
    }
    group = &g;
    gridDim = grid;
    blockDim = block;
    blockIdx = at;
    for (;;) {
        for (unsigned i = 0; i < n; ++i)
            if (g.lanes[i].wait == kRun) {
                g.cur = i;
                threadIdx = dim3(i, 0, 0);
                swapcontext(&g.main, &g.lanes[i].ctx);
            }
        bool any = false, barrier = true;
        for (unsigned w = 0; w < n; w += 64) {
            WaveVals& wave = g.waves[w / 64];
            bool waits[kDone + 1] = {};
            const unsigned end = w + 64 < n ? w + 64 : n;
            for (unsigned i = w; i < end; ++i) waits[g.lanes[i].wait] = true;
            any = any || waits[kBarrier] || waits[kVote] || waits[kWave];
            barrier = barrier && !waits[kVote] && !waits[kWave];
            if (!waits[kVote] && waits[kWave] && waits[kBarrier]) {
                fprintf(stderr, "wave %u: some lanes wait for the wave, some for the workgroup\n", w / 64);
                abort();
            }
            const Wait kind = waits[kVote] ? kVote : kWave;
            if (!waits[kind]) continue;
            wave.mask = 0;
            for (unsigned i = w; i < end; ++i) {
                Lane& l = g.lanes[i];
                if (l.wait != kind) continue;
                wave.mask |= 1ull << (i - w);
                wave.v[i - w] = l.in;
                l.wait = kRun;
            }
        }
        if (!any) break;
        if (barrier)
            for (Lane& l : g.lanes)
                if (l.wait == kBarrier) l.wait = kRun;
    }
    group = nullptr;
    munmap(stacks, kStack * n);
}

// Set by a test to see launches, and to run them or not.
struct Launch {
    const char* name;
    const void* kernel;
    dim3 grid, block;
    size_t lds;      // dynamic
    void* stream;
    std::function<void()> run;
};
inline std::function<void(const Launch&)> on_launch;

template <class... P, class... A>
void launch(const char* name, void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, void* stream, A&&... args)
{
    const std::tuple<std::decay_t<P>...> values(std::forward<A>(args)...);   // as they are now
    const std::function<void()> body = [=]() { std::apply(kernel, values); };
    auto run = [=]() {
        for (unsigned z = 0; z < grid.z; ++z)
            for (unsigned y = 0; y < grid.y; ++y)
                for (unsigned x = 0; x < grid.x; ++x) run_workgroup(grid, block, dim3(x, y, z), body);
    };
    if (on_launch) on_launch(Launch{name, (const void*)kernel, grid, block, lds, stream, run});
    else run();
}

}  // namespace cpu_hip

inline void __syncthreads() { cpu_hip::yield(cpu_hip::kBarrier); }
inline uint64_t __ballot(int v) { return cpu_hip::votes(v != 0, cpu_hip::kWave); }
inline int cpu_readfirstlane(int v)
{
    const cpu_hip::WaveVals& w = cpu_hip::collective((uint32_t)v);
    return (int)(uint32_t)w.v[__builtin_ctzll(w.mask)];
}
inline void __threadfence_system() {}
inline double __shfl_xor(double v, int m)
{
    uint64_t b;
    std::memcpy(&b, &v, 8);
    b = cpu_hip::collective(b).v[cpu_hip::lane() ^ m];
    std::memcpy(&v, &b, 8);
    return v;
}
inline int __popcll(uint64_t v) { return __builtin_popcountll(v); }
inline float __uint_as_float(uint32_t v) { float f; std::memcpy(&f, &v, 4); return f; }
inline uint32_t __float_as_uint(float f) { uint32_t v; std::memcpy(&v, &f, 4); return v; }
inline int64_t __double_as_longlong(double d) { int64_t v; std::memcpy(&v, &d, 8); return v; }
inline double __longlong_as_double(int64_t v) { double d; std::memcpy(&d, &v, 8); return d; }
inline int __double2loint(double d) { return (int)(uint32_t)__double_as_longlong(d); }
inline int __double2hiint(double d) { return (int)(__double_as_longlong(d) >> 32); }
inline double __hiloint2double(int h, int l) { return __longlong_as_double((int64_t)((uint64_t)(uint32_t)h << 32 | (uint32_t)l)); }
template <typename T> T atomicAdd(T* p, T v) { const T o = *p; *p = o + v; return o; }
template <typename T> T atomicMin(T* p, T v) { const T o = *p; if (v < o) *p = v; return o; }
inline uint64_t cpu_hip_clock = 0;
inline long long wall_clock64() { return (long long)(cpu_hip_clock += 100); }

// v_log_f32 (base 2) and v_rcp_f32 are good to an ulp; a test may move them by that.
inline int cpu_hip_ulp = 0;
inline float cpu_nudge(float x)
{
    if (!(x != 0.0f) || !std::isfinite(x)) return x;
    return cpu_hip_ulp > 0 ? std::nextafterf(x, INFINITY) : (cpu_hip_ulp < 0 ? std::nextafterf(x, -INFINITY) : x);
}

#define __builtin_amdgcn_bitop3_b32(a, b, c, t) ((uint32_t)(a) ^ (uint32_t)(b) ^ (uint32_t)(c))   /* table 0x96 */
#define __builtin_amdgcn_alignbit(hi, lo, s) ((uint32_t)(((uint64_t)(hi) << 32 | (uint32_t)(lo)) >> ((s) & 31u)))
#define __builtin_amdgcn_logf(x) cpu_nudge((float)std::log2((double)(float)(x)))
#define __builtin_amdgcn_rcpf(x) cpu_nudge((float)(1.0 / (double)(float)(x)))
#define __builtin_amdgcn_sqrtf(x) cpu_nudge((float)std::sqrt((double)(float)(x)))
#define __builtin_amdgcn_rsqf(x) cpu_nudge((float)(1.0 / std::sqrt((double)(float)(x))))
#define __builtin_amdgcn_exp2f(x) cpu_nudge((float)std::exp2((double)(float)(x)))
#define __builtin_amdgcn_readfirstlane(x) cpu_readfirstlane(x)
#define __builtin_amdgcn_ballot_w64(x) cpu_hip::votes(x, cpu_hip::kVote)
#define __builtin_amdgcn_s_waitcnt(x) ((void)0)
#define __builtin_amdgcn_s_sleep(x) ((void)0)
#define __builtin_amdgcn_update_dpp(old, src, ...) cpu_hip::update_dpp(old, src, __VA_ARGS__)
#define __builtin_amdgcn_permlane32_swap(x, y, ...) cpu_hip::permlane_swap(32, (uint32_t)(x), (uint32_t)(y))
#define __builtin_amdgcn_permlane16_swap(x, y, ...) cpu_hip::permlane_swap(16, (uint32_t)(x), (uint32_t)(y))
// each lane's bytes land behind the wave's LDS base
#define __builtin_amdgcn_global_load_lds(src, lds, n, ...) std::memcpy((char*)(lds) + (threadIdx.x & 63) * (n), (src), (n))
#ifndef __HIP_MEMORY_SCOPE_SYSTEM
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#endif
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n((p), (v), (order))

// ---- host API ------------------------------------------------------------------------
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999, hipErrorNotReady = 600 };
typedef void* hipGraph_t;
typedef void* hipGraphExec_t;
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum hipStreamCaptureMode { hipStreamCaptureModeThreadLocal };
struct hipDeviceProp_t { char gcnArchName[16]; int multiProcessorCount; };
enum { hipHostMallocDefault = 0, hipStreamNonBlocking = 1, hipEventDisableTiming = 2 };
enum hipDeviceAttribute_t { hipDeviceAttributeWallClockRate };
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize };
struct hipFuncAttributes { size_t sharedSizeBytes; };

namespace cpu_hip {
inline std::function<void(const char*, const void*)> on_call;   // (function, pointer it is about)
inline std::function<hipError_t(hipStream_t)> on_query;          // hipStreamQuery, hipStreamSynchronize
inline std::function<bool(size_t)> refuse;                       // device allocations of a size
inline std::function<size_t(const void*)> static_lds;            // of a kernel
inline std::function<hipError_t(const void*, int)> on_opt_in;    // to dynamic LDS above the default limit
inline int device = 0;
inline void called(const char* f, const void* p = nullptr) { if (on_call) on_call(f, p); }
}  // namespace cpu_hip

inline const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
inline hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)
{
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
inline hipError_t hipGetDevice(int* d) { *d = cpu_hip::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { cpu_hip::device = d; return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n)
{
    if (cpu_hip::refuse && cpu_hip::refuse(n)) return hipErrorOutOfMemory;
    *p = calloc(n, 1); 
    cpu_hip::called("hipMalloc", *p);
    return hipSuccess;
}
inline hipError_t hipFree(void* p) { cpu_hip::called("hipFree", p); free(p); return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(n, 1); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
template <typename T> hipError_t hipMalloc(T** p, size_t n) { return hipMalloc((void**)p, n); }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
inline hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, hipStream_t)
{
    for (size_t i = 0; i < h; ++i) std::memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    return hipSuccess;
}
// no capture here: what asks for it is told so
inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorUnknown; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, void*, void*, size_t) { return hipErrorUnknown; }
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
#define HIP_SYMBOL(x) (&(x))
inline hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = (void*)s; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = malloc(1); cpu_hip::called("hipStreamCreate", *s); return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t s) { cpu_hip::called("hipStreamDestroy", s); free(s); return hipSuccess; }
inline hipError_t hipStreamQuery(hipStream_t s) { return cpu_hip::on_query ? cpu_hip::on_query(s) : hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { return cpu_hip::on_query ? cpu_hip::on_query(s) : hipSuccess; }
inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) { cpu_hip::called("hipStreamWaitEvent", e); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = malloc(1); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t* e) { *e = malloc(1); return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void* f)
{
    a->sharedSizeBytes = cpu_hip::static_lds ? cpu_hip::static_lds(f) : 0;
    return hipSuccess;
}
inline hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int v)
{
    return cpu_hip::on_opt_in ? cpu_hip::on_opt_in(f, v) : hipSuccess;
}
inline hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }

#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    cpu_hip::launch(#kernel, (kernel), (grid), (block), (lds), (stream), __VA_ARGS__)
