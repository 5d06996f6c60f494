// Every access of the per-tile step kernels on lattices of any side, on the CPU
// (cpu_hip): the kernel runs on the first and the last tile of the lattice over sparse
// memory in which only the lattice's fields exist to be read and only the tile's pages to
// be written.  A cell of the tile left out, one written outside it, or an access past the
// fields ends the program with an error.
#include <csignal>
#include <string>
#include <unistd.h>

#include "tm_kernels.h"
#include "tm_veg.h"

using namespace tmk;

static char what[256];

static void on_fault(int, siginfo_t* i, void*)
{
    char b[320];
    const int n = snprintf(b, sizeof(b), "%s: access outside the fields at %p\n", what, i->si_addr);
    (void)!write(2, b, (size_t)n);
    _exit(1);
}

// n elements that can be read (zeros), between pages that cannot.
template <typename T>
struct Sparse {
    static constexpr size_t kPage = 4096, kGuard = 1 << 20;
    char* map;
    size_t bytes;
    T* p;
    Sparse(size_t n, int prot) : bytes((n * sizeof(T) + kPage - 1) & ~(kPage - 1))
    {
        map = (char*)mmap(nullptr, bytes + 2 * kGuard, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (map == MAP_FAILED) { perror("mmap"); _exit(2); }
        if (prot != PROT_NONE) mprotect(map + kGuard, bytes, prot);
        p = (T*)(map + kGuard);
    }
    ~Sparse() { munmap(map, bytes + 2 * kGuard); }
    // the pages of elements i .. i + n - 1
    T* page(size_t i) { return (T*)((uintptr_t)(p + i) & ~(uintptr_t)(kPage - 1)); }
    void open(size_t i, size_t n)
    {
        T* b = page(i);
        if (mprotect(b, (char*)(p + i + n) - (char*)b, PROT_READ | PROT_WRITE) != 0) { perror("mprotect"); _exit(2); }
    }
};

template <typename T> constexpr T kUnwritten = (T)-7;

// `out` holds nf fields of N cells; the tile's pages are writable and unwritten.
template <typename T>
void prepare_out(Sparse<T>& out, int nf, int64_t L, int x0, int y0, int w, int h)
{
    for (int f = 0; f < nf; ++f)
        for (int y = y0; y < y0 + h; ++y) {
            const size_t i = (size_t)(f * L * L + y * L + x0);
            out.open(i, (size_t)w);
            for (T* q = out.page(i); q < out.page(i + (size_t)w - 1) + 4096 / sizeof(T); ++q) *q = kUnwritten<T>;
        }
}
template <typename T>
bool check_out(Sparse<T>& out, int nf, int64_t L, int x0, int y0, int w, int h)
{
    for (int f = 0; f < nf; ++f)
        for (int y = y0; y < y0 + h; ++y) {
            const size_t i = (size_t)(f * L * L + y * L + x0);
            for (int x = 0; x < w; ++x)
                if (out.p[i + x] == kUnwritten<T>) {
                    fprintf(stderr, "%s: field %d, cell (%d, %d) not written\n", what, f, y, x0 + x);
                    return false;
                }
            for (T* q = out.page(i); q < out.page(i + (size_t)w - 1) + 4096 / sizeof(T); ++q) {
                const int64_t j = q - out.p - (int64_t)f * L * L;   // cell in this field
                const bool own = j >= 0 && j < L * L && j % L >= x0 && j % L < x0 + w && j / L >= y0 && j / L < y0 + h;
                // on small lattices a page holds cells of other fields too
                const int64_t g = q - out.p;
                const int64_t c = g >= 0 ? g % (L * L) : -1;
                const bool other = g >= 0 && g < nf * L * L && c % L >= x0 && c % L < x0 + w && c / L >= y0 && c / L < y0 + h;
                if (!own && !other && *q != kUnwritten<T>) {
                    fprintf(stderr, "%s: element %lld written outside the tile\n", what, (long long)g);
                    return false;
                }
            }
        }
    return true;
}

// One workgroup (or `wgs` of them) of `kernel` on the tile at (x0, y0) of a lattice of side L.
// nf_in, nf_out: fields of `in` and of what is written (out, or aux with AUX).
template <typename T, bool AUX, class Const, class K>
bool run_tile(const char* name, K kernel, int nt, int wgs, int TX, int TY, int nf_in, int nf_out, const Const& c,
              int64_t L, int x0, int y0)
{
    snprintf(what, sizeof(what), "%s, side %lld, tile (%d, %d)", name, (long long)L, y0, x0);
    const int w = (int)min<int64_t>(TX, L - x0), h = (int)min<int64_t>(TY, L - y0);
    Sparse<T> in((size_t)(nf_in * L * L), PROT_READ);
    Sparse<T> out((size_t)(nf_out * L * L), PROT_NONE), pstar((size_t)(L * L), PROT_READ);
    Sparse<int64_t> draws((size_t)(L * L), PROT_NONE);
    prepare_out(out, nf_out, L, x0, y0, w, h);
    prepare_out(draws, 1, L, x0, y0, w, h);
    in.open((size_t)(y0 * L + x0), 1);   // a live cell, so that nothing is skipped as absorbing
    in.p[y0 * L + x0] = (T)20;
    if (!AUX) {
        pstar.open((size_t)(y0 * L + x0), 1);
        pstar.p[y0 * L + x0] = (T)20;
    }
    const bool records = !(nf_in == 3 && nf_out == 3 && std::string(name).find("split") != std::string::npos);

    DevInst di{};
    di.L = (int32_t)L;
    di.ntiles = 1;
    di.seed = 3;
    DevTile tl{0, x0, y0, (int32_t)L, 0};
    DevState st{};
    for (Fault& f : st.fault) f = Fault{~0ull, ~0ull};
    std::vector<double2> partials(64);
    StepArgs a{};
    a.inst = &di;
    a.tiles = a.tiles_a = &tl;
    a.consts = &c;
    a.in = in.p;
    a.out = AUX ? nullptr : out.p;
    a.aux = AUX ? (void*)out.p : (void*)pstar.p;
    a.partials = partials.data();
    a.state = &st;
    a.draws = records ? draws.p : nullptr;
    a.ntiles = a.ntiles_a = a.ptiles = 1;
    a.nslots = 1;
    a.n_inst = 1;
    a.fault = st.fault;
    for (int b = 0; b < wgs; ++b)
        cpu_hip::run_workgroup(dim3((unsigned)wgs), dim3((unsigned)nt), dim3((unsigned)b), [&]() { kernel(a); });
    if (!(out.p[y0 * L + x0] > (T)0)) {   // 20 does not die out in a step: another cell was read
        fprintf(stderr, "%s: the tile's first cell was not read\n", what);
        return false;
    }
    return check_out(out, nf_out, L, x0, y0, w, h) && (!records || check_out(draws, 1, L, x0, y0, w, h));
}

template <typename T, bool AUX, class Const, class K>
bool run(const char* name, K kernel, int nt, int wgs, int TX, int TY, int nf_in, int nf_out, const Const& c, int64_t L)
{
    const int xl = (int)((L - 1) / TX * TX), yl = (int)((L - 1) / TY * TY);
    return run_tile<T, AUX>(name, kernel, nt, wgs, TX, TY, nf_in, nf_out, c, L, 0, 0) &&
           run_tile<T, AUX>(name, kernel, nt, wgs, TX, TY, nf_in, nf_out, c, L, xl, yl);
}

// The vegetation's sub-step of the consumer models: by tile, and by cell.
bool run_veg(const RKConstD& c, int64_t L, bool cells)
{
    const int TX = kVegTX, TY = cells ? 4 : kVegTY;
    for (int last = 0; last < 2; ++last) {
        const int x0 = last ? (int)((L - 1) / TX * TX) : 0, y0 = last ? (int)((L - 1) / TY * TY) : 0;
        snprintf(what, sizeof(what), "veg_%s, side %lld, tile (%d, %d)", cells ? "cell" : "tile", (long long)L, y0, x0);
        const int w = (int)min<int64_t>(TX, L - x0), h = (int)min<int64_t>(TY, L - y0);
        Sparse<double> in((size_t)(L * L), PROT_READ), out((size_t)(L * L), PROT_NONE);
        prepare_out(out, 1, L, x0, y0, w, h);
        in.open((size_t)(y0 * L + x0), 1);
        in.p[y0 * L + x0] = 20.0;
        cpu_hip::run_workgroup(dim3(1), dim3(256), dim3(0), [&]() {
            static VegLds sm;
            const VegConst vc = {c.k, 3u, 0u, 0, 0};
            const int y = y0 + (int)(threadIdx.x >> 6), x = x0 + (int)(threadIdx.x & 63);
            if (!cells) veg_tile(vc, (int)L, x0, y0, in.p, out.p, sm);
            else if (y < L && x < L) veg_cell(vc, (int)L, y, x, in.p, out.p);
        });
        if (!check_out(out, 1, L, x0, y0, w, h) || !(out.p[y0 * L + x0] > 0.0)) return false;
    }
    return true;
}

// kernel_indices frame|part|tile|veg SIDE...
int main(int argc, char** argv)
{
    struct sigaction sa = {};
    sa.sa_sigaction = on_fault;
    sa.sa_flags = SA_SIGINFO;
    sigaction(SIGSEGV, &sa, nullptr);
    sigaction(SIGBUS, &sa, nullptr);

    tm_rietkerk_params rp{};
    rp.c = 10; rp.gmax = 0.05; rp.alpha = 0.2; rp.rW = 0.2; rp.d = 0.25; rp.K[1] = 5; rp.K[2] = 5; rp.W0 = 0.2; rp.R = 1;
    rp.D[0] = 0.1; rp.D[1] = 0.1; rp.D[2] = 100; rp.sigma = 0.01; rp.dt = 0.001; rp.dx = 2;
    const RKConstD rk = rk_constants(rp, 0);
    tm_dp_params dpp{};
    dpp.a = 0.9; dpp.b = 0.2; dpp.D = 0.04; dpp.sigma = 1.4; dpp.dt = 0.1; dpp.dx = 1;
    const DPConst dp = dp_constants(dpp, 0);
    bool ok = true;
    auto frame = [&](auto t, auto fx, auto fy, auto split, int64_t L) {
        typedef decltype(t) T;
        constexpr int FX = decltype(fx)::value, FY = decltype(fy)::value;
        constexpr bool S = decltype(split)::value;
        const std::string n = std::string(S ? "split " : "") + "frame " + std::to_string(FX) + "x" + std::to_string(FY) +
                              (sizeof(T) == 8 ? " f64" : " f32");
        ok = ok && run<T, false>(n.c_str(), rk_frame_kernel<T, FX, FY, S>, FX * FY, 1, FX - 6, FY - 6, 3, 3, rk, L);
    };
    using std::integral_constant;
    const std::string only = argc > 1 ? argv[1] : "";
    for (int k = 2; k < argc && ok; ++k) {
        const int64_t L = atoll(argv[k]);
        if (only == "frame") {
            integral_constant<int, 16> c16;
            integral_constant<int, 24> c24;
            integral_constant<int, 32> c32;
            std::false_type fused;
            std::true_type split;
            frame(0.0, c16, c16, fused, L);
            frame(0.0, c32, c16, fused, L);
            frame(0.0, c32, c24, fused, L);
            frame(0.0, c32, c32, fused, L);
            frame(0.0, c32, c16, split, L);
            frame(0.0f, c16, c16, fused, L);
            frame(0.0f, c32, c16, fused, L);
            frame(0.0f, c32, c24, fused, L);
            frame(0.0f, c32, c32, fused, L);
        } else if (only == "part") {
            ok = ok && run<double, false>("part 64x32 f64", dp_part_kernel<double, 64, 32, 1>, 512, 4, 64, 32, 1, 1, dp, L);
            ok = ok && run<float, false>("part 128x24 f32", dp_part_kernel<float, 128, 24, 1>, 768, 4, 128, 24, 1, 1, dp, L);
            ok = ok && run<float, false>("part 128x24/3 f32", dp_part_kernel<float, 128, 24, 3>, 256, 4, 128, 24, 1, 1, dp, L);
        } else if (only == "tile") {
            ok = ok && run<double, true>("Dornic 64x16 f64", dp_step_kernel<double, 64, 16, 256, 1, 6, 1>, 256, 1, 64, 16, 3, 1, rk, L);
            ok = ok && run<float, true>("Dornic 128x24 f32", dp_step_kernel<float, 128, 24, 256, 1, 1, 1>, 256, 1, 128, 24, 3, 1, rk, L);
            ok = ok && run<double, false>("split 32x16 f64", rk_step_kernel<double, 32, 16, 256, true>, 256, 1, 32, 16, 3, 3, rk, L);
            ok = ok && run<float, false>("split 32x16 f32", rk_step_kernel<float, 32, 16, 256, true>, 256, 1, 32, 16, 3, 3, rk, L);
            ok = ok && run<double, false>("DP 64x32 f64", dp_step_kernel<double, 64, 32, 256, 0, 6, 1>, 256, 1, 64, 32, 1, 1, dp, L);
            ok = ok && run<float, false>("DP 128x24 f32", dp_step_kernel<float, 128, 24, 256, 0, 6, 1>, 256, 1, 128, 24, 1, 1, dp, L);
        } else if (only == "veg") {
            ok = ok && run_veg(rk, L, false) && run_veg(rk, L, true);
        } else {
            return 2;
        }
    }
    if (!ok) return 1;
    puts("ok");
    return 0;
}
