// CPU workgroup emulator of the two-stage FFT kernels of fts_fft_two.hpp (slab_two_kernel,
// pencil_two_kernel, flat_steps_kernel): the kernels' own source, compiled for the host against
// the stand-in hip/hip_runtime.h beside this file, one fiber per GPU thread, with barriers that
// report a mismatch. LDS is a heap block of exactly the kernel's dynamic size, filled with
// NaN before each workgroup, and every global buffer has exactly its own size, so that
// -fsanitize=address reports each index that leaves one and never-written values poison the
// result.
//
//   fft_two_emu <op> <precision 4|8> nx ny nz <in> <out>
//
// op conv: real field -> slab FWD, pencil (bond factors), slab INV1 -> real field
//    fft: real field -> slab FWD, pencil forward -> half spectrum [nx][ny][nz/2+1]
//    ifft: half spectrum -> pencil inverse, slab INV1 -> real field
//    step: a continuous Richardson step by slab and pencil passes (FWD of two spectra, INV1 with
//          forward, INV2 with forward), twice; input: q, w, mask; output: both slices
//    flat: the same two steps by flat_steps_kernel (nx = 1)
//    flatd: two discrete steps by flat_steps_kernel (nx = 1)
//    line, lined: the same by line_steps_kernel in the launch shape of the length (nx = ny = 1)
//    factor: exp(-w ds/2) and exp(-w ds/4) as the steps take them, w in the place of q
//    linec: the coefficients that line_steps_kernel makes of the full and the half bond (nx = ny = 1, FP64)
// Bond factors along each axis: exp(-0.3 (k / L)^2) full, exp(-0.15 (k / L)^2) half, k folded.
#include <hip/hip_runtime.h>

#include <sanitizer/common_interface_defs.h>
#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

namespace fts {
unsigned char* smem_raw_ptr;
}
inline double cospi(double x) { return (double)cosl(3.14159265358979323846264338327950288L * x); }
double __shfl_xor(double v, int mask, int width);
#define FTS_DYNAMIC_LDS(name) unsigned char* name = smem_raw_ptr
#include "fts_fft_two.hpp"

thread_local dim3 threadIdx;
thread_local dim3 blockIdx;
dim3 blockDim;
dim3 gridDim;

namespace {

// The GPU threads of a workgroup are fibers of one OS thread: a barrier switches to the next
// fiber, so a round of the ring takes every thread from one barrier to the next.
struct Fiber {
    ucontext_t ctx;
    std::vector<char> stack;
    void* fake = nullptr;
    bool done = false;
    long barriers = 0;
};
std::vector<Fiber> fibers;
ucontext_t scheduler;
void* scheduler_fake = nullptr;
const void* scheduler_stack = nullptr;
size_t scheduler_size = 0;
size_t current = 0;
std::vector<float> lds_left;   // what the last workgroup left in its LDS
void (*body)(void*) = nullptr;
void* body_arg = nullptr;

void to_scheduler(bool last) {
    Fiber& f = fibers[current];
    __sanitizer_start_switch_fiber(last ? nullptr : &f.fake, scheduler_stack, scheduler_size);
    swapcontext(&f.ctx, &scheduler);
    __sanitizer_finish_switch_fiber(f.fake, &scheduler_stack, &scheduler_size);
}

void fiber_main() {
    __sanitizer_finish_switch_fiber(nullptr, &scheduler_stack, &scheduler_size);
    body(body_arg);
    fibers[current].done = true;
    to_scheduler(true);
}

}  // namespace

void emu_syncthreads() {
    fibers[current].barriers++;
    to_scheduler(false);
}

// every thread of the workgroup takes part, as in the kernels: one round of the ring stores, the next one reads
double __shfl_xor(double v, int mask, int) {
    static double lanes[1024];
    lanes[current] = v;
    emu_syncthreads();
    const double r = lanes[current ^ (size_t)mask];
    emu_syncthreads();
    return r;
}

namespace {

template <typename F>
void run_grid(dim3 grid, int threads, size_t lds, F&& kernel) {
    gridDim = grid;
    blockDim = dim3{(unsigned)threads, 1, 1};
    body = [](void* p) { (*static_cast<std::remove_reference_t<F>*>(p))(); };
    body_arg = &kernel;
    fibers.clear();
    fibers.resize(threads);
    for (auto& f : fibers) f.stack.resize(256 * 1024);
    for (unsigned by = 0; by < grid.y; by++)
        for (unsigned bx = 0; bx < grid.x; bx++) {
            std::vector<float> mem(lds / sizeof(float), std::nanf(""));
            fts::smem_raw_ptr = reinterpret_cast<unsigned char*>(mem.data());
            blockIdx = dim3{bx, by, 0};
            for (auto& f : fibers) {
                getcontext(&f.ctx);
                f.ctx.uc_stack.ss_sp = f.stack.data();
                f.ctx.uc_stack.ss_size = f.stack.size();
                f.ctx.uc_link = nullptr;
                f.done = false;
                f.fake = nullptr;
                f.barriers = 0;
                makecontext(&f.ctx, fiber_main, 0);
            }
            for (bool alive = true; alive;) {
                alive = false;
                for (current = 0; current < fibers.size(); current++) {
                    Fiber& f = fibers[current];
                    if (f.done) continue;
                    threadIdx = dim3{(unsigned)current, 0, 0};
                    __sanitizer_start_switch_fiber(&scheduler_fake, f.stack.data(), f.stack.size());
                    swapcontext(&scheduler, &f.ctx);
                    __sanitizer_finish_switch_fiber(scheduler_fake, nullptr, nullptr);
                    alive = alive || !f.done;
                }
                // every thread is at the same barrier, or has ended after the same number of them
                for (auto& f : fibers)
                    if (f.barriers != fibers[0].barriers || f.done != fibers[0].done) {
                        std::fprintf(stderr, "BARRIER MISMATCH in block (%u, %u)\n", bx, by);
                        std::exit(4);
                    }
            }
            lds_left = mem;
        }
}

template <typename T>
struct Emu {
    using T2 = typename fts::vec2<T>::type;
    int n[3];
    fts::TwoGeom g{};
    size_t M, Ms;
    std::vector<T2> tw[3];
    std::vector<T> bx, by, bz;

    explicit Emu(const int* dims) {
        std::copy(dims, dims + 3, n);
        if (!fts::two_geometry(n, sizeof(T2), 160 * 1024, g)) {
            std::fprintf(stderr, "no two-stage plan\n");
            std::exit(5);
        }
        M = (size_t)n[0] * n[1] * n[2];
        Ms = (size_t)n[0] * n[1] * g.sp;
        for (int a = 0; a < 3; a++)
            for (int m = 0; m < n[a]; m++) {
                const double x = 2.0 * M_PI * m / n[a];
                tw[a].push_back(T2{(T)std::cos(x), (T)-std::sin(x)});
            }
        auto table = [](std::vector<T>& v, int L, int count) {
            for (int h = 0; h < 2; h++)
                for (int k = 0; k < count; k++) {
                    const double f = k > L / 2 ? L - k : k;
                    v.push_back((T)std::exp((h ? -0.15 : -0.3) * f * f / L / L));
                }
        };
        table(bx, n[0], n[0]);
        table(by, n[1], n[1]);
        table(bz, n[2], g.nzc);
        std::printf("y %d x %d, z %d x %d, x %d x %d, threads %d, pitch %d, lds %zu + %zu\n", g.y.r1, g.y.r2, g.z.r1,
                    g.z.r2, g.x.r1, g.x.r2, fts::two_slab_threads(g), g.pitch, fts::two_slab_lds(g, sizeof(T2)),
                    fts::two_pencil_lds(g, fts::two_pencil_columns(sizeof(T2)), sizeof(T2)));
    }
    void slab(int mode, const fts::SlabItem<T>& it) {
        fts::SlabBatch<T> b{};
        b.n = 1;
        b.it[0] = it;
        run_grid(dim3{(unsigned)n[0], 1, 1}, fts::two_slab_threads(g), fts::two_slab_lds(g, sizeof(T2)),
                 [&] {
                     // Grid::launch_slab_two's choice
                     if (sizeof(T) == 8 && (mode == fts::SLAB_INV2 || (mode == fts::SLAB_FWD && it.n_out > 1)))
                         fts::slab_two_kernel<T, sizeof(T) == 8>(g, mode, b, tw[1].data(), tw[2].data());
                     else fts::slab_two_kernel<T, false>(g, mode, b, tw[1].data(), tw[2].data());
                 });
    }
    void pencil(T2* c, int table) {
        fts::XBatch<T> b{};
        b.n = 1;
        b.it[0] = fts::XItem<T>{c, table};
        const int C = fts::two_pencil_columns(sizeof(T2));
        run_grid(dim3{(unsigned)(n[1] * ((g.nzc + C - 1) / C)), 1, 1}, 64, fts::two_pencil_lds(g, fts::two_pencil_columns(sizeof(T2)), sizeof(T2)),
                 [&] { fts::pencil_two_kernel<T>(g, b, tw[0].data(), bx.data(), by.data(), bz.data()); });
    }
    std::vector<T2> spectrum() const { return std::vector<T2>(Ms, T2{(T)NAN, (T)NAN}); }
};

template <typename T>
int run(const char* op, const int* n, const char* in_path, const char* out_path) {
    using T2 = typename fts::vec2<T>::type;
    Emu<T> e(n);
    const size_t M = e.M;
    const int rows = n[0] * n[1];
    auto is = [&](const char* s) { return std::strcmp(op, s) == 0; };
    std::vector<T> in;
    {
        FILE* f = std::fopen(in_path, "rb");
        if (!f) return 2;
        std::fseek(f, 0, SEEK_END);
        in.resize(std::ftell(f) / sizeof(T));
        std::rewind(f);
        if (std::fread(in.data(), sizeof(T), in.size(), f) != in.size()) return 2;
        std::fclose(f);
    }
    std::vector<T> out;
    if (is("conv") || is("fft")) {
        auto c = e.spectrum();
        fts::SlabItem<T> it{};
        it.qin = in.data();
        it.c0 = c.data();
        it.n_out = 1;
        e.slab(fts::SLAB_FWD, it);
        e.pencil(c.data(), is("fft") ? -1 : 0);
        if (is("fft")) {
            for (int r = 0; r < rows; r++)
                for (int k = 0; k < e.g.nzc; k++) {
                    out.push_back(c[(size_t)r * e.g.sp + k].x);
                    out.push_back(c[(size_t)r * e.g.sp + k].y);
                }
        } else {
            out.assign(M, (T)NAN);
            fts::SlabItem<T> b{};
            b.c0 = c.data();
            b.qout = out.data();
            e.slab(fts::SLAB_INV1, b);
        }
    } else if (is("ifft")) {
        auto c = e.spectrum();
        for (int r = 0; r < rows; r++)
            for (int k = 0; k < e.g.nzc; k++) {
                const size_t s = 2 * ((size_t)r * e.g.nzc + k);
                c[(size_t)r * e.g.sp + k] = T2{in[s], in[s + 1]};
            }
        e.pencil(c.data(), -2);
        out.assign(M, (T)NAN);
        fts::SlabItem<T> b{};
        b.c0 = c.data();
        b.qout = out.data();
        e.slab(fts::SLAB_INV1, b);
    } else {
        // input: q, w, mask
        std::vector<T> w(in.begin() + M, in.begin() + 2 * M), mask(in.begin() + 2 * M, in.begin() + 3 * M);
        // factors are read from a table: exp(-w ds) of discrete steps, else exp(-w ds/2) in FP64 and exp(-w ds/4)
        const double ds = 0.25;
        constexpr bool fp64 = sizeof(T) == 8;
        for (T& x : w) x = (T)std::exp(-(double)x * (is("flatd") || is("lined") ? ds : fp64 ? ds / 2 : ds / 4));
        const T half_w = (T)(fp64 ? fts::FACTOR_TABLE : fts::FACTOR_SQUARE), full_w = (T)fts::FACTOR_TABLE;
        const T quarter_w = (T)(fp64 ? fts::FACTOR_ROOT : fts::FACTOR_TABLE);
        out.assign(2 * M, (T)NAN);
        if (is("factor")) {
            for (size_t i = 0; i < M; i++) {
                out[i] = fts::factor<T>(w[i], true, half_w);
                out[M + i] = fts::factor<T>(w[i], true, quarter_w);
            }
        } else if (is("step")) {
            std::vector<T> q(in.begin(), in.begin() + M);
            auto c0 = e.spectrum(), c1 = e.spectrum();
            fts::SlabItem<T> a{};
            a.qin = q.data();
            a.c0 = c0.data();
            a.c1 = c1.data();
            a.w = w.data();
            a.pre0 = half_w;
            a.pre1 = quarter_w;
            a.n_out = 2;
            e.slab(fts::SLAB_FWD, a);
            for (int s = 0; s < 2; s++) {
                e.pencil(c0.data(), 0);
                e.pencil(c1.data(), 1);
                fts::SlabItem<T> b{};
                b.c0 = c1.data();
                b.w = w.data();
                b.post0 = half_w;
                b.forward = 1;
                e.slab(fts::SLAB_INV1, b);
                e.pencil(c1.data(), 1);
                fts::SlabItem<T> c{};
                c.c0 = c0.data();
                c.c1 = c1.data();
                c.w = w.data();
                c.post0 = c.pre0 = half_w;
                c.post1 = c.pre1 = quarter_w;
                c.mask = mask.data();
                c.qout = out.data() + s * M;
                c.forward = s == 0;
                e.slab(fts::SLAB_INV2, c);
            }
        } else {
            std::vector<T> q(3 * M, (T)NAN), half(M, (T)NAN);
            std::copy(in.begin(), in.begin() + M, q.begin());
            fts::FlatBatch<T> b{};
            b.n = 1;
            b.stride = M;
            fts::FlatItem<T>& it = b.it[0];
            it.q = q.data();
            it.half = half.data();
            it.w = w.data();
            it.mask = mask.data();
            it.steps = is("linec") ? 0 : 2;
            it.full_table = 0;
            it.half_table = 1;
            const bool cont = is("flat") || is("line") || is("linec");
            it.full_w = cont ? half_w : full_w;
            it.half_w = quarter_w;
            if (is("line") || is("lined") || is("linec")) {
                const int L = n[2], P = fts::line_lanes(L);
                run_grid(dim3{1, 1, 1}, (L * P + 63) / 64 * 64, fts::line_lds(L), [&] {
                    auto go = [&](auto p, auto ch) {
                        constexpr int PP = decltype(p)::value, CH = decltype(ch)::value;
                        if (cont) fts::line_steps_kernel<T, true, PP, CH>(L, b, e.bz.data());
                        else fts::line_steps_kernel<T, false, PP, CH>(L, b, e.bz.data());
                    };
                    using std::integral_constant;
                    if (L <= 64) go(integral_constant<int, 8>{}, integral_constant<int, 8>{});
                    else if (L <= 128) go(integral_constant<int, 8>{}, integral_constant<int, 16>{});
                    else go(integral_constant<int, 4>{}, integral_constant<int, 0>{});
                });
            } else
            run_grid(dim3{1, 1, 1}, fts::two_slab_threads(e.g), fts::two_slab_lds(e.g, sizeof(T2)), [&] {
                if (cont)
                    fts::flat_steps_kernel<T, true>(e.g, b, e.tw[1].data(), e.tw[2].data(), e.by.data(), e.bz.data());
                else
                    fts::flat_steps_kernel<T, false>(e.g, b, e.tw[1].data(), e.tw[2].data(), e.by.data(), e.bz.data());
            });
            std::copy(q.begin() + M, q.end(), out.begin());
            if (is("linec")) std::memcpy(out.data(), lds_left.data(), 2 * M * sizeof(T));
        }
    }
    FILE* f = std::fopen(out_path, "wb");
    if (!f || std::fwrite(out.data(), sizeof(T), out.size(), f) != out.size()) return 2;
    std::fclose(f);
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc != 8) return 2;
    const int n[3] = {std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5])};
    return std::atoi(argv[2]) == 4 ? run<float>(argv[1], n, argv[6], argv[7])
                                   : run<double>(argv[1], n, argv[6], argv[7]);
}
