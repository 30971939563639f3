// Launches of the two-stage FFT kernels (fts_fft_two.hpp).
#include "fts_fft_two.hpp"
#include "fts_internal.hpp"

namespace fts {

namespace {
constexpr int LDS_LIMIT = 160 * 1024;

template <typename K>
void allow_lds(K kernel) {
    FTS_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_LIMIT));
}

template <typename T>
constexpr int prec() {
    return sizeof(T) == sizeof(float) ? 1 : 0;
}

// the plan for spectra of the grid's padded rows, or of rows of nzc values (a caller's layout)
TwoGeom two_rows(TwoGeom t, bool contiguous) {
    if (contiguous) t.sp = t.nzc;
    return t;
}
}  // namespace

template <typename T>
void two_set_lds_limits() {
    static bool done = false;
    if (done) return;
    allow_lds(&slab_two_kernel<T, false>);
    if constexpr (sizeof(T) == 8) allow_lds(&slab_two_kernel<T, true>);
    allow_lds(&pencil_two_kernel<T>);
    allow_lds(&flat_steps_kernel<T, true>);
    allow_lds(&flat_steps_kernel<T, false>);
    done = true;
}

template <typename T>
void Grid::launch_slab_two(int mode, const SlabBatch<T>& b, bool contiguous) const {
    // the first half step of a Richardson pair waits in the output slice
    bool two_spectra = mode == SLAB_INV2;
    for (int i = 0; i < b.n; i++) {
        if (mode == SLAB_INV2 && !b.it[i].qout) throw Error("slab item without the real slice its second pass reads");
        if (mode == SLAB_FWD && b.it[i].n_out > 1) two_spectra = true;
    }
    const TwoGeom t = two_rows(two[prec<T>()], contiguous);
    const dim3 grid(tnx[0], b.n), block(two_slab_threads(t));
    const size_t lds = two_slab_lds(t, sizeof(typename vec2<T>::type));
    if constexpr (sizeof(T) == 8) {
        if (two_spectra) {
            hipLaunchKernelGGL((slab_two_kernel<T, true>), grid, block, lds, stream(), t, mode, b, tw<T>(1), tw<T>(2));
            return;
        }
    }
    hipLaunchKernelGGL((slab_two_kernel<T, false>), grid, block, lds, stream(), t, mode, b, tw<T>(1), tw<T>(2));
}

template <typename T>
void Grid::launch_xpass_two(const XBatch<T>& b, const T* bx, const T* by, const T* bz, bool contiguous) const {
    const TwoGeom t = two_rows(two[prec<T>()], contiguous);
    constexpr int e = sizeof(typename vec2<T>::type);
    const int tiles = ceil_div(t.nzc, two_pencil_columns(e));
    hipLaunchKernelGGL((pencil_two_kernel<T>), dim3(tnx[1] * tiles, b.n), dim3(64), two_pencil_lds(t, two_pencil_columns(e), e), stream(), t,
                       b, tw<T>(0), bx, by, bz);
}

template <typename T>
void Grid::launch_flat(bool continuous, const FlatBatch<T>& b, const T* by, const T* bz) const {
    if (b.n == 0) return;
    FTS_REQUIRE(flat<T>(), "flat steps need a grid of one x-slab with a two-stage plan");
    const TwoGeom& t = two[prec<T>()];
    const dim3 grid(b.n), block(two_slab_threads(t));
    const size_t lds = two_slab_lds(t, sizeof(typename vec2<T>::type));
    KernelTimer& timer = ctx->timer;
    hipEvent_t start = timer.begin(stream(), FTS_KERNEL_SLAB);
    const int n = tnx[2], P = line_lanes(n);
    if (tnx[1] == 1 && n <= LINE_POINTS) {
        const dim3 threads(ceil_div(n * P, 64) * 64);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, threads, line_lds(n), stream(), n, b, bz);
        };
        if (n <= 64) go(continuous ? line_steps_kernel<T, true, 8, 8> : line_steps_kernel<T, false, 8, 8>);
        else if (n <= 128) go(continuous ? line_steps_kernel<T, true, 8, 16> : line_steps_kernel<T, false, 8, 16>);
        else go(continuous ? line_steps_kernel<T, true, 4, 0> : line_steps_kernel<T, false, 4, 0>);
    } else if (continuous)
        hipLaunchKernelGGL((flat_steps_kernel<T, true>), grid, block, lds, stream(), t, b, tw<T>(1), tw<T>(2), by, bz);
    else
        hipLaunchKernelGGL((flat_steps_kernel<T, false>), grid, block, lds, stream(), t, b, tw<T>(1), tw<T>(2), by, bz);
    FTS_HIP_CHECK(hipGetLastError());
    if (start) {
        // each step writes its slice once; the first slice, w and the mask are read once
        double bytes = 0.0;
        for (int i = 0; i < b.n; i++) bytes += (double)sizeof(T) * M * (b.it[i].steps + 2 + (b.it[i].mask ? 1 : 0));
        timer.end(stream(), start, FTS_KERNEL_SLAB, bytes);
    }
}

#define FTS_TWO_INSTANCES(T)                                                                        \
    template void two_set_lds_limits<T>();                                                          \
    template void Grid::launch_slab_two<T>(int, const SlabBatch<T>&, bool) const;                   \
    template void Grid::launch_xpass_two<T>(const XBatch<T>&, const T*, const T*, const T*, bool) const; \
    template void Grid::launch_flat<T>(bool, const FlatBatch<T>&, const T*, const T*) const;
FTS_TWO_INSTANCES(double)
FTS_TWO_INSTANCES(float)

}  // namespace fts
