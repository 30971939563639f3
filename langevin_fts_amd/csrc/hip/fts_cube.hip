// Launches of the N^3 slab and pencil kernels (fts_fft_two.hpp) in every launch shape.
#include "fts_fft_two.hpp"
#include "fts_internal.hpp"

namespace fts {

namespace {

template <typename K>
void allow_lds(K kernel) {
    FTS_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
}

template <typename T, int N, int BD>
void slab(const Grid& g, int mode, const SlabBatch<T>& b) {
    using T2 = typename vec2<T>::type;
    const dim3 grid(N, b.n), block(BD);
    const size_t lds = two_slab_lds(TwoCube<N, sizeof(T2)>::G, sizeof(T2));
    for (int i = 0; i < b.n; i++)
        if ((mode == SLAB_INV2 || (mode == SLAB_FWD && b.it[i].n_out > 1)) && !b.it[i].w)
            throw Error("slab item of two spectra without a factor table");
    const T2 *twy = g.tw<T>(1), *twz = g.tw<T>(2);
    if (mode == SLAB_FWD)
        hipLaunchKernelGGL((slab_cube_kernel<T, SLAB_FWD, N, BD>), grid, block, lds, g.stream(), b, twy, twz);
    else if (mode == SLAB_INV1)
        hipLaunchKernelGGL((slab_cube_kernel<T, SLAB_INV1, N, BD>), grid, block, lds, g.stream(), b, twy, twz);
    else
        hipLaunchKernelGGL((slab_cube_kernel<T, SLAB_INV2, N, BD>), grid, block, lds, g.stream(), b, twy, twz);
}

template <typename T, int N>
void slab_bd(const Grid& g, int bd, int mode, const SlabBatch<T>& b) {
    switch (bd) {
        case 128: if constexpr (slab_bd_ok(N, 128)) return slab<T, N, 128>(g, mode, b); break;
        case 256: if constexpr (slab_bd_ok(N, 256)) return slab<T, N, 256>(g, mode, b); break;
        case 320: if constexpr (slab_bd_ok(N, 320)) return slab<T, N, 320>(g, mode, b); break;
        case 384: if constexpr (slab_bd_ok(N, 384)) return slab<T, N, 384>(g, mode, b); break;
        case 512: if constexpr (slab_bd_ok(N, 512)) return slab<T, N, 512>(g, mode, b); break;
        case 1024: if constexpr (slab_bd_ok(N, 1024)) return slab<T, N, 1024>(g, mode, b); break;
        default: break;
    }
    throw Error("no slab kernel of " + std::to_string(bd) + " threads for N=" + std::to_string(N));
}

template <typename T, int N, int NL>
void pencil(const Grid& g, const XBatch<T>& b, const T* bx, const T* by, const T* bz) {
    using T2 = typename vec2<T>::type;
    hipLaunchKernelGGL((pencil_cube_kernel<T, N, NL>), dim3(N * cube_pencil_tiles<T2, N, NL>(), b.n), dim3(64),
                       two_pencil_lds(TwoCube<N, sizeof(T2)>::G, NL, sizeof(T2)), g.stream(), b, g.tw<T>(0), bx, by,
                       bz);
}

template <typename T, int N>
void pencil_nl(const Grid& g, int nl, const XBatch<T>& b, const T* bx, const T* by, const T* bz) {
    switch (nl) {
        case 4: return pencil<T, N, 4>(g, b, bx, by, bz);
        case 8: return pencil<T, N, 8>(g, b, bx, by, bz);
        case 16: return pencil<T, N, 16>(g, b, bx, by, bz);
        default: break;
    }
    throw Error("no pencil kernel of " + std::to_string(nl) + " columns");
}

// LDS limits of every variant, set before any launch (and so before any graph capture
// could record the first one)
template <typename T, int N, int BD>
void limits_bd() {
    if constexpr (slab_bd_ok(N, BD)) {
        allow_lds(&slab_cube_kernel<T, SLAB_FWD, N, BD>);
        allow_lds(&slab_cube_kernel<T, SLAB_INV1, N, BD>);
        allow_lds(&slab_cube_kernel<T, SLAB_INV2, N, BD>);
    }
}
template <typename T, int N>
void limits() {
    limits_bd<T, N, 128>();
    limits_bd<T, N, 256>();
    limits_bd<T, N, 320>();
    limits_bd<T, N, 384>();
    limits_bd<T, N, 512>();
    limits_bd<T, N, 1024>();
    allow_lds(&pencil_cube_kernel<T, N, 4>);
    allow_lds(&pencil_cube_kernel<T, N, 8>);
    allow_lds(&pencil_cube_kernel<T, N, 16>);
}

}  // namespace

template <typename T>
void launch_slab_cube(const Grid& g, int n, int bd, int mode, const SlabBatch<T>& b) {
    switch (n) {
        case 32: return slab_bd<T, 32>(g, bd, mode, b);
        case 48: return slab_bd<T, 48>(g, bd, mode, b);
        case 64: return slab_bd<T, 64>(g, bd, mode, b);
        case 96: return slab_bd<T, 96>(g, bd, mode, b);
        default: return slab_bd<T, 128>(g, bd, mode, b);
    }
}

template <typename T>
void launch_pencil_cube(const Grid& g, int n, int nl, const XBatch<T>& b, const T* bx, const T* by, const T* bz) {
    switch (n) {
        case 32: return pencil_nl<T, 32>(g, nl, b, bx, by, bz);
        case 48: return pencil_nl<T, 48>(g, nl, b, bx, by, bz);
        case 64: return pencil_nl<T, 64>(g, nl, b, bx, by, bz);
        case 96: return pencil_nl<T, 96>(g, nl, b, bx, by, bz);
        default: return pencil_nl<T, 128>(g, nl, b, bx, by, bz);
    }
}

template <typename T>
void cube_set_lds_limits() {
    static bool done = false;
    if (done) return;
    limits<T, 32>();
    limits<T, 48>();
    limits<T, 64>();
    limits<T, 96>();
    limits<T, 128>();
    done = true;
}

#define FTS_CUBE_INSTANCES(T)                                                                              \
    template void launch_slab_cube<T>(const Grid&, int, int, int, const SlabBatch<T>&);                    \
    template void launch_pencil_cube<T>(const Grid&, int, int, const XBatch<T>&, const T*, const T*, const T*); \
    template void cube_set_lds_limits<T>();
FTS_CUBE_INSTANCES(double)
FTS_CUBE_INSTANCES(float)

}  // namespace fts
