// Wave-local line transforms for cubic grids N = 32, 48, 64, 96, 128, used by the stress pass.
//
// Every 1D line transform belongs to one wavefront for all its Stockham stages:
// a stage's butterflies take their inputs from registers, and the exchange between
// stages goes through the wave's own LDS lines with no workgroup barrier (LDS
// operations of one wavefront complete in issue order; wave_sync keeps the
// compiler from moving them). The result stays in registers at the positions the last
// stage writes, the same for every line, so two spectra can be multiplied there.
#pragma once

#include "fts_fft_ct.hpp"

namespace fts {

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// radix plan of a length-L transform, optionally reversed
template <int L, bool REV>
struct WPlan {
    static constexpr CPlan P = make_cplan(L);
    static constexpr int n = P.n;
    static constexpr int r(int s) { return REV ? P.r[P.n - 1 - s] : P.r[s]; }
    static constexpr int ns(int s) { return s == 0 ? 1 : ns(s - 1) * r(s - 1); }
};

// Butterfly g of a stage with radix R over NLW lines of a wavefront: lane g % 64,
// register slot g / 64; line-fast order (LF) puts consecutive lanes on consecutive
// lines, otherwise on consecutive butterflies of one line.
template <int L, int R, int NLW, bool LF>
struct WMap {
    static constexpr int B = L / R;
    static constexpr int TOTAL = NLW * B;
    static constexpr int NT = (TOTAL + 63) / 64;
    static __device__ __forceinline__ int line(int g) { return LF ? g % NLW : g / B; }
    static __device__ __forceinline__ int idx(int g) { return LF ? g / NLW : g % B; }
    static __device__ __forceinline__ bool ok(int g, int nvalid) {
        return (TOTAL % 64 == 0 || g < TOTAL) && line(g) < nvalid;
    }
};

template <int L, bool REV, int S, int NLW, bool LF>
using WStageMap = WMap<L, WPlan<L, REV>::r(S), NLW, LF>;

// registers of one stage's inputs: [slots][radix]
template <typename T2, int L, bool REV, int S, int NLW, bool LF>
struct WRegs {
    using type = T2[WStageMap<L, REV, S, NLW, LF>::NT][WPlan<L, REV>::r(S)];
};

// Position of element i of a line in the exchange between two stages: with SK one pad
// slot after every 8 elements, so that the stride-R stores of a stage's butterflies
// (positions R j + r) fall on different LDS banks; the line then spans L + (L-1)/8 slots.
template <bool SK>
__device__ __forceinline__ int wl_slot(int i) {
    return SK ? i + (i >> 3) : i;
}

// Stages S.. of the plan over this wavefront's lines (line l at X + l LP, element i
// at stride ES; skewed exchange positions with SK). v holds stage S's inputs; `done`
// receives the last stage's outputs in registers (positions j + r L/R_last).
template <int DIR, typename T, typename T2, int L, bool REV, int NLW, bool LF, int LP, int ES, bool SK, int S,
          typename F>
__device__ __forceinline__ void wl_stages(typename WRegs<T2, L, REV, S, NLW, LF>::type& v, T2* X, const T2* W,
                                          int lane, int nvalid, F&& done) {
    using PL = WPlan<L, REV>;
    constexpr int R = PL::r(S);
    constexpr int NS = PL::ns(S);
    constexpr int TWS = L / (NS * R);
    using M = WMap<L, R, NLW, LF>;
#pragma unroll
    for (int t = 0; t < M::NT; t++) {
        const int g = lane + 64 * t;
        if (M::ok(g, nvalid)) {
            if constexpr (NS > 1) {
                const int k = M::idx(g) % NS;
#pragma unroll
                for (int r = 1; r < R; r++) v[t][r] = cmul(v[t][r], root<DIR>(W, (r * k * TWS) % L));
            }
            Dft<R, DIR, T, T2>::run(v[t], W, L);
        }
    }
    if constexpr (S + 1 == PL::n) {
        done(v);
    } else {
        wave_sync();
#pragma unroll
        for (int t = 0; t < M::NT; t++) {
            const int g = lane + 64 * t;
            if (M::ok(g, nvalid)) {
                const int j = M::idx(g);
                const int d = (j / NS) * NS * R + j % NS;
                T2* base = X + M::line(g) * LP;
#pragma unroll
                for (int r = 0; r < R; r++) base[wl_slot<SK>(d + r * NS) * ES] = v[t][r];
            }
        }
        wave_sync();
        using M2 = WStageMap<L, REV, S + 1, NLW, LF>;
        constexpr int R2 = PL::r(S + 1);
        T2 u[M2::NT][R2];
#pragma unroll
        for (int t = 0; t < M2::NT; t++) {
            const int g = lane + 64 * t;
            if (M2::ok(g, nvalid)) {
                const T2* base = X + M2::line(g) * LP;
                const int j = M2::idx(g);
#pragma unroll
                for (int r = 0; r < R2; r++) u[t][r] = base[wl_slot<SK>(j + r * M2::B) * ES];
            }
        }
        wl_stages<DIR, T, T2, L, REV, NLW, LF, LP, ES, SK, S + 1>(u, X, W, lane, nvalid, done);
    }
}

// ------------------------------------------------------------------ pencils of the stress pass
template <int N, int NL_>
struct WPencil {
    static constexpr int NZC = N / 2 + 1;
    static constexpr int NL = NL_;   // kz columns per wavefront
    static constexpr int TILES = (NZC + NL - 1) / NL;
    static constexpr int BD = 64;
    static constexpr size_t lds_elems = (size_t)N * NL + N;
    using F = WPlan<N, false>;
};

}  // namespace fts
