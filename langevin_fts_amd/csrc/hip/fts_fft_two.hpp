// Two-stage in-place line transforms for general grid sizes: every axis length is a product
// r1 r2 of two register radices (1..16), so a line transform is two butterflies with one LDS
// round trip between them.
//
// Forward (decimation in frequency) of n = n1 r2 + n2:
//   stage A, per n2: r1-point transform over n1 -> k1, times W_L^(k1 n2), left at (k1, n2);
//   stage B, per k1: r2-point transform over n2 -> k2: X[k1 + r1 k2].
// The inverse runs B then A with conjugate roots. Every butterfly writes the LDS slots it has
// read, so a stage needs no second buffer and no registers beyond its own R values, a thread can
// loop over any number of butterflies, and one barrier between stages is enough. The order of
// the result is a permutation that the next pass undoes by the row it reads or stores, so it
// costs nothing.
//
// Slab plane. Two rows of a z pair travel as one complex line, x = row a + i row b. The pair is
// (2a) r2 + n2 and (2a + 1) r2 + n2 of the y plan: both rows are outputs of one inverse y
// butterfly and inputs of one forward one, so the Hermitian merge and split
//   Z[k] = A[k] + i B[k], Z[nz - k] = conj A[k] + i conj B[k]
// happen in that butterfly's registers, with no LDS pass of their own. Column c of the half
// spectrum owns the slots c and nz - c of every packed line (c = 0 and c = nz / 2, where these
// meet, take a spare slot after the line): the y stages work in place there.
#pragma once

#include <type_traits>

#include "fts_two_plan.hpp"

namespace fts {

// the workgroup's dynamic LDS
#ifndef FTS_DYNAMIC_LDS
#define FTS_DYNAMIC_LDS(name) extern __shared__ __align__(16) unsigned char name[]
#endif

// ------------------------------------------------------------------ register transforms
// RDft<R, DIR>::run: R-point transform in registers, natural order in and out, DIR -1 forward.
// 2, 3, 4 and 5 are fts_fft.hpp's butterflies; R = A B with coprime A, B by the prime-factor
// algorithm (no twiddles); 9 and 16 as 3 x 3 and 4 x 4; 7, 11 and 13 from the symmetric sums
// v_j +- v_(R - j).
template <int R>
struct PrimeRoots;   // cos, sin of 2 pi j / R, j = 1..(R - 1) / 2
template <>
struct PrimeRoots<7> {
    static constexpr double c[3] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
    static constexpr double s[3] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
};
template <>
struct PrimeRoots<11> {
    static constexpr double c[5] = {0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                    -0.65486073394528506406, -0.95949297361449738989};
    static constexpr double s[5] = {0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                    0.75574957435425828377, 0.28173255684142969771};
};
template <>
struct PrimeRoots<13> {
    static constexpr double c[6] = {0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                                    -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
    static constexpr double s[6] = {0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                                    0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
};
// cos, sin of 2 pi m / 9 and 2 pi m / 16 for the twiddles of the 3 x 3 and 4 x 4 forms
__host__ __device__ constexpr double root_cos(int R, int m) {
    constexpr double c9[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
    constexpr double c16[10] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0,
                                -0.38268343236508977173, -0.70710678118654752440, -0.92387953251128675613, -1.0,
                                -0.92387953251128675613};
    return R == 9 ? c9[m] : c16[m];
}
__host__ __device__ constexpr double root_sin(int R, int m) {
    constexpr double s9[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                              0.34202014332566873304};
    constexpr double s16[10] = {0.0, 0.38268343236508977173, 0.70710678118654752440, 0.92387953251128675613, 1.0,
                                0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0,
                                -0.38268343236508977173};
    return R == 9 ? s9[m] : s16[m];
}

// Products with roots are written as fused operations: the compiler's own choice of which product of a sum
// to fuse can differ between instances of one kernel. Lines of 32, 64 and 128 points so give the same bits in
// every launch shape. Radices 3 and 5 and the prime ones leave their sums to the compiler: at 48^3 and 96^3
// FP64 has been the same in all shapes, FP32 differs by 5e-7 between some pencil widths.
__device__ __forceinline__ double two_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float two_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <typename T2>
__device__ __forceinline__ T2 tmul(T2 a, T2 w) {
    return T2{two_fma(a.x, w.x, -(a.y * w.y)), two_fma(a.x, w.y, a.y * w.x)};
}
// a times the conjugate of w
template <typename T2>
__device__ __forceinline__ T2 tmul_conj(T2 a, T2 w) {
    return T2{two_fma(a.x, w.x, a.y * w.y), two_fma(a.y, w.x, -(a.x * w.y))};
}

template <int R, int DIR, typename T, typename T2>
struct RDft;

template <int DIR, typename T, typename T2>
struct RDft<1, DIR, T, T2> {
    static __device__ __forceinline__ void run(T2 (&)[1]) {}
};

template <int R, int DIR, typename T, typename T2>
struct RDftBase {
    static __device__ __forceinline__ void run(T2 (&v)[R]) { Dft<R, DIR, T, T2>::run(v, (const T2*)nullptr, 0); }
};
template <int DIR, typename T, typename T2>
struct RDft<2, DIR, T, T2> : RDftBase<2, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<3, DIR, T, T2> : RDftBase<3, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<4, DIR, T, T2> : RDftBase<4, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<5, DIR, T, T2> : RDftBase<5, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<8, DIR, T, T2> {
    static __device__ __forceinline__ void run(T2 (&v)[8]) {
        const T h = (T)0.70710678118654752440;
        T2 e[4] = {v[0], v[2], v[4], v[6]};
        T2 o[4] = {v[1], v[3], v[5], v[7]};
        RDft<4, DIR, T, T2>::run(e);
        RDft<4, DIR, T, T2>::run(o);
        // o[1] and o[3] times W8 = (1 + DIR i) h and W8^3 = (-1 + DIR i) h, h in the final sums
        const T2 a = T2{o[1].x - DIR * o[1].y, o[1].y + DIR * o[1].x};
        const T2 b = T2{-o[3].x - DIR * o[3].y, DIR * o[3].x - o[3].y};
        const T2 c = mul_is<DIR>(o[2]);
        v[0] = cadd(e[0], o[0]);
        v[4] = csub(e[0], o[0]);
        v[1] = T2{two_fma(a.x, h, e[1].x), two_fma(a.y, h, e[1].y)};
        v[5] = T2{two_fma(a.x, -h, e[1].x), two_fma(a.y, -h, e[1].y)};
        v[2] = cadd(e[2], c);
        v[6] = csub(e[2], c);
        v[3] = T2{two_fma(b.x, h, e[3].x), two_fma(b.y, h, e[3].y)};
        v[7] = T2{two_fma(b.x, -h, e[3].x), two_fma(b.y, -h, e[3].y)};
    }
};

// coprime A, B: input index (B a + A b) mod R, output k with k mod A = ka and k mod B = kb
template <int A, int B, int DIR, typename T, typename T2>
struct RDftCoprime {
    static constexpr int R = A * B;
    static constexpr int crt(int ka, int kb) {
        int k = ka;
        while (k % B != kb) k += A;
        return k;
    }
    static __device__ __forceinline__ void run(T2 (&v)[R]) {
        T2 t[B][A];
#pragma unroll
        for (int b = 0; b < B; b++) {
#pragma unroll
            for (int a = 0; a < A; a++) t[b][a] = v[(B * a + A * b) % R];
            RDft<A, DIR, T, T2>::run(t[b]);
        }
#pragma unroll
        for (int a = 0; a < A; a++) {
            T2 u[B];
#pragma unroll
            for (int b = 0; b < B; b++) u[b] = t[b][a];
            RDft<B, DIR, T, T2>::run(u);
#pragma unroll
            for (int b = 0; b < B; b++) v[crt(a, b)] = u[b];
        }
    }
};
template <int DIR, typename T, typename T2>
struct RDft<6, DIR, T, T2> : RDftCoprime<2, 3, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<10, DIR, T, T2> : RDftCoprime<2, 5, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<12, DIR, T, T2> : RDftCoprime<4, 3, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<14, DIR, T, T2> : RDftCoprime<2, 7, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<15, DIR, T, T2> : RDftCoprime<3, 5, DIR, T, T2> {};

// R = A A with constant twiddles
template <int A, int DIR, typename T, typename T2>
struct RDftSquare {
    static constexpr int R = A * A;
    static __device__ __forceinline__ void run(T2 (&v)[R]) {
        T2 t[A][A];
#pragma unroll
        for (int b = 0; b < A; b++) {
#pragma unroll
            for (int a = 0; a < A; a++) t[b][a] = v[A * a + b];
            RDft<A, DIR, T, T2>::run(t[b]);
#pragma unroll
            for (int a = 1; a < A; a++)
                if (b > 0) {
                    if (R == 16 && a * b == 4) t[b][a] = mul_is<DIR>(t[b][a]);
                    else t[b][a] = tmul(t[b][a], T2{(T)root_cos(R, a * b), (T)(DIR * root_sin(R, a * b))});
                }
        }
#pragma unroll
        for (int a = 0; a < A; a++) {
            T2 u[A];
#pragma unroll
            for (int b = 0; b < A; b++) u[b] = t[b][a];
            RDft<A, DIR, T, T2>::run(u);
#pragma unroll
            for (int b = 0; b < A; b++) v[a + A * b] = u[b];
        }
    }
};
template <int DIR, typename T, typename T2>
struct RDft<9, DIR, T, T2> : RDftSquare<3, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<16, DIR, T, T2> : RDftSquare<4, DIR, T, T2> {};

template <int R, int DIR, typename T, typename T2>
struct RDftPrime {
    static __device__ __forceinline__ void run(T2 (&v)[R]) {
        constexpr int H = (R - 1) / 2;
        T2 p[H], m[H];
#pragma unroll
        for (int j = 0; j < H; j++) {
            p[j] = cadd(v[j + 1], v[R - 1 - j]);
            m[j] = csub(v[j + 1], v[R - 1 - j]);
        }
        T2 s = v[0];
#pragma unroll
        for (int j = 0; j < H; j++) s = cadd(s, p[j]);
#pragma unroll
        for (int k = 1; k <= H; k++) {
            T2 a = v[0], b = T2{(T)0, (T)0};
#pragma unroll
            for (int j = 1; j <= H; j++) {
                const int q = (j * k) % R;
                const int h = q <= H ? q : R - q;
                const T c = (T)PrimeRoots<R>::c[h - 1];
                const T d = (T)(q <= H ? PrimeRoots<R>::s[h - 1] : -PrimeRoots<R>::s[h - 1]);
                a = T2{a.x + c * p[j - 1].x, a.y + c * p[j - 1].y};
                b = T2{b.x + d * m[j - 1].x, b.y + d * m[j - 1].y};
            }
            const T2 r = mul_is<DIR>(b);
            v[k] = cadd(a, r);
            v[R - k] = csub(a, r);
        }
        // v[0] is still the input's: every output above reads it
        v[0] = s;
    }
};
template <int DIR, typename T, typename T2>
struct RDft<7, DIR, T, T2> : RDftPrime<7, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<11, DIR, T, T2> : RDftPrime<11, DIR, T, T2> {};
template <int DIR, typename T, typename T2>
struct RDft<13, DIR, T, T2> : RDftPrime<13, DIR, T, T2> {};

// f with a compile-time radix equal to r
template <typename T, typename F, int R>
__device__ __forceinline__ void two_radix_call(std::integral_constant<int, R> r, F&& f) {
    f(r);
}
template <typename T, typename F>
__device__ __forceinline__ void two_radix_call(int r, F&& f) {
    constexpr bool fp64 = std::is_same<T, double>::value;
    switch (r) {
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        case 10: f(std::integral_constant<int, 10>{}); break;
        case 12: f(std::integral_constant<int, 12>{}); break;
        case 15: f(std::integral_constant<int, 15>{}); break;
        case 16: f(std::integral_constant<int, 16>{}); break;
        default:
            if constexpr (fp64) {
                switch (r) {
                    case 7: f(std::integral_constant<int, 7>{}); break;
                    case 11: f(std::integral_constant<int, 11>{}); break;
                    case 13: f(std::integral_constant<int, 13>{}); break;
                    case 14: f(std::integral_constant<int, 14>{}); break;
                    default: break;
                }
            }
    }
}

// v, opaque to the compiler where it is a value of the grid: the products r v of every radix's
// branch stay in the branch (they cost one scalar multiplication each there). Hoisted out of the
// loops they fill and spill the scalar registers: 390 spills in the FP64 slab kernel.
__device__ __forceinline__ int two_opaque(const TwoView&, int v) {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+s"(v));
#endif
    return v;
}
template <int N, int E>
__device__ __forceinline__ constexpr int two_opaque(const TwoCube<N, E>&, int v) {
    return v;
}

// ------------------------------------------------------------------ the plane of a slab
template <typename T, typename G>
struct TwoPlane {
    using T2 = typename vec2<T>::type;
    G g;
    T2* S;            // packed lines
    const T2 *Wy, *Wz;
    int tid, bd;

    // the slots of half-spectrum column c in a packed line: e holds Z[c], o holds Z[nz - c]
    struct Col {
        int e, o;
        bool self;    // c = nz - c (mod nz): one value, o is a spare slot
        // of row k1's values (a choice of values: one between the members would put them in memory)
        __device__ __forceinline__ int slot(int k1) const { return e + (k1 & 1) * (o - e); }
    };
    __device__ __forceinline__ int zslot(int k) const { return g.pad ? k + two_div(k, g.m_zr1) : k; }
    __device__ __forceinline__ Col column(int c) const {
        const int nz = g.z.L, end = nz + g.pad * g.zr2;
        if (c == 0) return Col{0, end, true};
        if (2 * c == nz) return Col{zslot(c), end + 1, true};
        return Col{zslot(c), zslot(nz - c), false};
    }

    // stage B of y for butterfly (column c, k1 = j), inverse: v holds rows j + r1 r of the column
    template <int R>
    __device__ __forceinline__ void y_scatter(T2 (&v)[R], const Col& q, int j) const {
        RDft<R, +1, T, T2>::run(v);
        const int pitch = two_opaque(g, g.pitch);
        T2* base = S + (j >> 1) * g.yr2 * pitch + q.slot(j);
#pragma unroll
        for (int r = 0; r < R; r++) base[r * pitch] = v[r];
    }
    // the LDS table's root for output r of butterfly j
    struct Table {
        const T2* W;
        __device__ __forceinline__ T2 operator()(int r, int j) const { return W[r * j]; }
    };
    // stage A of y, inverse, with the merge of the row pairs; w(r, j): the forward root W^(r j)
    __device__ __forceinline__ void y_merge() const { y_merge(Table{Wy}); }
    template <typename W>
    __device__ __forceinline__ void y_merge(const W& w) const {
        const int total = g.nzc * g.yr2;
        for (int t = tid; t < total; t += bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const Col q = column(c);
            two_radix_call<T>(g.yr1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                const int pair = two_opaque(g, g.yr2 * g.pitch);   // from line (a, j) to (a + 1, j)
                T2* const even = S + j * g.pitch + q.e;
                T2* const odd = S + j * g.pitch + q.o;
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = ((r & 1) ? odd : even)[(r >> 1) * pair];
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = tmul_conj(v[r], w(r, j));
                RDft<R, +1, T, T2>::run(v);
#pragma unroll
                for (int a = 0; a < (R + 1) / 2; a++) {
                    T2 A = v[2 * a], B = 2 * a + 1 < R ? v[(2 * a + 1) % R] : T2{(T)0, (T)0};
                    if (q.self) A.y = B.y = (T)0;
                    even[a * pair] = T2{A.x - B.y, A.y + B.x};
                    if (!q.self) odd[a * pair] = T2{A.x + B.y, B.x - A.y};
                }
            });
        }
    }
    // stage B of z: inverse (k natural -> (k1, n2)) or forward ((k1, n2) -> k natural)
    template <int DIR>
    __device__ __forceinline__ void z_outer() const {
        const int total = g.lines * g.zr1;
        for (int t = tid; t < total; t += bd) {
            const int line = two_div(t, g.m_zr1), j = t - line * g.zr1;
            T2* base = S + line * g.pitch + j;
            two_radix_call<T>(g.zr2, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                const int step = two_opaque(g, g.zr1 + g.pad);
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = base[r * step];
                RDft<R, DIR, T, T2>::run(v);
#pragma unroll
                for (int r = 0; r < R; r++) base[r * step] = v[r];
            });
        }
    }
    // Stage A of z both ways around the real values: op(i, two, v) gets the index of a value of the
    // pair's first row, whether the second row exists (at i + second), and both values in v.x and
    // v.y; it returns through them what the forward transform takes.
    template <typename Op>
    __device__ __forceinline__ void z_inner(bool inverse, bool forward, Op&& op) const {
        const int total = g.lines * g.zr2;
        const int nz = g.z.L;
        for (int t = tid; t < total; t += bd) {
            const int line = two_div(t, g.m_zr2), j = t - line * g.zr2;
            const int a = two_div(line, g.m_yr2);
            const int row = line + a * g.yr2;    // (2 a) r2 + n2 with line = a r2 + n2
            const bool two = 2 * a + 1 < g.yr1;
            const int i0 = row * nz + j;
            T2* base = S + line * g.pitch + j * (g.zr1 + g.pad);
            two_radix_call<T>(g.zr1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                if (inverse) {
#pragma unroll
                    for (int r = 0; r < R; r++) v[r] = base[r];
#pragma unroll
                    for (int r = 1; r < R; r++) v[r] = tmul_conj(v[r], Wz[r * j]);
                    RDft<R, +1, T, T2>::run(v);
                }
                const int run = two_opaque(g, g.zr2);
#pragma unroll
                for (int r = 0; r < R; r++) op(i0 + r * run, two, v[r]);
                if (forward) {
                    RDft<R, -1, T, T2>::run(v);
#pragma unroll
                    for (int r = 1; r < R; r++) v[r] = tmul(v[r], Wz[r * j]);
#pragma unroll
                    for (int r = 0; r < R; r++) base[r] = v[r];
                }
            });
        }
    }
    // stage A of y, forward, with the split of the packed lines (twice the rows' spectra: the
    // caller halves the real values)
    __device__ __forceinline__ void y_split() const { y_split(Table{Wy}); }
    template <typename W>
    __device__ __forceinline__ void y_split(const W& w) const {
        const int total = g.nzc * g.yr2;
        for (int t = tid; t < total; t += bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const Col q = column(c);
            two_radix_call<T>(g.yr1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                const int pair = two_opaque(g, g.yr2 * g.pitch);
                T2* const even = S + j * g.pitch + q.e;
                T2* const odd = S + j * g.pitch + q.o;
#pragma unroll
                for (int a = 0; a < (R + 1) / 2; a++) {
                    const T2 A = even[a * pair];
                    const T2 B = q.self ? A : odd[a * pair];
                    v[2 * a] = T2{A.x + B.x, A.y - B.y};
                    if (2 * a + 1 < R) v[(2 * a + 1) % R] = T2{A.y + B.y, B.x - A.x};
                }
                RDft<R, -1, T, T2>::run(v);
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = tmul(v[r], w(r, j));
#pragma unroll
                for (int r = 0; r < R; r++) ((r & 1) ? odd : even)[(r >> 1) * pair] = v[r];
            });
        }
    }
    // stage B of y, forward: v[r] becomes row j + r1 r of the column
    template <int R>
    __device__ __forceinline__ void y_gather(T2 (&v)[R], const Col& q, int j) const {
        const int pitch = two_opaque(g, g.pitch);
        const T2* base = S + (j >> 1) * g.yr2 * pitch + q.slot(j);
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = base[r * pitch];
        RDft<R, -1, T, T2>::run(v);
    }
};

// ------------------------------------------------------------------ slab pass
// The pass of fts_fft.hpp's slab_kernel (same items, modes and results) for grids with a
// TwoGeom; spectra have rows of g.sp values. INV2 items must have qout: the first half step
// waits there. ROOT: FP64 items of two spectra, whose second one takes the root of the factor; the other
// launches go without that code (with it, discrete FP64 steps took 3 to 4% longer for its registers).
template <bool ROOT, typename T, typename G>
__device__ __forceinline__ void slab_two(const G& g, int mode, int bd, const SlabBatch<T>& batch,
                                         const typename vec2<T>::type* twy, const typename vec2<T>::type* twz) {
    using T2 = typename vec2<T>::type;
    using Plane = TwoPlane<T, G>;
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wy = S + g.lines * g.pitch;
    T2* Wz = Wy + g.y.L;
    for (int m = threadIdx.x; m < g.y.L; m += bd) Wy[m] = twy[m];
    for (int m = threadIdx.x; m < g.z.L; m += bd) Wz[m] = twz[m];
    const SlabItem<T>& it = batch.it[blockIdx.y];
    const int ny = g.y.L, nz = g.z.L;
    const size_t roff = (size_t)blockIdx.x * ny * nz;
    const size_t coff = (size_t)blockIdx.x * ny * g.sp;
    const T inv_m = (T)g.inv_m;
    const bool has_w = it.w != nullptr;
    const T* w = has_w ? it.w + roff : nullptr;
    const T* mask = it.mask ? it.mask + roff : nullptr;
    T* qout = it.qout ? it.qout + roff : nullptr;
    const int second = g.yr2 * nz;   // from a value of a pair's first row to the second's
    const Plane pl{g, S, Wy, Wz, (int)threadIdx.x, bd};

    // FWD: n_out forward transforms of qin. INV1: inverse, store, forward. INV2: the inverse of
    // the full step (parked in qout); that of the half steps, combined with it, and the first
    // forward transform; the second from qout.
    const bool go_on = mode == SLAB_FWD || it.forward != 0;
    const int n_iter = mode == SLAB_FWD ? it.n_out : mode == SLAB_INV1 ? 1 : (go_on ? 3 : 2);
    for (int s = 0; s < n_iter; s++) {
        const bool inverse = mode == SLAB_INV1 || (mode == SLAB_INV2 && s < 2);
        const bool park = mode == SLAB_INV2 && s == 0;
        const bool comb = mode == SLAB_INV2 && s == 1;
        const bool forward = go_on && !park;
        const int out = mode == SLAB_INV2 ? s - 1 : s;   // which spectrum the forward transform writes
        __syncthreads();   // twiddles stored; the previous use of the plane is over
        if (inverse) {
            const T2* spec = (comb ? it.c1 : it.c0) + coff;
            const int total = g.nzc * g.yr1;
            for (int t = pl.tid; t < total; t += pl.bd) {
                const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
                const typename Plane::Col q = pl.column(c);
                two_radix_call<T>(g.yr2, [&](auto RC) {
                    constexpr int R = decltype(RC)::value;
                    T2 v[R];
                    const T2* src = spec + j * g.sp + c;
                    const int rows = two_opaque(g, g.yr1 * g.sp);
#pragma unroll
                    for (int r = 0; r < R; r++) v[r] = src[r * rows];
                    pl.template y_scatter<R>(v, q, j);
                });
            }
            __syncthreads();
            pl.y_merge();
            __syncthreads();
            pl.template z_outer<+1>();
            __syncthreads();
        }
        const T post = comb ? it.post1 : it.post0;
        const T pre = out == 1 ? it.pre1 : it.pre0;
        const T* load = mode == SLAB_FWD ? it.qin + roff : (inverse ? nullptr : qout);
        auto real = [&](int i, T v) -> T {
            const T wv = has_w ? w[i] : (T)0;
            if (inverse) {
                v = v * (ROOT ? factor<T>(wv, has_w, post) : factor_at<false>(wv, has_w, post)) * inv_m;
                if (comb) v = ((T)4.0 * v - qout[i]) / (T)3.0;
                if (!park && mask) v *= mask[i];
                if (qout) qout[i] = v;
            } else {
                v = load[i];
            }
            if (!forward) return v;
            return v * (ROOT ? factor<T>(wv, has_w, pre) : factor_at<false>(wv, has_w, pre)) * (T)0.5;
        };
        pl.z_inner(inverse, forward, [&](int i, bool two, T2& v) {
            v.x = real(i, v.x);
            v.y = two ? real(i + second, v.y) : (T)0;
        });
        if (!forward) continue;
        __syncthreads();
        pl.template z_outer<-1>();
        __syncthreads();
        pl.y_split();
        __syncthreads();
        T2* spec = (out == 1 ? it.c1 : it.c0) + coff;
        const int total = g.nzc * g.yr1;
        for (int t = pl.tid; t < total; t += pl.bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const typename Plane::Col q = pl.column(c);
            two_radix_call<T>(g.yr2, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                pl.template y_gather<R>(v, q, j);
                T2* dst = spec + j * g.sp + c;
                const int rows = two_opaque(g, g.yr1 * g.sp);
#pragma unroll
                for (int r = 0; r < R; r++) dst[r * rows] = v[r];
            });
        }
    }
}

template <typename T, bool ROOT>
__global__ void __launch_bounds__(TWO_BD) slab_two_kernel(TwoGeom g, int mode, SlabBatch<T> batch,
                                                          const typename vec2<T>::type* twy,
                                                          const typename vec2<T>::type* twz) {
    slab_two<ROOT, T>(TwoView(g), mode, blockDim.x, batch, twy, twz);
}
// The same pass for an N^3 grid with the plan, the workgroup size and the number of butterflies
// per thread as constants. The real values of a thread's z butterflies stay in registers from
// the inverse to the last forward transform, and every global load is issued a phase or more before
// its use: the first spectrum and w before the first barrier, the second spectrum of a
// Richardson step when the first has left its registers.
template <typename T, int MODE, int N, int BD>
struct CubeSlab {
    using T2 = typename vec2<T>::type;
    using G = TwoCube<N, sizeof(T2)>;
    static constexpr int YT = (G::nzc * G::y.r1 + BD - 1) / BD;    // y stage B butterflies per thread
    static constexpr int ZT = (G::lines * G::z.r2 + BD - 1) / BD;  // z stage A butterflies per thread
    static constexpr int RY = G::y.r2, RZ = G::z.r1;
    // w stays in registers for the whole kernel unless its values, the real values and a butterfly
    // of the largest radix exceed the registers of BD threads
    static constexpr int VGPRS = BD > 512 ? 128 : 256;
    static constexpr int WORDS = sizeof(T) / 4;
    static constexpr bool W_RESIDENT = WORDS * (2 * 2 * ZT * RZ + 2 * 16) <= VGPRS - 40;
    // the second spectrum is loaded ahead when that many registers are left
    static constexpr bool AHEAD = WORDS * (2 * 2 * ZT * RZ + 2 * YT * RY + 2 * 16) <= VGPRS - 40;
    // Where every stage has at most one butterfly per thread, the roots a thread needs can stay in
    // registers, read from the tables in HBM before the first barrier, instead of 4 (r1 - 1) LDS
    // reads per transform pair. The shapes of few workgroups do: 64^3 with 320 threads 9.3 -> 8.9 and
    // 15.8 -> 15.2 us (half step, Richardson step of two propagators in FP64), 32^3 5.1 -> 4.8. In the
    // shapes of large batches the registers cost workgroups per CU (64^3 with 512 threads, 16
    // propagators: 27 -> 37 us; the Richardson step of 32 propagators at 32^3: 14.6 -> 18.1 us). 48^3 with
    // 256 threads, its only default, has one butterfly per thread too and keeps the tables: in registers,
    // evaluations of 2 propagators took 0.97 to 0.99 of the time in FP64, of 16 discrete ones 1.04, in FP32 1.05
    // to 1.09 with 16.
    static constexpr bool ROOTS =
        (sizeof(T) == 8 && N == 64 && BD == 320) || (N == 32 && BD == 256 && MODE != SLAB_INV2);
    static_assert(!ROOTS || (ZT == 1 && G::nzc * G::y.r2 <= BD), "one butterfly per thread");
};

template <typename T, int MODE, int N, int BD>
__global__ void __launch_bounds__(BD) slab_cube_kernel(SlabBatch<T> batch, const typename vec2<T>::type* twy,
                                                       const typename vec2<T>::type* twz) {
    using T2 = typename vec2<T>::type;
    using K = CubeSlab<T, MODE, N, BD>;
    using G = typename K::G;
    using Plane = TwoPlane<T, G>;
    constexpr int YT = K::YT, ZT = K::ZT, RY = K::RY, RZ = K::RZ;
    constexpr int Y_TASKS = G::nzc * G::y.r1, Z_TASKS = G::lines * G::z.r2;
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wy = S + G::lines * G::pitch;
    T2* Wz = Wy + N;
    const int tid = threadIdx.x;
    const SlabItem<T>& it = batch.it[blockIdx.y];
    const size_t roff = (size_t)blockIdx.x * N * N, coff = (size_t)blockIdx.x * N * G::sp;
    const T inv_m = (T)G::inv_m;
    const bool has_w = it.w != nullptr;
    constexpr G g{};
    const Plane pl{g, S, Wy, Wz, tid, BD};
    constexpr int SECOND = G::y.r2 * N;   // from a value of a pair's first row to the second's

    // y stage B butterfly k of this thread: column and k1
    auto y_task = [&](int k, int& c, int& j) {
        const int t = tid + k * BD;
        j = t / G::nzc;
        c = t - j * G::nzc;
        return Y_TASKS % BD == 0 || t < Y_TASKS;
    };
    auto fetch = [&](const T2* spec, T2 (&v)[YT][RY]) {
#pragma unroll
        for (int k = 0; k < YT; k++) {
            int c, j;
            if (y_task(k, c, j)) {
#pragma unroll
                for (int r = 0; r < RY; r++) v[k][r] = spec[(j + r * G::y.r1) * G::sp + c];
            }
        }
    };
    // z stage A butterfly k: its LDS values and the index of its first real value
    auto z_task = [&](int k, int& j, T2*& base, int& i0) {
        const int t = tid + k * BD;
        const int line = t / G::z.r2;
        j = t - line * G::z.r2;
        base = S + line * G::pitch + j * (G::z.r1 + G::pad);
        i0 = (line + line / G::y.r2 * G::y.r2) * N + j;
        return Z_TASKS % BD == 0 || t < Z_TASKS;
    };
    T we[ZT][RZ], wo[ZT][RZ];
    auto fetch_real = [&](const T* src, T (&e)[ZT][RZ], T (&o)[ZT][RZ]) {
#pragma unroll
        for (int k = 0; k < ZT; k++) {
            int j, i0;
            T2* base;
            if (z_task(k, j, base, i0)) {
#pragma unroll
                for (int r = 0; r < RZ; r++) {
                    e[k][r] = src[i0 + r * G::z.r2];
                    o[k][r] = src[i0 + r * G::z.r2 + SECOND];
                }
            }
        }
    };
    auto fetch_w = [&] {
        if (has_w) fetch_real(it.w + roff, we, wo);
    };
    constexpr int NR = K::ROOTS ? 1 : 0;
    T2 ry[NR * G::y.r1 + 1], rz[NR * G::z.r1 + 1];
    auto load_twiddles = [&] {
        if constexpr (K::ROOTS) {
            const int jy = min(tid / G::nzc, G::y.r2 - 1), jz = tid % G::z.r2;
#pragma unroll
            for (int r = 1; r < G::y.r1; r++) ry[r] = twy[r * jy];
#pragma unroll
            for (int r = 1; r < G::z.r1; r++) rz[r] = twz[r * jz];
        } else {
            for (int m = tid; m < N; m += BD) {
                Wy[m] = twy[m];
                Wz[m] = twz[m];
            }
        }
    };
    auto y_root = [&](int r, int j) { return K::ROOTS ? ry[NR * r] : Wy[r * j]; };
    auto z_root = [&](int r, int j) { return K::ROOTS ? rz[NR * r] : Wz[r * j]; };
    T qe[ZT][RZ], qo[ZT][RZ];
    // a fetched spectrum -> real values times factor(coef) / M; COMB: (4 x - q) / 3 against the
    // values already in q. `between`: loads to issue once the spectrum has left its registers.
    auto inverse = [&](T2 (&v)[YT][RY], T coef, auto comb, auto&& between) {
        constexpr bool COMB = decltype(comb)::value;
#pragma unroll
        for (int k = 0; k < YT; k++) {
            int c, j;
            if (y_task(k, c, j)) pl.template y_scatter<RY>(v[k], pl.column(c), j);
        }
        between();
        __syncthreads();
        pl.y_merge(y_root);
        __syncthreads();
        if constexpr (!K::W_RESIDENT) fetch_w();
        pl.template z_outer<+1>();
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ZT; k++) {
            int j, i0;
            T2* base;
            if (z_task(k, j, base, i0)) {
                T2 u[RZ];
#pragma unroll
                for (int r = 0; r < RZ; r++) u[r] = base[r];
#pragma unroll
                for (int r = 1; r < RZ; r++) u[r] = tmul_conj(u[r], z_root(r, j));
                RDft<RZ, +1, T, T2>::run(u);
#pragma unroll
                for (int r = 0; r < RZ; r++) {
                    const T xe = u[r].x * factor_at<COMB>(we[k][r], has_w, coef) * inv_m;
                    const T xo = u[r].y * factor_at<COMB>(wo[k][r], has_w, coef) * inv_m;
                    qe[k][r] = COMB ? ((T)4.0 * xe - qe[k][r]) / (T)3.0 : xe;
                    qo[k][r] = COMB ? ((T)4.0 * xo - qo[k][r]) / (T)3.0 : xo;
                }
            }
        }
    };
    // real values times factor(coef) -> spectrum
    auto forward = [&](T coef, auto root, T2* spec) {
        constexpr bool ROOT = decltype(root)::value;
#pragma unroll
        for (int k = 0; k < ZT; k++) {
            int j, i0;
            T2* base;
            if (z_task(k, j, base, i0)) {
                T2 u[RZ];
#pragma unroll
                for (int r = 0; r < RZ; r++)
                    u[r] = T2{qe[k][r] * factor_at<ROOT>(we[k][r], has_w, coef) * (T)0.5,
                              qo[k][r] * factor_at<ROOT>(wo[k][r], has_w, coef) * (T)0.5};
                RDft<RZ, -1, T, T2>::run(u);
#pragma unroll
                for (int r = 1; r < RZ; r++) u[r] = tmul(u[r], z_root(r, j));
#pragma unroll
                for (int r = 0; r < RZ; r++) base[r] = u[r];
            }
        }
        __syncthreads();
        pl.template z_outer<-1>();
        __syncthreads();
        pl.y_split(y_root);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < YT; k++) {
            int c, j;
            if (y_task(k, c, j)) {
                T2 v[RY];
                pl.template y_gather<RY>(v, pl.column(c), j);
#pragma unroll
                for (int r = 0; r < RY; r++) spec[(j + r * G::y.r1) * G::sp + c] = v[r];
            }
        }
    };

    int n_out = 1;
    if constexpr (MODE == SLAB_FWD) {
        fetch_real(it.qin + roff, qe, qo);
        fetch_w();
        load_twiddles();
        __syncthreads();
        n_out = it.n_out;
    } else {
        T2 v[YT][RY];
        fetch(it.c0 + coff, v);
        if constexpr (K::W_RESIDENT) fetch_w();
        load_twiddles();
        __syncthreads();
        if constexpr (MODE == SLAB_INV1) {
            inverse(v, it.post0, std::false_type{}, [] {});
        } else {
            inverse(v, it.post0, std::false_type{}, [&] {
                if constexpr (K::AHEAD) fetch(it.c1 + coff, v);
            });
            if constexpr (!K::AHEAD) fetch(it.c1 + coff, v);
            __syncthreads();   // the plane's values are read
            inverse(v, it.post1, std::true_type{}, [] {});
            n_out = 2;
        }
#pragma unroll
        for (int k = 0; k < ZT; k++) {
            int j, i0;
            T2* base;
            if (z_task(k, j, base, i0)) {
#pragma unroll
                for (int r = 0; r < RZ; r++) {
                    const size_t ie = roff + i0 + r * G::z.r2, io = ie + SECOND;
                    if (it.mask) {
                        qe[k][r] *= it.mask[ie];
                        qo[k][r] *= it.mask[io];
                    }
                    if (it.qout) {
                        it.qout[ie] = qe[k][r];
                        it.qout[io] = qo[k][r];
                    }
                }
            }
        }
        if (!it.forward) return;
    }
    forward(it.pre0, std::false_type{}, it.c0 + coff);
    if (n_out < 2) return;
    __syncthreads();   // the plane of the first spectrum is read
    forward(it.pre1, std::true_type{}, it.c1 + coff);
}

// ------------------------------------------------------------------ pencil (x) pass
// One wavefront per y row and tile of C kz columns.
__device__ __forceinline__ void two_wave_sync() {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#else
    __syncthreads();
#endif
}

template <int C, typename T, typename G>
__device__ __forceinline__ void pencil_two(const G& g, int jy, int k0, const XItem<T>& it,
                                           const typename vec2<T>::type* twx, const T* bx, const T* by, const T* bz) {
    using T2 = typename vec2<T>::type;
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    const int group = two_pencil_group(g.xr2, C, sizeof(T2));   // slots of one k1
    T2* Wx = S + g.xr1 * group;
    const int lane = threadIdx.x;
    for (int m = lane; m < g.x.L; m += 64) Wx[m] = twx[m];
    const int cw = min(C, g.nzc - k0);
    const int row = g.y.L * g.sp;
    T2* c = it.c + (size_t)jy * g.sp + k0;
    const int table = it.table;
    const auto r1 = g.xr1;
    const auto r2 = g.xr2;
    // FP32: the x line of ky = kz = 0 holds the planes' means, the rest of it is small. The value of
    // the first plane passes by the transforms (its bond factor is 1) and is added to what they
    // leave of the differences, so the field's mean is not rounded to an FP32 sum of all points
    // in every convolution (that error, 4e-8 at random, made up most of Q's after 100 steps).
    const bool mean = sizeof(T) == sizeof(float) && table >= 0 && jy == 0 && k0 == 0;
    const T first = mean ? c[0].x : (T)0;
    if (table != -2) {
        two_wave_sync();   // twiddles
        for (int t = lane; t < C * r2; t += 64) {
            const int j = t / C, l = t % C;
            if (l >= cw) continue;
            two_radix_call<T>(r1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                const T2* src = c + (size_t)(j * row + l);
                const int next = two_opaque(g, r2 * row);
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = src[r * next];
                if (mean && l == 0) {
#pragma unroll
                    for (int r = 0; r < R; r++) v[r].x -= first;
                }
                RDft<R, -1, T, T2>::run(v);
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = tmul(v[r], Wx[r * j]);
#pragma unroll
                for (int r = 0; r < R; r++) S[r * two_opaque(g, group) + j * C + l] = v[r];
            });
        }
        two_wave_sync();
    }
    for (int t = lane; t < C * r1; t += 64) {
        const int j = t / C, l = t % C;
        if (l >= cw) continue;
        T2* base = S + j * group + l;
        two_radix_call<T>(r2, [&](auto RC) {
            constexpr int R = decltype(RC)::value;
            T2 v[R];
            if (table != -2) {
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = base[r * C];
                RDft<R, -1, T, T2>::run(v);
                if (table == -1) {
#pragma unroll
                    for (int r = 0; r < R; r++) c[(j + r * r1) * row + l] = v[r];
                    return;
                }
                const T* tx = bx + (size_t)table * g.x.L + j;
                const T bl = by[(size_t)table * g.y.L + jy] * bz[(size_t)table * g.nzc + k0 + l];
                const int next = two_opaque(g, r1);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const T b = tx[r * next] * bl;
                    v[r] = T2{v[r].x * b, v[r].y * b};
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = c[(j + r * r1) * row + l];
            }
            RDft<R, +1, T, T2>::run(v);
#pragma unroll
            for (int r = 0; r < R; r++) base[r * C] = v[r];
        });
    }
    if (table == -1) return;
    two_wave_sync();
    for (int t = lane; t < C * r2; t += 64) {
        const int j = t / C, l = t % C;
        if (l >= cw) continue;
        two_radix_call<T>(r1, [&](auto RC) {
            constexpr int R = decltype(RC)::value;
            T2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = S[r * two_opaque(g, group) + j * C + l];
#pragma unroll
            for (int r = 1; r < R; r++) v[r] = tmul_conj(v[r], Wx[r * j]);
            RDft<R, +1, T, T2>::run(v);
            if (mean && l == 0) {
                // the slab pass scales by 1 / M rounded to T: the difference belongs to the mean too.
                // The forward and the inverse transform along x scale the differences by nx.
                const T nx = (T)g.x.L;
                const T scale = (T)(1.0 - g.inv_m / (double)(T)g.inv_m);
#pragma unroll
                for (int r = 0; r < R; r++) v[r].x = first * nx + (v[r].x - first * nx * scale);
            }
#pragma unroll
            for (int r = 0; r < R; r++) c[r * two_opaque(g, r2 * row) + j * row + l] = v[r];
        });
    }
}

// a tile of one 128-byte line per wavefront
template <typename T>
__global__ void __launch_bounds__(64) pencil_two_kernel(TwoGeom g, XBatch<T> batch,
                                                        const typename vec2<T>::type* twx, const T* bx, const T* by,
                                                        const T* bz) {
    constexpr int C = 128 / (int)sizeof(typename vec2<T>::type);
    const int tiles = (g.nzc + C - 1) / C;
    const int jy = blockIdx.x / tiles;
    pencil_two<C>(TwoView(g), jy, (blockIdx.x - jy * tiles) * C, batch.it[blockIdx.y], twx, bx, by, bz);
}

// Pencil tiles narrower than a 128-byte line share that line of a spectrum row (rows start
// on a line) with SH - 1 neighbours. Workgroups go to the 8 XCDs round-robin by linear id,
// and each XCD has its own L2, so neighbouring tiles would each fetch the line. The grid
// then pads a row's tiles to a whole number of lines, and xcd_tile orders the tiles so that
// the SH tiles of one line get ids 8 apart: one XCD, one fetch.
template <typename T2, int NL>
constexpr int cube_pencil_share() {
    return 128 / (NL * (int)sizeof(T2)) > 1 ? 128 / (NL * (int)sizeof(T2)) : 1;
}
template <typename T2, int N, int NL>
constexpr int cube_pencil_tiles() {
    constexpr int SH = cube_pencil_share<T2, NL>();
    return ((N / 2 + 1 + NL - 1) / NL + SH - 1) / SH * SH;
}
// tile of block b: b = 8 SH g + 8 s + k (k < 8, s < SH) takes tile SH (8 g + k) + s; a
// bijection when the grid's x extent is a multiple of 8 SH (N x a multiple of SH, N % 8 == 0)
template <int SH>
__device__ __forceinline__ int xcd_tile(int b) {
    if constexpr (SH == 1) {
        return b;
    } else {
        const int g = b / (8 * SH), r = b - g * 8 * SH;
        return SH * (8 * g + (r & 7)) + (r >> 3);
    }
}
template <typename T, int N, int NL>
__global__ void __launch_bounds__(64) pencil_cube_kernel(XBatch<T> batch, const typename vec2<T>::type* twx,
                                                         const T* bx, const T* by, const T* bz) {
    using T2 = typename vec2<T>::type;
    constexpr int TILES = cube_pencil_tiles<T2, N, NL>();
    static_assert(N % 8 == 0, "the XCD tile order needs a grid extent of a multiple of 8 lines' tiles");
    const int b = xcd_tile<cube_pencil_share<T2, NL>()>(blockIdx.x);
    const int jy = b / TILES, k0 = (b - jy * TILES) * NL;
    if (k0 > N / 2) return;   // a pad tile: the whole wavefront leaves
    pencil_two<NL>(TwoCube<N, sizeof(T2)>{}, jy, k0, batch.it[blockIdx.y], twx, bx, by, bz);
}

// ------------------------------------------------------------------ whole steps of flat grids
// A grid of one x-slab (one and two dimensions) holds its whole transform in one workgroup's
// LDS: the bond factors apply between the forward and the inverse y stage B in registers, and a
// workgroup runs all consecutive steps of a propagator in one launch.
template <typename T, bool CONTINUOUS>
__global__ void __launch_bounds__(TWO_BD) flat_steps_kernel(TwoGeom geom, FlatBatch<T> batch,
                                                            const typename vec2<T>::type* twy,
                                                            const typename vec2<T>::type* twz, const T* by,
                                                            const T* bz) {
    using T2 = typename vec2<T>::type;
    using Plane = TwoPlane<T, TwoView>;
    const TwoView g(geom);
    const int bd = blockDim.x;
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wy = S + g.lines * g.pitch;
    T2* Wz = Wy + g.y.L;
    for (int m = threadIdx.x; m < g.y.L; m += blockDim.x) Wy[m] = twy[m];
    for (int m = threadIdx.x; m < g.z.L; m += blockDim.x) Wz[m] = twz[m];
    const FlatItem<T>& it = batch.it[blockIdx.x];
    const int second = g.yr2 * g.z.L;
    const T inv_m = (T)g.inv_m;
    const Plane pl{g, S, Wy, Wz, (int)threadIdx.x, bd};
    const T* mask = it.mask;
    // convolutions per step: continuous full step, half step, half step; discrete one
    constexpr int NCONV = CONTINUOUS ? 3 : 1;
    const int rounds = it.steps * NCONV;
    __syncthreads();
    for (int s = 0; s <= rounds; s++) {
        // the values between convolution s - 1 and s: what the inverse left, then what the next
        // forward transform takes
        const bool inverse = s > 0, forward = s < rounds;
        const int prev = (s + NCONV - 1) % NCONV, next = s % NCONV;
        const int n = (s + NCONV - 1) / NCONV;   // CONTINUOUS, prev = 2: this pass completes slice n
        T* qn = it.q + (size_t)(s / NCONV) * batch.stride;          // slice the current step starts from
        T* qdone = it.q + (size_t)n * batch.stride;
        auto real = [&](int i, T v) -> T {
            const T wv = it.w[i];
            if constexpr (!CONTINUOUS) {
                if (inverse) {
                    v = v * factor_at<false>(wv, true, it.full_w) * inv_m;
                    if (mask) v *= mask[i];
                    qdone[i] = v;
                } else {
                    v = qn[i];
                }
                return v * (T)0.5;
            } else {
                if (inverse) {
                    v = v * (prev == 2 ? factor_at<true>(wv, true, it.half_w) : factor_at<false>(wv, true, it.full_w)) * inv_m;
                    if (prev == 0) {
                        it.half[i] = v;
                        v = qn[i];
                    } else if (prev == 2) {
                        v = ((T)4.0 * v - it.half[i]) / (T)3.0;
                        if (mask) v *= mask[i];
                        qdone[i] = v;
                    }
                } else {
                    v = qn[i];
                }
                if (next == 0) v *= factor_at<false>(wv, true, it.full_w);
                else if (next == 1) v *= factor_at<true>(wv, true, it.half_w);
                return v * (T)0.5;
            }
        };
        pl.z_inner(inverse, forward, [&](int i, bool two, T2& v) {
            v.x = real(i, v.x);
            v.y = two ? real(i + second, v.y) : (T)0;
        });
        if (!forward) break;
        __syncthreads();
        pl.template z_outer<-1>();
        __syncthreads();
        pl.y_split();
        __syncthreads();
        // stage B of y both ways, with the bond factors between them
        const int table = CONTINUOUS && next > 0 ? it.half_table : it.full_table;
        const T* ty = by + (size_t)table * g.y.L;
        const T* tz = bz + (size_t)table * g.nzc;
        const int total = g.nzc * g.yr1;
        for (int t = pl.tid; t < total; t += pl.bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const typename Plane::Col q = pl.column(c);
            two_radix_call<T>(g.yr2, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                pl.template y_gather<R>(v, q, j);
                const T b = tz[c];
                const int rows = two_opaque(g, g.yr1);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const T f = ty[j + r * rows] * b;
                    v[r] = T2{v[r].x * f, v[r].y * f};
                }
                pl.template y_scatter<R>(v, q, j);
            });
        }
        __syncthreads();
        pl.y_merge();
        __syncthreads();
        pl.template z_outer<+1>();
        __syncthreads();
    }
}

// ------------------------------------------------------------------ whole steps in one dimension
// A line of up to LINE_POINTS points takes its convolutions directly: the bond factors' inverse
// transform is a row of n coefficients, and a thread group sums a point's n products, every
// value in LDS or registers. Two barriers per Richardson step (a buffer is written again only two
// barriers after its readers), where two butterflies each way and
// the row pairing (with an empty partner) take eighteen: a step of 128 points took 23 us by
// flat_steps_kernel, bound by those phases' latency, and takes 2.2 us (50 steps of two propagators: 110 us). Sums are FP64 in either
// precision.
template <typename T, bool CONTINUOUS, int P, int CH>
__global__ void __launch_bounds__(1024) line_steps_kernel(int n, FlatBatch<T> batch, const T* bz) {
    FTS_DYNAMIC_LDS(smem_raw);
    double* full = reinterpret_cast<double*>(smem_raw);   // coefficients of the full and the half bond
    double* half = full + n;
    double* xa = half + n;                                // inputs of the three convolutions, two buffers each
    double* xb = xa + 2 * n;
    double* xc = xb + 2 * n;
    double* parts = xc + 2 * n;                           // partial sums of the coefficients
    const FlatItem<T>& it = batch.it[blockIdx.x];
    const int nzc = n / 2 + 1;
    // P neighbouring lanes share point i; lane p takes the inputs j = p (mod P)
    const int i = threadIdx.x / P, p = threadIdx.x % P;
    const bool on = i < n;
    for (int m = threadIdx.x; m < n; m += blockDim.x) {
        // cos(2 pi m / n) by its symmetries, so that a period's values cancel
        const int h = min(m, n - m);
        xa[m] = 4 * h <= n ? cospi(2.0 * h / n) : -cospi((double)(n - 2 * h) / n);
        if (m < nzc) {
            xb[m] = (double)bz[(size_t)it.full_table * nzc + m];
            if (CONTINUOUS) xc[m] = (double)bz[(size_t)it.half_table * nzc + m];
        }
    }
    __syncthreads();
    for (int m = threadIdx.x; m < (CONTINUOUS ? 2 : 1) * n; m += blockDim.x) {
        const int d = m < n ? m : m - n;
        const double* b = m < n ? xb : xc;
        // compensated: the coefficients' errors act the same way in every step
        double sum = b[0], lost = 0.0;
        int a = 0;   // k d mod n
        for (int k = 1; k < nzc; k++) {
            a += d;
            if (a >= n) a -= n;
            const double y = (2 * k == n ? 1.0 : 2.0) * (b[k] * xa[a]) - lost;
            const double next = sum + y;
            lost = (next - sum) - y;
            sum = next;
        }
        full[m] = sum / n;
    }
    __syncthreads();
    // The coefficients add up to b[0]: what rounding left of that would scale the field's mean in every
    // step (half an ulp of c[0] is 2^-54 a convolution: 1e-14 after 100 steps, 3 to 4 times the error of
    // transforms at 16 and 64 points). The roots' errors, which leave much the same in every
    // coefficient, go back evenly, where only the mean sees it; then c[0] takes the rest, and
    // its neighbours in turn what the finer grid of their values holds of it, nearest first, where every
    // mode of a smooth field weighs them alike.
    constexpr int BONDS = CONTINUOUS ? 2 : 1;
    const bool owner = threadIdx.x < BONDS;
    double* c = threadIdx.x == 0 ? full : half;
    // b[0] less the coefficients, every addition with its rounding error: LINE_PARTS partial sums, then the
    // owner of a bond adds them (one thread's walk over 128 coefficients is 2 us of a launch)
    auto rest = [&] {
        if (threadIdx.x < BONDS * LINE_PARTS) {
            const double* v = full + threadIdx.x / LINE_PARTS * n;
            double s = 0.0, lost = 0.0;
            for (int k = threadIdx.x % LINE_PARTS; k < n; k += LINE_PARTS) {
                const double t = s + v[k], z = t - s;
                lost += (s - (t - z)) + (v[k] - z);
                s = t;
            }
            parts[2 * threadIdx.x] = s;
            parts[2 * threadIdx.x + 1] = lost;
        }
        __syncthreads();
        double s = threadIdx.x == 0 ? xb[0] : xc[0], lost = 0.0;
        if (owner)
            for (int k = LINE_PARTS * threadIdx.x; k < LINE_PARTS * (threadIdx.x + 1); k++) {
                const double x = -parts[2 * k], t = s + x, z = t - s;
                lost += (s - (t - z)) + (x - z) - parts[2 * k + 1];
                s = t;
            }
        return s + lost;
    };
    double left = rest();
    if (owner) xa[threadIdx.x] = left / n;
    __syncthreads();
    for (int m = threadIdx.x; m < BONDS * n; m += blockDim.x) full[m] += xa[m < n ? 0 : 1];
    __syncthreads();
    left = rest();
    if (owner) {
        // 2^-61: 1e-16 of the mean after 300 convolutions
        for (int d = 0; 2 * d <= n && fabs(left) > 0x1p-61; d++) {
            const int e = d == 0 ? 0 : n - d;
            const double share = e == d ? left : 0.5 * left;
            const double a = c[d] + share;
            left -= a - c[d];
            c[d] = a;
            if (e != d) {
                const double b = c[e] + share;
                left -= b - c[e];
                c[e] = b;
            }
        }
    }
    __syncthreads();
    T* q = it.q;
    // discrete: exp(-w ds), in e2; continuous: exp(-w ds/2) and exp(-w ds/4), as the slab passes take them
    const T f = on ? it.w[i] : (T)0;
    const double e2 = (double)factor<T>(f, true, it.full_w);
    const double e4 = CONTINUOUS ? (double)factor<T>(f, true, it.half_w) : 0.0;
    const double mask = on && it.mask ? (double)it.mask[i] : 1.0;
    double x = on ? (double)q[i] : 0.0;
    // this lane's coefficients c[(i - j) mod n] of j = p + P t, and the places of v[j]: in registers
    // for all steps (CH of them, those beyond the line zero), or read from the LDS (CH 0)
    double cf[CH + 1], ch[CH + 1];
#pragma unroll
    for (int t = 0; t < CH; t++) {
        const int j = p + P * t, d = i - j;
        const bool valid = on && j < n;
        cf[t] = valid ? full[d < 0 ? d + n : d] : 0.0;
        ch[t] = CONTINUOUS && valid ? half[d < 0 ? d + n : d] : 0.0;
    }
    // sum over j of c[(i - j) mod n] v[j], in every lane of the group
    auto conv = [&](const double (&reg)[CH + 1], const double* c, const double* v) {
        double s = 0.0;
        if constexpr (CH > 0) {
#pragma unroll
            for (int t = 0; t < CH; t++) s += reg[t] * v[min(p + P * t, n - 1)];
        } else if (on) {
            int d = i - p;
            if (d < 0) d += n;
            for (int j = p; j < n; j += P) {
                s += c[d] * v[j];
                d -= P;
                if (d < 0) d += n;
            }
        }
#pragma unroll
        for (int m = 1; m < P; m <<= 1) s += __shfl_xor(s, m, 64);
        return s;
    };
    for (int s = 0; s < it.steps; s++) {
        double* a = xa + (s & 1) * n;
        double* b = xb + (s & 1) * n;
        double* c = xc + (s & 1) * n;
        if (on && p == 0) {
            a[i] = CONTINUOUS ? e2 * x : x;
            if (CONTINUOUS) b[i] = e4 * x;
        }
        __syncthreads();
        if constexpr (CONTINUOUS) {
            const double q1 = e2 * conv(cf, full, a);
            const double t = e2 * conv(ch, half, b);
            if (on && p == 0) c[i] = t;
            __syncthreads();
            x = (4.0 * (e4 * conv(ch, half, c)) - q1) / 3.0 * mask;
        } else {
            x = e2 * conv(cf, full, a) * mask;
        }
        x = (double)(T)x;   // the stored slice is what the next step starts from
        q += batch.stride;
        if (on && p == 0) q[i] = (T)x;
    }
}

}  // namespace fts
