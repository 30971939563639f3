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

#include "fts_fft.hpp"

namespace fts {

// the workgroup's dynamic LDS
#ifndef FTS_DYNAMIC_LDS
#define FTS_DYNAMIC_LDS(name) extern __shared__ __align__(16) unsigned char name[]
#endif

// ------------------------------------------------------------------ register transforms
// RDft<R, DIR>::run: R-point transform in registers, natural order in and out, DIR -1 forward.
// 2, 3, 4, 5 and 8 are fts_fft.hpp's butterflies; R = A B with coprime A, B by the prime-factor
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
struct RDft<8, DIR, T, T2> : RDftBase<8, DIR, T, T2> {};

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
                    else t[b][a] = cmul(t[b][a], T2{(T)root_cos(R, a * b), (T)(DIR * root_sin(R, a * b))});
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

// ------------------------------------------------------------------ plans
constexpr int TWO_MAXR = 16;

// radices the kernels of a precision are built with (FP32 plans take prime factors 2, 3 and 5 only)
constexpr bool two_radix(int r, bool fp32) {
    return r >= 1 && r <= TWO_MAXR && !(fp32 && (r % 7 == 0 || r % 11 == 0 || r % 13 == 0));
}

struct TwoAxis {
    int L, r1, r2;
};

// L = r1 r2 with the smallest larger radix. y axis: r1 even when L is (rows pair up inside a
// butterfly), and the larger one when L is odd (one row of r1 has no partner). Other axes: the
// larger radix is r2, the run of consecutive z values that a wavefront stores.
inline bool two_axis(int L, bool y_axis, bool fp32, TwoAxis& a) {
    a = TwoAxis{L, 0, 0};
    for (int m = 1; m <= TWO_MAXR && !a.r1; m++)
        for (int s = 1; s <= m && !a.r1; s++) {
            if (m * s != L || !two_radix(m, fp32) || !two_radix(s, fp32)) continue;
            const bool first_large = y_axis && (L % 2 == 1 || s % 2 == 1);
            a.r1 = first_large ? m : s;
            a.r2 = first_large ? s : m;
        }
    return a.r1 != 0;
}

struct TwoGeom {
    int nx, nzc, sp;      // x-slabs, half-spectrum columns and their row pitch
    TwoAxis x, y, z;
    int lines;            // packed z lines: ceil(y.r1 / 2) y.r2
    int pad;              // one pad slot after every z.r1 positions of a line (z.r1 even), else 0
    int pitch;            // slots of a line
    int xpad;             // pencil pass: extra slots between the stage-B groups
    unsigned m_nzc, m_zr1, m_zr2, m_yr2;   // reciprocals for two_div
    double inv_m;
};

// t / d for t d < 2^32 by one multiplication with m = two_recip(d)
constexpr unsigned two_recip(int d) { return d == 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d); }
__device__ __forceinline__ int two_div(int t, unsigned m) {
    return m == 0 ? t : (int)(((unsigned long long)(unsigned)t * m) >> 32);
}

// Wavefront accesses of the two z stages that share an LDS bank, counted over groups of `row`
// consecutive lanes (row: elements of one 256-byte bank row)
inline int two_conflicts(const TwoGeom& g, int pitch, int row) {
    int total = 0;
    for (int stage = 0; stage < 2; stage++) {
        const int r = stage == 0 ? g.z.r1 : g.z.r2, step = stage == 0 ? 1 : g.z.r1 + g.pad;
        for (int t0 = 0; t0 < 64; t0 += row) {
            int hit[64] = {}, worst = 0;
            for (int t = t0; t < t0 + row; t++) {
                const int b = ((t / r) * pitch + (t % r) * step) % row;
                worst = std::max(worst, ++hit[b]);
            }
            total += worst;
        }
    }
    return total;
}

// The geometry of an nx x ny x nz grid, or false when a length has no plan or a plane does not
// fit the LDS
inline bool two_geometry(const int* n, int elem_bytes, size_t lds_limit, TwoGeom& g) {
    g = TwoGeom{};
    const bool fp32 = elem_bytes == 8;
    if (!two_axis(n[0], false, fp32, g.x) || !two_axis(n[1], true, fp32, g.y) || !two_axis(n[2], false, fp32, g.z))
        return false;
    g.nx = n[0];
    g.nzc = n[2] / 2 + 1;
    const int line = 128 / elem_bytes;
    g.sp = (g.nzc + line - 1) / line * line;
    g.lines = (g.y.r1 + 1) / 2 * g.y.r2;
    g.pad = g.z.r1 % 2 == 0 ? 1 : 0;
    const int row = 256 / elem_bytes, least = n[2] + g.pad * g.z.r2 + 2;
    int best = 1 << 30;
    for (int p = least; p < least + row; p++) {
        const int c = two_conflicts(g, p, row);
        if (c < best) {
            best = c;
            g.pitch = p;
        }
    }
    auto bytes = [&] { return (size_t)(g.lines * g.pitch + n[1] + n[2]) * elem_bytes; };
    if (bytes() > lds_limit) g.pitch = least;
    if (bytes() > lds_limit) return false;
    // pencil pass: groups of r2 rows of a tile's `line` columns, started line columns apart (mod the bank row)
    g.xpad = (line - g.x.r2 * line % row + row) % row;
    g.m_nzc = two_recip(g.nzc);
    g.m_zr1 = two_recip(g.z.r1);
    g.m_zr2 = two_recip(g.z.r2);
    g.m_yr2 = two_recip(g.y.r2);
    g.inv_m = 1.0 / ((double)n[0] * n[1] * n[2]);
    return true;
}
inline size_t two_slab_lds(const TwoGeom& g, int elem_bytes) {
    return (size_t)(g.lines * g.pitch + g.y.L + g.z.L) * elem_bytes;
}
inline int two_pencil_columns(int elem_bytes) { return 128 / elem_bytes; }
inline size_t two_pencil_lds(const TwoGeom& g, int elem_bytes) {
    const int C = two_pencil_columns(elem_bytes);
    return (size_t)(g.x.r1 * (g.x.r2 * C + g.xpad) + g.x.L) * elem_bytes;
}
// threads of a slab workgroup: one butterfly of the busiest stage each, at most TWO_BD
constexpr int TWO_BD = 512;
inline int two_slab_threads(const TwoGeom& g) {
    const int y = g.nzc * std::max(g.y.r1, g.y.r2), z = g.lines * std::max(g.z.r1, g.z.r2);
    return std::min(TWO_BD, (std::max(y, z) + 63) / 64 * 64);
}

// f with a compile-time radix equal to r
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

// ------------------------------------------------------------------ the plane of a slab
template <typename T>
struct TwoPlane {
    using T2 = typename vec2<T>::type;
    const TwoGeom& g;
    T2* S;            // packed lines
    const T2 *Wy, *Wz;
    int tid, bd;

    // the slots of half-spectrum column c in a packed line: e holds Z[c], o holds Z[nz - c]
    struct Col {
        int e, o;
        bool self;    // c = nz - c (mod nz): one value, o is a spare slot
    };
    __device__ __forceinline__ int zslot(int k) const { return g.pad ? k + two_div(k, g.m_zr1) : k; }
    __device__ __forceinline__ Col column(int c) const {
        const int nz = g.z.L, end = nz + g.pad * g.z.r2;
        if (c == 0) return Col{0, end, true};
        if (2 * c == nz) return Col{zslot(c), end + 1, true};
        return Col{zslot(c), zslot(nz - c), false};
    }

    // stage B of y for butterfly (column c, k1 = j), inverse: v holds rows j + r1 r of the column
    template <int R>
    __device__ __forceinline__ void y_scatter(T2 (&v)[R], const Col& q, int j) const {
        RDft<R, +1, T, T2>::run(v);
        T2* base = S + (j >> 1) * g.y.r2 * g.pitch + ((j & 1) ? q.o : q.e);
#pragma unroll
        for (int r = 0; r < R; r++) base[r * g.pitch] = v[r];
    }
    // stage A of y, inverse, with the merge of the row pairs
    __device__ __forceinline__ void y_merge() const {
        const int total = g.nzc * g.y.r2;
        for (int t = tid; t < total; t += bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const Col q = column(c);
            two_radix_call<T>(g.y.r1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = S[((r >> 1) * g.y.r2 + j) * g.pitch + ((r & 1) ? q.o : q.e)];
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = cmul(v[r], root<+1>(Wy, r * j));
                RDft<R, +1, T, T2>::run(v);
#pragma unroll
                for (int a = 0; a < (R + 1) / 2; a++) {
                    T2 A = v[2 * a], B = 2 * a + 1 < R ? v[(2 * a + 1) % R] : T2{(T)0, (T)0};
                    if (q.self) A.y = B.y = (T)0;
                    T2* base = S + (a * g.y.r2 + j) * g.pitch;
                    base[q.e] = T2{A.x - B.y, A.y + B.x};
                    if (!q.self) base[q.o] = T2{A.x + B.y, B.x - A.y};
                }
            });
        }
    }
    // stage B of z: inverse (k natural -> (k1, n2)) or forward ((k1, n2) -> k natural)
    template <int DIR>
    __device__ __forceinline__ void z_outer() const {
        const int total = g.lines * g.z.r1, step = g.z.r1 + g.pad;
        for (int t = tid; t < total; t += bd) {
            const int line = two_div(t, g.m_zr1), j = t - line * g.z.r1;
            T2* base = S + line * g.pitch + j;
            two_radix_call<T>(g.z.r2, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = base[r * step];
                RDft<R, DIR, T, T2>::run(v);
#pragma unroll
                for (int r = 0; r < R; r++) base[r * step] = v[r];
            });
        }
    }
    // Stage A of z both ways around the real values: op(i0, two, v, vb) gets the index of a value
    // of the pair's first row, whether the second row exists (at i0 + second), and the two
    // values; it returns through them what the forward transform takes.
    template <typename Op>
    __device__ __forceinline__ void z_inner(bool inverse, bool forward, Op&& op) const {
        const int total = g.lines * g.z.r2;
        const int nz = g.z.L;
        for (int t = tid; t < total; t += bd) {
            const int line = two_div(t, g.m_zr2), j = t - line * g.z.r2;
            const int a = two_div(line, g.m_yr2);
            const int row = line + a * g.y.r2;    // (2 a) r2 + n2 with line = a r2 + n2
            const bool two = 2 * a + 1 < g.y.r1;
            const int i0 = row * nz + j;
            T2* base = S + line * g.pitch + j * (g.z.r1 + g.pad);
            two_radix_call<T>(g.z.r1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                if (inverse) {
#pragma unroll
                    for (int r = 0; r < R; r++) v[r] = base[r];
#pragma unroll
                    for (int r = 1; r < R; r++) v[r] = cmul(v[r], root<+1>(Wz, r * j));
                    RDft<R, +1, T, T2>::run(v);
                }
#pragma unroll
                for (int r = 0; r < R; r++) op(i0 + r * g.z.r2, two, v[r]);
                if (forward) {
                    RDft<R, -1, T, T2>::run(v);
#pragma unroll
                    for (int r = 1; r < R; r++) v[r] = cmul(v[r], root<-1>(Wz, r * j));
#pragma unroll
                    for (int r = 0; r < R; r++) base[r] = v[r];
                }
            });
        }
    }
    // stage A of y, forward, with the split of the packed lines (twice the rows' spectra: the
    // caller halves the real values)
    __device__ __forceinline__ void y_split() const {
        const int total = g.nzc * g.y.r2;
        for (int t = tid; t < total; t += bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const Col q = column(c);
            two_radix_call<T>(g.y.r1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
#pragma unroll
                for (int a = 0; a < (R + 1) / 2; a++) {
                    const T2* base = S + (a * g.y.r2 + j) * g.pitch;
                    const T2 A = base[q.e];
                    const T2 B = q.self ? A : base[q.o];
                    v[2 * a] = T2{A.x + B.x, A.y - B.y};
                    if (2 * a + 1 < R) v[(2 * a + 1) % R] = T2{A.y + B.y, B.x - A.x};
                }
                RDft<R, -1, T, T2>::run(v);
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = cmul(v[r], root<-1>(Wy, r * j));
#pragma unroll
                for (int r = 0; r < R; r++) S[((r >> 1) * g.y.r2 + j) * g.pitch + ((r & 1) ? q.o : q.e)] = v[r];
            });
        }
    }
    // stage B of y, forward: v[r] becomes row j + r1 r of the column
    template <int R>
    __device__ __forceinline__ void y_gather(T2 (&v)[R], const Col& q, int j) const {
        const T2* base = S + (j >> 1) * g.y.r2 * g.pitch + ((j & 1) ? q.o : q.e);
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = base[r * g.pitch];
        RDft<R, -1, T, T2>::run(v);
    }
};

// ------------------------------------------------------------------ slab pass
// The pass of fts_fft.hpp's slab_kernel (same items, modes and results) for grids with a
// TwoGeom; spectra have rows of g.sp values. INV2 items must have qout: the first half step
// waits there.
template <typename T>
__global__ void __launch_bounds__(TWO_BD) slab_two_kernel(TwoGeom g, int mode, SlabBatch<T> batch,
                                                          const typename vec2<T>::type* twy,
                                                          const typename vec2<T>::type* twz) {
    using T2 = typename vec2<T>::type;
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wy = S + g.lines * g.pitch;
    T2* Wz = Wy + g.y.L;
    for (int m = threadIdx.x; m < g.y.L; m += blockDim.x) Wy[m] = twy[m];
    for (int m = threadIdx.x; m < g.z.L; m += blockDim.x) Wz[m] = twz[m];
    const SlabItem<T>& it = batch.it[blockIdx.y];
    const int ny = g.y.L, nz = g.z.L;
    const size_t roff = (size_t)blockIdx.x * ny * nz;
    const size_t coff = (size_t)blockIdx.x * ny * g.sp;
    const T inv_m = (T)g.inv_m;
    const bool has_w = it.w != nullptr;
    const T* w = has_w ? it.w + roff : nullptr;
    const T* mask = it.mask ? it.mask + roff : nullptr;
    T* qout = it.qout ? it.qout + roff : nullptr;
    const int second = g.y.r2 * nz;   // from a value of a pair's first row to the second's
    const TwoPlane<T> pl{g, S, Wy, Wz, (int)threadIdx.x, (int)blockDim.x};

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
            const int total = g.nzc * g.y.r1;
            for (int t = pl.tid; t < total; t += pl.bd) {
                const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
                const typename TwoPlane<T>::Col q = pl.column(c);
                two_radix_call<T>(g.y.r2, [&](auto RC) {
                    constexpr int R = decltype(RC)::value;
                    T2 v[R];
                    const T2* src = spec + (size_t)j * g.sp + c;
#pragma unroll
                    for (int r = 0; r < R; r++) v[r] = src[r * g.y.r1 * g.sp];
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
                v = v * factor<T>(wv, has_w, post) * inv_m;
                if (comb) v = ((T)4.0 * v - qout[i]) / (T)3.0;
                if (!park && mask) v *= mask[i];
                if (qout) qout[i] = v;
            } else {
                v = load[i];
            }
            return forward ? v * factor<T>(wv, has_w, pre) * (T)0.5 : v;
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
        const int total = g.nzc * g.y.r1;
        for (int t = pl.tid; t < total; t += pl.bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const typename TwoPlane<T>::Col q = pl.column(c);
            two_radix_call<T>(g.y.r2, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                pl.template y_gather<R>(v, q, j);
                T2* dst = spec + (size_t)j * g.sp + c;
#pragma unroll
                for (int r = 0; r < R; r++) dst[r * g.y.r1 * g.sp] = v[r];
            });
        }
    }
}

// ------------------------------------------------------------------ pencil (x) pass
// One wavefront per y row and tile of one 128-byte line of kz columns.
__device__ __forceinline__ void two_wave_sync() {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#else
    __syncthreads();
#endif
}

template <typename T>
__global__ void __launch_bounds__(64) pencil_two_kernel(TwoGeom g, XBatch<T> batch,
                                                        const typename vec2<T>::type* twx, const T* bx, const T* by,
                                                        const T* bz) {
    using T2 = typename vec2<T>::type;
    constexpr int C = 128 / (int)sizeof(T2);
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    const int group = g.x.r2 * C + g.xpad;   // slots of one k1
    T2* Wx = S + g.x.r1 * group;
    const int lane = threadIdx.x;
    for (int m = lane; m < g.x.L; m += 64) Wx[m] = twx[m];
    const XItem<T>& it = batch.it[blockIdx.y];
    const int tiles = (g.nzc + C - 1) / C;
    const int jy = blockIdx.x / tiles;
    const int k0 = (blockIdx.x - jy * tiles) * C;
    const int cw = min(C, g.nzc - k0);
    const size_t row = (size_t)g.y.L * g.sp;
    T2* c = it.c + (size_t)jy * g.sp + k0;
    const int table = it.table;
    const int r1 = g.x.r1, r2 = g.x.r2;
    if (table != -2) {
        two_wave_sync();   // twiddles
        for (int t = lane; t < C * r2; t += 64) {
            const int j = t / C, l = t % C;
            if (l >= cw) continue;
            two_radix_call<T>(r1, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = c[(size_t)(r * r2 + j) * row + l];
                RDft<R, -1, T, T2>::run(v);
#pragma unroll
                for (int r = 1; r < R; r++) v[r] = cmul(v[r], root<-1>(Wx, r * j));
#pragma unroll
                for (int r = 0; r < R; r++) S[r * group + j * C + l] = v[r];
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
                    for (int r = 0; r < R; r++) c[(size_t)(j + r * r1) * row + l] = v[r];
                    return;
                }
                const T* tx = bx + (size_t)table * g.x.L + j;
                const T bl = by[(size_t)table * g.y.L + jy] * bz[(size_t)table * g.nzc + k0 + l];
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const T b = tx[r * r1] * bl;
                    v[r] = T2{v[r].x * b, v[r].y * b};
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) v[r] = c[(size_t)(j + r * r1) * row + l];
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
            for (int r = 0; r < R; r++) v[r] = S[r * group + j * C + l];
#pragma unroll
            for (int r = 1; r < R; r++) v[r] = cmul(v[r], root<+1>(Wx, r * j));
            RDft<R, +1, T, T2>::run(v);
#pragma unroll
            for (int r = 0; r < R; r++) c[(size_t)(r * r2 + j) * row + l] = v[r];
        });
    }
}

// ------------------------------------------------------------------ whole steps of flat grids
// A grid of one x-slab (one and two dimensions) holds its whole transform in one workgroup's
// LDS: the bond factors apply between the forward and the inverse y stage B in registers, and a
// workgroup runs all consecutive steps of a propagator in one launch.
template <typename T>
struct FlatItem {
    T* q;            // slice n0; slice n0 + s at + s stride
    T* half;         // continuous: one field of scratch (the full step's result)
    const T* w;      // as SlabItem::w
    const T* mask;
    T full_w, half_w;        // factor coefficients: continuous exp(-w ds/2), exp(-w ds/4); discrete exp(-w ds), unused
    int steps;
    int full_table, half_table;
};

constexpr int FLAT_BATCH = 32;
template <typename T>
struct FlatBatch {
    int n;
    size_t stride;
    FlatItem<T> it[FLAT_BATCH];
};

template <typename T, bool CONTINUOUS>
__global__ void __launch_bounds__(TWO_BD) flat_steps_kernel(TwoGeom g, FlatBatch<T> batch,
                                                            const typename vec2<T>::type* twy,
                                                            const typename vec2<T>::type* twz, const T* by,
                                                            const T* bz) {
    using T2 = typename vec2<T>::type;
    FTS_DYNAMIC_LDS(smem_raw);
    T2* S = reinterpret_cast<T2*>(smem_raw);
    T2* Wy = S + g.lines * g.pitch;
    T2* Wz = Wy + g.y.L;
    for (int m = threadIdx.x; m < g.y.L; m += blockDim.x) Wy[m] = twy[m];
    for (int m = threadIdx.x; m < g.z.L; m += blockDim.x) Wz[m] = twz[m];
    const FlatItem<T>& it = batch.it[blockIdx.x];
    const int second = g.y.r2 * g.z.L;
    const T inv_m = (T)g.inv_m;
    const TwoPlane<T> pl{g, S, Wy, Wz, (int)threadIdx.x, (int)blockDim.x};
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
                    v = v * factor<T>(wv, true, it.full_w) * inv_m;
                    if (mask) v *= mask[i];
                    qdone[i] = v;
                } else {
                    v = qn[i];
                }
                return v * (T)0.5;
            } else {
                if (inverse) {
                    v = v * factor<T>(wv, true, prev == 2 ? it.half_w : it.full_w) * inv_m;
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
                if (next == 0) v *= factor<T>(wv, true, it.full_w);
                else if (next == 1) v *= factor<T>(wv, true, it.half_w);
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
        const int total = g.nzc * g.y.r1;
        for (int t = pl.tid; t < total; t += pl.bd) {
            const int j = two_div(t, g.m_nzc), c = t - j * g.nzc;
            const typename TwoPlane<T>::Col q = pl.column(c);
            two_radix_call<T>(g.y.r2, [&](auto RC) {
                constexpr int R = decltype(RC)::value;
                T2 v[R];
                pl.template y_gather<R>(v, q, j);
                const T b = tz[c];
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const T f = ty[j + r * g.y.r1] * b;
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

}  // namespace fts
