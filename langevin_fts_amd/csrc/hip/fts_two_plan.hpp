// Plans and launch items of the two-stage FFT kernels (fts_fft_two.hpp): which grids they take,
// the LDS geometry of a plane and of a pencil tile.
#pragma once

#include <algorithm>
#include <type_traits>

#include "fts_fft.hpp"

namespace fts {

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
// larger radix is r2, the run of consecutive z values that a wavefront loads and stores; FP32
// takes 4 x 16 for 64, runs of 64 bytes: evaluations with 8 x 8 took 1.05 to 1.09 of the time at
// 40 x 48 x 64 and 72 x 60 x 64, 1.15 to 1.25 at 60 x 64, and 0.97 to 1.00 at 64^3.
enum TwoAxisKind { TWO_X, TWO_Y, TWO_Z };
constexpr bool two_axis(int L, TwoAxisKind kind, bool fp32, TwoAxis& a) {
    a = TwoAxis{L, 0, 0};
    for (int m = 1; m <= TWO_MAXR && !a.r1; m++)
        for (int s = 1; s <= m && !a.r1; s++) {
            if (m * s != L || !two_radix(m, fp32) || !two_radix(s, fp32)) continue;
            const bool first_large = kind == TWO_Y && (L % 2 == 1 || s % 2 == 1);
            a.r1 = first_large ? m : s;
            a.r2 = first_large ? s : m;
        }
    if (kind == TWO_Z && fp32 && L == 64) a = TwoAxis{L, 4, 16};
    return a.r1 != 0;
}

struct TwoGeom {
    int nx, nzc, sp;      // x-slabs, half-spectrum columns and their row pitch
    TwoAxis x, y, z;
    int lines;            // packed z lines: ceil(y.r1 / 2) y.r2
    int pad;              // one pad slot after every z.r1 positions of a line (z.r1 even), else 0
    int pitch;            // slots of a line
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
constexpr int two_conflicts(const TwoGeom& g, int pitch, int row) {
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

// Row pitch (complex elements) of the half spectra that the passes exchange through HBM: nzc rounded up to a
// whole number of 128-byte lines (8 columns in FP64, 16 in FP32), so that every row, and with it every
// pencil tile of that many columns, starts on a line. A tile that straddles two lines, or shares one with a
// neighbouring tile on another XCD (its own L2), fetches lines twice. The pad columns are never read
// or written.
constexpr int two_pitch(int nzc, int elem_bytes) {
    const int line = 128 / elem_bytes;
    return (nzc + line - 1) / line * line;
}
// The geometry of an nx x ny x nz grid, or false when a length has no plan or a plane does not
// fit the LDS
constexpr size_t two_slab_lds(const TwoGeom& g, int elem_bytes) {
    return (size_t)(g.lines * g.pitch + g.y.L + g.z.L) * elem_bytes;
}
constexpr bool two_geometry(const int* n, int elem_bytes, size_t lds_limit, TwoGeom& g) {
    g = TwoGeom{};
    const bool fp32 = elem_bytes == 8;
    if (!two_axis(n[0], TWO_X, fp32, g.x) || !two_axis(n[1], TWO_Y, fp32, g.y) || !two_axis(n[2], TWO_Z, fp32, g.z))
        return false;
    g.nx = n[0];
    g.nzc = n[2] / 2 + 1;
    g.sp = two_pitch(g.nzc, elem_bytes);
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
    if (two_slab_lds(g, elem_bytes) > lds_limit) g.pitch = least;
    if (two_slab_lds(g, elem_bytes) > lds_limit) return false;
    g.m_nzc = two_recip(g.nzc);
    g.m_zr1 = two_recip(g.z.r1);
    g.m_zr2 = two_recip(g.z.r2);
    g.m_yr2 = two_recip(g.y.r2);
    g.inv_m = 1.0 / ((double)n[0] * n[1] * n[2]);
    return true;
}
constexpr int two_pencil_columns(int elem_bytes) { return 128 / elem_bytes; }
// slots of one stage-B group of a tile of C columns: r2 rows, and the pad that puts the next
// group's first row beside this one's on the banks of a 256-byte bank row
__host__ __device__ constexpr int two_pencil_group(int r2, int C, int elem_bytes) {
    const int row = 256 / elem_bytes;
    return r2 * C + (C - r2 * C % row + row) % row;
}
constexpr size_t two_pencil_lds(const TwoGeom& g, int C, int elem_bytes) {
    return (size_t)(g.x.r1 * two_pencil_group(g.x.r2, C, elem_bytes) + g.x.L) * elem_bytes;
}
// threads of a slab workgroup: one butterfly of the busiest stage each, at most TWO_BD
constexpr int TWO_BD = 512;
constexpr int two_slab_threads(const TwoGeom& g) {
    const int y = g.nzc * std::max(g.y.r1, g.y.r2), z = g.lines * std::max(g.z.r1, g.z.r2);
    return std::min(TWO_BD, (std::max(y, z) + 63) / 64 * 64);
}

// The geometry as the kernels see it, radices under names of their own: values of the grid
// (TwoView), or constants of an N^3 grid (TwoCube), whose index arithmetic and radix dispatch
// then fold away.
struct TwoView : TwoGeom {
    int xr1, xr2, yr1, yr2, zr1, zr2;
    __host__ __device__ explicit TwoView(const TwoGeom& g)
        : TwoGeom(g), xr1(g.x.r1), xr2(g.x.r2), yr1(g.y.r1), yr2(g.y.r2), zr1(g.z.r1), zr2(g.z.r2) {}
};
template <int N, int ELEM_BYTES>
struct TwoCube {
    static constexpr TwoGeom make() {
        const int n[3] = {N, N, N};
        TwoGeom g{};
        two_geometry(n, ELEM_BYTES, 160 * 1024, g);
        return g;
    }
    static constexpr TwoGeom G = make();
    static_assert(G.pitch > 0, "the grid has a two-stage plan");
    template <int V>
    using Const = std::integral_constant<int, V>;
    static constexpr TwoAxis x = G.x, y = G.y, z = G.z;
    static constexpr Const<G.x.r1> xr1{};
    static constexpr Const<G.x.r2> xr2{};
    static constexpr Const<G.y.r1> yr1{};
    static constexpr Const<G.y.r2> yr2{};
    static constexpr Const<G.z.r1> zr1{};
    static constexpr Const<G.z.r2> zr2{};
    static constexpr int nx = G.nx, nzc = G.nzc, sp = G.sp, lines = G.lines, pad = G.pad, pitch = G.pitch;
    static constexpr unsigned m_nzc = G.m_nzc, m_zr1 = G.m_zr1, m_zr2 = G.m_zr2, m_yr2 = G.m_yr2;
    static constexpr double inv_m = G.inv_m;
};

// Launch shapes of the N^3 kernels: workgroup sizes of the slab pass (the autotuner's
// candidates, all with the same per-line transforms) and kz columns of a pencil wavefront.
constexpr bool slab_bd_ok(int N, int bd) {
    return (N == 32 && (bd == 128 || bd == 256)) || (N == 48 && (bd == 256 || bd == 384)) ||
           (N == 64 && (bd == 256 || bd == 320 || bd == 512)) || (N == 96 && (bd == 512 || bd == 1024)) ||
           (N == 128 && (bd == 512 || bd == 1024));
}
constexpr int SLAB_BD_ALL[] = {128, 256, 320, 384, 512, 1024};
constexpr int PENCIL_NL_ALL[] = {4, 8, 16};
// Default slab workgroups. 48^3: 256 threads against 384 measured 20.8 against 24.9 us for a
// half step of 32 propagators (every stage has at most 200 butterflies).
constexpr int slab_default_bd(int N) { return N <= 48 ? 256 : (N <= 64 ? 320 : 1024); }
// A mode's own default, 0: slab_default_bd. With 1024 threads the FP64 Richardson step of 96^3
// and 128^3 and the 128^3 forward pass of two spectra spill: 512 threads measured 30.4 against
// 50.4 us, 76 against 132 us and 34.4 against 40.0 us for two propagators.
constexpr int slab_default_bd_mode(int N, int elem_bytes, int mode) {
    const bool spills = elem_bytes == 16 && ((N >= 96 && mode == SLAB_INV2) || (N == 128 && mode == SLAB_FWD));
    return spills ? 512 : 0;
}
// With more than one 64^3 workgroup per CU, whole wavefronts on every SIMD count instead of one
// workgroup's latency: 16 propagators took 27.2 us per half step with 512 threads (320: 32.8,
// 256: 28.8) and, its registers leaving room for three workgroups of 256 threads but one of 512,
// 53.5 us per FP64 Richardson step with 256 (320: 63.9, 512: 64.2). It takes the place of a tuned shape there, unless
// the caller has set one. Other sizes keep one shape: 32^3 and 48^3 default to 256 threads already, and larger
// launches of 96^3 and 128^3, of 8 or 16 wavefronts a workgroup, were not tried in other shapes.
constexpr int slab_batch_bd(int N, int mode) { return N != 64 ? 0 : (mode == SLAB_INV2 ? 256 : 512); }
constexpr int SLAB_BATCH_BLOCKS = 256;   // workgroups of a launch above which slab_batch_bd applies: the CUs
// kz columns: 4 in FP64 from 96^3 (the XCD tile order keeps a line's tiles on one L2)
constexpr int pencil_default_nl(int N, int elem_bytes) { return elem_bytes == 16 && N >= 96 ? 4 : 8; }

// Consecutive steps of one propagator on a grid of one x-slab, in one launch
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

// Points of a line that takes its convolutions directly (n products per point), and the lanes that
// share a point: at most 1024 threads
constexpr int LINE_POINTS = 256;
constexpr int line_lanes(int n) { return n <= 128 ? 8 : 4; }
constexpr int LINE_PARTS = 8;   // partial sums per bond of its coefficients
constexpr size_t line_lds(int n) { return sizeof(double) * (8 * (size_t)n + 4 * LINE_PARTS); }

}  // namespace fts
