// Row sweeps: the four half steps of the 3D solver (forward H and E, adjoint
// E and H), V consecutive z cells a thread.
//
// The half steps stream the fields from HBM, so their floor is their bytes:
// 40 B a cell, plus 8 B an active CPML auxiliary. The adjoint therefore forms
// the weights of its transposed stencils where it reads them (one product, or
// in the CPML the auxiliary's term) instead of storing six arrays of them
// between two sweeps. A thread's taps along x and y are one V-wide load each. A
// workgroup covers whole rows, the z-CPML included, so every cache line is
// fetched and written once; the ends of its rows, with the z-CPML work, are put
// into as few of its wavefronts as hold them. Rows away from the x and y faces
// (the whole workgroup) run code without any test of those axes (XY).
//
// Four cells a thread in plain rows: a 64-lane load then moves 1 KiB, where a
// load of one float a lane occupies the address unit nearly as long; wider or
// fewer cells a thread were slower (two cells: 2 % on 289 x 289 x 225 fields,
// 17 % on 161 x 161 x 129 x 4 shots). Measured on an MI355X, order 4, CPML 16,
// 289 x 289 x 225 fields, us per launch, before (one thread per cell, stored
// weights) and now: forward H 283 and 229, forward E 286 and 248, adjoint 1038
// (three launches) and 615 (two). With the ends of the rows in every wavefront
// these were 243, 256 and 607; 129 x 129 x 129 x 2 shots, order 4, 63, 73 and 189
// against 58, 68 and 179 now; order 2 on 165 x 141 x 189, 45, 51 and 101 against
// 42, 45 and 98. What bounds them now is the chain of a wavefront (loads, row
// exchange, z-CPML loads, stores) at 4 wavefronts a SIMD and, in the adjoint,
// the vector instructions (42 % of the cycles), not the bytes.
//
// Four wavefronts need at most 128 registers a lane, so what only the end of a
// sweep uses is loaded there: with the old fields, cb and the adjoint's outputs
// held from the start (136 to 140 registers, 3 wavefronts) forward E took 293 and
// the adjoint 677. At 96 registers (5 wavefronts) the plain groups spill: forward
// 396 and 570, adjoint 1052.
#include <algorithm>

#include "dgx_device.h"
#include "dgx_internal.h"
#include "dgx_rows.h"

namespace dgx {

namespace {

constexpr int kRowCells = 4;         // V: cells of a thread in plain rows
constexpr int kRowThreads = 256;     // threads of a workgroup, unless a row needs more
constexpr int kRowMaxThreads = 512;  // the longest row in groups of V / 2

template <int V>
struct Vec {
    typedef float type __attribute__((ext_vector_type(V)));
    typedef float utype __attribute__((ext_vector_type(V), aligned(4)));
};
template <int V>
using fv = typename Vec<V>::type;

// Elements [idx, idx + V) of an array below 4 GiB: a wave-uniform base and a
// 32-bit offset.
template <int V>
__device__ __forceinline__ fv<V> ldv(const float* base, unsigned idx)
{
    return *(const typename Vec<V>::utype*)((const char*)base + (size_t)(idx * 4u));
}
__device__ __forceinline__ float ld1(const float* base, unsigned idx)
{
    return *(const float*)((const char*)base + (size_t)(idx * 4u));
}
// Own cells: elements before dup belong to another thread.
template <int V>
__device__ __forceinline__ void stv(float* base, unsigned idx, fv<V> v, int dup)
{
    float* p = (float*)((char*)base + (size_t)(idx * 4u));
    if (dup == 0) {
        *(typename Vec<V>::utype*)p = v;
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (e >= dup) p[e] = v[e];
    }
}
// The first n elements of a group at p (0 beyond).
template <int V>
__device__ __forceinline__ fv<V> ldn(const float* p, int n)
{
    fv<V> o = 0.0f;
    if (n >= V) {
        o = *(const typename Vec<V>::utype*)p;
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (e < n) o[e] = p[e];
    }
    return o;
}
template <int V>
__device__ __forceinline__ void stn(float* p, fv<V> v, int dup, int n)
{
    if (dup == 0 && n >= V) {
        *(typename Vec<V>::utype*)p = v;
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (e >= dup && e < n) p[e] = v[e];
    }
}

template <int V>
__device__ __forceinline__ fv<V> pick(bool c, const fv<V>& a, const fv<V>& b)
{
    fv<V> o;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = c ? a[e] : b[e];
    return o;
}

// Curl coefficients on axis a (axis_coeff of every element).
template <int V>
__device__ __forceinline__ fv<V> axis_coeffs(const Grid& g, fv<V> c1, int a)
{
    if (a == 0 || g.d[a] == g.d[0]) return c1;
    fv<V> out;
#pragma unroll
    for (int e = 0; e < V; ++e) out[e] = c1[e] * g.d[0] / g.d[a];
    return out;
}

// The part of a sweep's geometry a thread works on.
struct Group {
    int i, j, k;   // k: first cell
    int dup;       // cells that belong to another thread
    int s;         // shot
    unsigned m;    // first cell in the model
    bool zplain;   // every cell in the plain z-range
};

// ---------------------------------------------------------------------------
// Differences
// ---------------------------------------------------------------------------
// Along x or y (stride st) of V cells: full-width (PLAIN), or fitted to
// coordinate c of n cells, every tap of a row that is not live reading the cell.
template <int ORDER, int V, bool FWD, bool PLAIN>
__device__ __forceinline__ fv<V> diff_row(const float* f, unsigned m, int st, int c, int n, bool live)
{
    constexpr int R = Radius<ORDER>::value;
    const int rr = PLAIN ? R : (FWD ? fit_fwd_sel(c, n, R) : fit_bwd_sel(c, n, R));
    fv<V> hi[R], lo[R];
#pragma unroll
    for (int r = 1; r <= R; ++r) {
        const int h = FWD ? r : r - 1, l = FWD ? 1 - r : -r;
        if constexpr (PLAIN) {
            hi[r - 1] = ldv<V>(f + (ptrdiff_t)h * st, m);
            lo[r - 1] = ldv<V>(f + (ptrdiff_t)l * st, m);
        } else {
            const bool use = live && (ORDER <= 2 || r <= rr);
            hi[r - 1] = ldv<V>(f, m + (unsigned)((use ? h : 0) * st));
            lo[r - 1] = ldv<V>(f, m + (unsigned)((use ? l : 0) * st));
        }
    }
    if constexpr (ORDER <= 2) {
        return hi[0] - lo[0];
    } else {
        fv<V> out = 0.0f;
#pragma unroll
        for (int q = PLAIN ? R : 1; q <= R; ++q) {
            fv<V> acc = 0.0f;
#pragma unroll
            for (int r = 1; r <= q; ++r) acc += stencil_c(q, r) * (hi[r - 1] - lo[r - 1]);
            if constexpr (PLAIN) out = acc;
            else out = pick<V>(rr == q, acc, out);
        }
        return out;
    }
}

// Along z: c holds the cells of the group, row (in LDS) all cells of their row
// (a tap outside the row reads its end and is not used).
template <int ORDER, int V, bool FWD>
__device__ __forceinline__ fv<V> diff_z(const fv<V>& c, const float* row, const Group& q, int n)
{
    constexpr int R = Radius<ORDER>::value;
    constexpr int L = FWD ? R - 1 : R, U = FWD ? R : R - 1;
    float w[V + L + U];
#pragma unroll
    for (int e = 0; e < L; ++e) w[e] = row[max(q.k - L + e, 0)];
#pragma unroll
    for (int e = 0; e < V; ++e) w[L + e] = c[e];
#pragma unroll
    for (int e = 0; e < U; ++e) w[L + V + e] = row[min(q.k + V + e, n - 1)];
    fv<V> out;
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const int h = L + e + (FWD ? 0 : -1);  // window index of tap r: h + r and h + 1 - r
        if constexpr (ORDER <= 2) {
            out[e] = w[h + 1] - w[h];
        } else {
            float acc = 0.0f;
#pragma unroll
            for (int r = 1; r <= R; ++r) acc += stencil_c(R, r) * (w[h + r] - w[h + 1 - r]);
            out[e] = acc;
        }
    }
    if constexpr (ORDER > 2) {
        if (q.k < R || q.k + V - 1 > n - 1 - R) {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const int h = L + e + (FWD ? 0 : -1);
                const int rr = FWD ? fit_fwd_sel(q.k + e, n, R) : fit_bwd_sel(q.k + e, n, R);
#pragma unroll
                for (int t = 1; t < R; ++t) {
                    float acc = 0.0f;
#pragma unroll
                    for (int r = 1; r <= t; ++r) acc += stencil_c(t, r) * (w[h + r] - w[h + 1 - r]);
                    out[e] = rr == t ? acc : out[e];
                }
            }
        }
    }
    return out;
}

// ---------------------------------------------------------------------------
// CPML
// ---------------------------------------------------------------------------
// A choice of values. (With cond ? a : b of two array elements the compiler
// chooses an address and then loads: for a kernel argument that is a vector
// load and a wait.)
template <typename T>
__device__ __forceinline__ T choose(bool c, T a, T b)
{
    return c ? a : b;
}

// The face of axis a on the side of coordinate c (row_face_fits: the only one in
// the thread's reach): the cells [lo, hi] of its region and their profile index,
// hi - c on the low side, c - lo on the high.
struct Side {
    bool high;
    int p, lo, hi;
    __device__ __forceinline__ bool in(int c) const { return p > 0 && c >= lo && c <= hi; }
    __device__ __forceinline__ int at(int c) const { return high ? c - lo : hi - c; }
};

template <bool EL>
__device__ __forceinline__ Side side_of(const Grid& g, int a, int c)
{
    Side o;
    const int n = g.N[a];
    o.high = row_high_side(c, n);
    o.p = choose(o.high, g.pml[2 * a + 1], g.pml[2 * a]);
    o.lo = o.high ? n - 1 - o.p : (EL ? 1 : 0);
    o.hi = o.high ? n - 2 : (EL ? o.p : o.p - 1);
    return o;
}

// The row of auxiliary w of a face on axis x or y at profile index q: its
// elements along z, and their count (0: the grid row (i, j) has none).
template <bool EL>
__device__ __forceinline__ float* psi_row(const Grid& g, float* const (&psi)[6][2], int a, int w, const Side& sd,
                                          int q, int i, int j, int s, int& n)
{
    const int t = EL ? face_target(a, w) : face_source(a, w);  // one element less along this axis
    const int d0 = g.N[0] - (t == 0 ? 1 : 0), d1 = g.N[1] - (t == 1 ? 1 : 0), d2 = g.N[2] - (t == 2 ? 1 : 0);
    const int depth = EL ? sd.p + 1 : sd.p;
    n = (a == 0 ? j < d1 : i < d0) ? d2 : 0;
    const long long r = a == 0 ? ((long long)s * depth + q) * d1 + min(j, d1 - 1)
                               : ((long long)s * d0 + min(i, d0 - 1)) * depth + q;
    return choose(sd.high, psi[2 * a + 1][w], psi[2 * a][w]) + r * d2;
}

// The profiles by cell: RA - 1, RB, RE and RF of the cells of axis x, then of
// y and z (zero outside the faces), so that they load like the fields.
__device__ __forceinline__ const float* axis_table(const Grid& g, const float* tab, int a)
{
    return tab + 4 * (a == 0 ? 0 : (a == 1 ? g.N[0] : g.N[0] + g.N[1]));
}

// The face of axis a (0 or 1) that a row lies in, with its auxiliaries loaded.
template <int V>
struct RowFace {
    bool any;
    int n[2];         // cells of the group that have an element
    float* p[2];
    fv<V> phi[2];
    float ra1, rb, re, rf;
};

template <int V, bool EL>
__device__ __forceinline__ RowFace<V> row_face(const Grid& g, const Cpml& cp, const float* tab, int has_cpml, int a,
                                               const Group& q)
{
    RowFace<V> o;
    const int c = a == 0 ? q.i : q.j;
    const Side sd = side_of<EL>(g, a, c);
    o.any = has_cpml && sd.in(c);
    o.n[0] = o.n[1] = 0;
    o.p[0] = o.p[1] = nullptr;
    o.phi[0] = o.phi[1] = 0.0f;
    o.ra1 = o.rb = o.re = o.rf = 0.0f;
    if (o.any) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            int n;
            o.p[w] = psi_row<EL>(g, cp.psi, a, w, sd, sd.at(c), q.i, q.j, q.s, n) + q.k;
            o.n[w] = n - q.k;
            o.phi[w] = ldn<V>(o.p[w], o.n[w]);
        }
        const float* T = axis_table(g, tab, a) + c;
        const int n = g.N[a];
        o.ra1 = T[0];
        o.rb = T[n];
        o.re = T[2 * n];
        o.rf = T[3 * n];
    }
    return o;
}

// Corrections of the two target components, and the advanced auxiliaries.
template <int V, bool EL>
__device__ __forceinline__ void row_face_apply(const Grid& g, int a, const Group& gr, const RowFace<V>& rf,
                                               const fv<V>& upd, const fv<V>& d0, const fv<V>& d1, fv<V>& t0,
                                               fv<V>& t1)
{
    if (!rf.any) return;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const fv<V>& dv = w == 0 ? d0 : d1;
        fv<V>& t = w == 0 ? t0 : t1;
        fv<V> der;
#pragma unroll
        for (int e = 0; e < V; ++e) der[e] = dv[e] / g.d[a];
        const fv<V> corr = upd * (rf.ra1 * der + rf.rb * rf.phi[w]);
        const bool minus = (EL ? e_face_sign(a, w) : h_face_sign(a, w)) < 0.0f;
        const fv<V> nt = minus ? t - corr : t + corr;
#pragma unroll
        for (int e = 0; e < V; ++e) t[e] = e < rf.n[w] ? nt[e] : t[e];
        stn<V>(rf.p[w], rf.re * rf.phi[w] - rf.rf * der, gr.dup, rf.n[w]);
    }
}

// The z-face that a group reaches into: every cell has its own profile index.
template <int V>
struct ZFace {
    bool any, all;      // some / every cell of the group is in the face
    Side sd;
    int q0;             // profile index of the group's first (low face: last) cell
    bool on[2];         // the row has auxiliaries w
    float* row[2];      // its elements by profile index
    fv<V> phi[2];
    fv<V> upd;
    fv<V> ra1, rb, re, rf;
};

// The group's elements of an auxiliary row, in cell order.
template <int V>
__device__ __forceinline__ fv<V> z_load(const ZFace<V>& o, const float* row)
{
    fv<V> v, r;
    if (o.all) {
        v = *(const typename Vec<V>::utype*)(row + o.q0);
    } else {
        const int p = o.sd.p - 1;  // a cell outside the face reads the nearest element
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = row[min(max(o.q0 + e, 0), p)];
    }
#pragma unroll
    for (int e = 0; e < V; ++e) r[e] = o.sd.high ? v[e] : v[V - 1 - e];
    return r;
}

template <int V>
__device__ __forceinline__ void z_store(const ZFace<V>& o, float* row, const fv<V>& v, const Group& gr)
{
    if (o.all && gr.dup == 0) {
        fv<V> r;
#pragma unroll
        for (int e = 0; e < V; ++e) r[e] = o.sd.high ? v[e] : v[V - 1 - e];
        *(typename Vec<V>::utype*)(row + o.q0) = r;
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int k = gr.k + e;
            if (o.sd.in(k) && e >= gr.dup) row[o.sd.at(k)] = v[e];
        }
    }
}

template <int V, bool EL>
__device__ __forceinline__ ZFace<V> z_face(const Grid& g, const Cpml& cp, const float* tab, const float* upd,
                                           const Group& q)
{
    ZFace<V> o;
    o.sd = side_of<EL>(g, 2, q.k);
    o.any = o.sd.p > 0 && q.k <= o.sd.hi && q.k + V - 1 >= o.sd.lo;
    o.all = q.k >= o.sd.lo && q.k + V - 1 <= o.sd.hi;
    o.q0 = o.sd.high ? q.k - o.sd.lo : o.sd.hi - (q.k + V - 1);
    o.on[0] = o.on[1] = false;
    o.row[0] = o.row[1] = nullptr;
    o.phi[0] = o.phi[1] = o.upd = o.ra1 = o.rb = o.re = o.rf = 0.0f;
    if (o.any) {
        const int depth = EL ? o.sd.p + 1 : o.sd.p;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            // shape (N0, N1, depth), one less along the E target / H source
            const int t = EL ? face_target(2, w) : face_source(2, w);
            const int d0 = g.N[0] - (t == 0 ? 1 : 0), d1 = g.N[1] - (t == 1 ? 1 : 0);
            o.on[w] = q.i < d0 && q.j < d1;
            const long long r = ((long long)q.s * d0 + min(q.i, d0 - 1)) * d1 + min(q.j, d1 - 1);
            o.row[w] = choose(o.sd.high, cp.psi[5][w], cp.psi[4][w]) + r * depth;
            o.phi[w] = z_load<V>(o, o.row[w]);
        }
        const float* T = axis_table(g, tab, 2);
        const unsigned k = (unsigned)q.k, n = (unsigned)g.N[2];
        o.upd = ldv<V>(upd, q.m);
        o.ra1 = ldv<V>(T, k);
        o.rb = ldv<V>(T, n + k);
        o.re = ldv<V>(T, 2u * n + k);
        o.rf = ldv<V>(T, 3u * n + k);
    }
    return o;
}

// Whether cell k of the group has an element in auxiliary w of the face.
template <int V>
__device__ __forceinline__ bool z_has(const ZFace<V>& zf, int w, int k)
{
    return zf.on[w] && k >= zf.sd.lo && k <= zf.sd.hi;
}

template <int V, bool EL>
__device__ __forceinline__ void z_face_apply(const Grid& g, const Group& gr, const ZFace<V>& zf, const fv<V>& d0,
                                             const fv<V>& d1, fv<V>& t0, fv<V>& t1)
{
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const fv<V>& dv = w == 0 ? d0 : d1;
        fv<V>& t = w == 0 ? t0 : t1;
        const bool minus = (EL ? e_face_sign(2, w) : h_face_sign(2, w)) < 0.0f;
        fv<V> der;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            der[e] = dv[e] / g.d[2];
            const float corr = zf.upd[e] * (zf.ra1[e] * der[e] + zf.rb[e] * zf.phi[w][e]);
            t[e] = z_has(zf, w, gr.k + e) ? (minus ? t[e] - corr : t[e] + corr) : t[e];
        }
        if (zf.on[w]) z_store<V>(zf, zf.row[w], zf.re * zf.phi[w] - zf.rf * der, gr);
    }
}

// Component t of the field EL (E, otherwise H) is updated at the cells of a
// row as far as the coordinates on x and y decide it; z decides the rest:
// 0 < k < N2 - 1 for Ex, Ey and Hz, k < N2 - 1 for Ez, Hx and Hy.
template <bool EL>
__device__ __forceinline__ bool row_updated(const Grid& g, int t, int i, int j)
{
    const bool i0 = i > 0, i1 = i < g.N[0] - 1, j0 = j > 0, j1 = j < g.N[1] - 1;
    if (EL) return t == 0 ? i1 && j0 && j1 : (t == 1 ? j1 && i0 && i1 : i0 && i1 && j0 && j1);
    return t == 0 ? i0 && i1 && j1 : (t == 1 ? j0 && j1 && i1 : i1 && j1);
}

template <int V, bool BOTH>
__device__ __forceinline__ fv<V> pick_z(bool row, int k, int n, const fv<V>& a, const fv<V>& b)
{
    fv<V> o;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = row && k + e < n - 1 && (!BOTH || k + e > 0) ? a[e] : b[e];
    return o;
}

// ---------------------------------------------------------------------------
// Forward magnetic half step (deepgpr_cpu.c:886-1100)
// ---------------------------------------------------------------------------
template <int ORDER, int V, bool XY>
__device__ __forceinline__ void fwd_h_group(const Grid& g, const float* hcurl, const float* hrhs, const CF3& E,
                                            const F3& H, const Cpml& cp, const float* tab, int has_cpml,
                                            const Group& q, float* s0, float* s1)
{
    const int sx = g.plane, sy = g.N[2], n2 = g.N[2];
    RowFace<V> fx, fy;
    fv<V> upd = 0.0f;
    if constexpr (!XY) {
        upd = ldv<V>(hrhs, q.m);
        fx = row_face<V, false>(g, cp, tab, has_cpml, 0, q);
        fy = row_face<V, false>(g, cp, tab, has_cpml, 1, q);
    }
    const fv<V> ex = ldv<V>(E.c[0], q.m), ey = ldv<V>(E.c[1], q.m);
    fv<V> h0 = ldv<V>(H.c[0], q.m), h1 = ldv<V>(H.c[1], q.m), h2 = ldv<V>(H.c[2], q.m);
    const fv<V> u1 = ldv<V>(hcurl, q.m);
    const bool lx = q.i < g.N[0] - 1, ly = q.j < g.N[1] - 1;
    stv<V>(s0, (unsigned)q.k, ex, q.dup);
    stv<V>(s1, (unsigned)q.k, ey, q.dup);
    const fv<V> dzy = diff_row<ORDER, V, true, XY>(E.c[2], q.m, sy, q.j, g.N[1], ly);
    const fv<V> dzx = diff_row<ORDER, V, true, XY>(E.c[2], q.m, sx, q.i, g.N[0], lx);
    const fv<V> dyx = diff_row<ORDER, V, true, XY>(E.c[1], q.m, sx, q.i, g.N[0], lx);
    const fv<V> dxy = diff_row<ORDER, V, true, XY>(E.c[0], q.m, sy, q.j, g.N[1], ly);
    __syncthreads();
    const fv<V> dyz = diff_z<ORDER, V, true>(ey, s1, q, n2), dxz = diff_z<ORDER, V, true>(ex, s0, q, n2);
    const fv<V> uy = axis_coeffs<V>(g, u1, 1), uz = axis_coeffs<V>(g, u1, 2);
    const fv<V> n0 = h0 - uy * dzy + uz * dyz, n1 = h1 - uz * dxz + u1 * dzx, nz = h2 - u1 * dyx + uy * dxy;
    if (XY && q.zplain) {
        h0 = n0;
        h1 = n1;
        h2 = nz;
    } else {
        h0 = pick_z<V, false>(XY || row_updated<false>(g, 0, q.i, q.j), q.k, n2, n0, h0);
        h1 = pick_z<V, false>(XY || row_updated<false>(g, 1, q.i, q.j), q.k, n2, n1, h1);
        h2 = pick_z<V, true>(XY || row_updated<false>(g, 2, q.i, q.j), q.k, n2, nz, h2);
    }
    if constexpr (!XY) {
        {
            // x faces: (Hy, Ez), (Hz, Ey); y faces: (Hx, Ez), (Hz, Ex)
            row_face_apply<V, false>(g, 0, q, fx, upd, dzx, dyx, h1, h2);
            row_face_apply<V, false>(g, 1, q, fy, upd, dzy, dxy, h0, h2);
        }
    }
    // z faces: (Hx, Ey), (Hy, Ex)
    if (!q.zplain && has_cpml) {
        const ZFace<V> zf = z_face<V, false>(g, cp, tab, hrhs, q);
        if (zf.any) z_face_apply<V, false>(g, q, zf, dyz, dxz, h0, h1);
    }
    stv<V>(H.c[0], q.m, h0, q.dup);
    stv<V>(H.c[1], q.m, h1, q.dup);
    stv<V>(H.c[2], q.m, h2, q.dup);
}

__device__ __forceinline__ CF3 shot_of(const CF3& f, long long off)
{
    return {{f.c[0] + off, f.c[1] + off, f.c[2] + off}};
}
__device__ __forceinline__ F3 shot_of(const F3& f, long long off)
{
    return {{f.c[0] + off, f.c[1] + off, f.c[2] + off}};
}

// This thread's group. An idle thread takes a copy of another's, with every
// cell owned elsewhere: it keeps step with the barriers and stores nothing.
template <int V>
__device__ __forceinline__ void thread_group(const Grid& g, const RowMap& rm, const RowKind& kd, int i, int j0, int nj,
                                             Group& q, int& row)
{
    const bool live = row_thread(rm, kd, V, threadIdx.x, nj, row, q.k, q.dup);
    q.i = i;
    q.j = j0 + row;
    q.s = blockIdx.y;
    q.m = (unsigned)(i * g.plane + q.j * g.N[2] + q.k);
    q.zplain = q.k >= rm.zlo && q.k + V - 1 <= rm.zhi;
    if (!live) q.dup = V;
}

// Threads of the wavefronts that hold groups of a workgroup; the others end at
// once (a barrier does not count wavefronts that have ended). An edge row of 257
// cells holds 129 of 256 threads: with the idle wavefront kept, 99 x 99 x 257
// fields at order 4 took 4 to 6 % longer, 89 x 89 x 257 with CPML 24 11 %.
__device__ __forceinline__ int live_threads(const RowKind& kd) { return (kd.rb * kd.gpr + 63) / 64 * 64; }

template <int ORDER, int V>
__global__ __launch_bounds__(kRowMaxThreads) void k_row_fwd_h(Grid g, const float* hcurl, const float* hrhs, CF3 E, F3 H, Cpml cp,
                                                   const float* tab, int has_cpml, RowMap rm)
{
    extern __shared__ __align__(16) float sw[];  // two components of the workgroup's rows
    int i, j0, nj, row;
    const int kind = row_block(rm, blockIdx.x, i, j0, nj);
    if (kind < 0) return;
    if ((int)threadIdx.x >= live_threads(kind == 1 ? rm.plain : rm.edge)) return;
    const long long so = (long long)blockIdx.y * g.cells;
    const CF3 Es = shot_of(E, so);
    const F3 Hs = shot_of(H, so);
    Group q;
    if (kind == 1) {
        thread_group<V>(g, rm, rm.plain, i, j0, nj, q, row);
        float* s0 = sw + row * rm.plain.gpr * V;
        fwd_h_group<ORDER, V, true>(g, hcurl, hrhs, Es, Hs, cp, tab, has_cpml, q, s0, s0 + rm.lds);
    } else {
        thread_group<V / 2>(g, rm, rm.edge, i, j0, nj, q, row);
        float* s0 = sw + row * rm.edge.gpr * (V / 2);
        fwd_h_group<ORDER, V / 2, false>(g, hcurl, hrhs, Es, Hs, cp, tab, has_cpml, q, s0, s0 + rm.lds);
    }
}

// ---------------------------------------------------------------------------
// Forward electric half step: curl update, CPML, sources, history, receivers
// (deepgpr_cpu.c:670-883, 644-668, 1559-1633)
// ---------------------------------------------------------------------------
// History values of the group's own cells from element idx on.
template <int V>
__device__ __forceinline__ void store_hist_group(void* base, long long idx, fv<V> v, int kind, bool whole,
                                                 const bool (&own)[V])
{
    if (kind == kF32) {
        float* p = (float*)base + idx;
        if (whole) {
            *(typename Vec<V>::utype*)p = v;
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (own[e]) p[e] = v[e];
        }
        return;
    }
    typedef unsigned short us __attribute__((ext_vector_type(V)));
    typedef unsigned short usu __attribute__((ext_vector_type(V), aligned(2)));
    us b;
#pragma unroll
    for (int e = 0; e < V; ++e) b[e] = kind == kF16 ? f32_to_f16_bits(v[e]) : f32_to_bf16_bits(v[e]);
    uint16_t* p = (uint16_t*)base + idx;
    if (whole) {
        *(usu*)p = b;
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (own[e]) p[e] = b[e];
    }
}

// Sources of a workgroup up to which every thread looks at each of them. More
// (they are in order of their cells) a thread searches for its own: with a plane
// of 80 x 80 sources on 80 x 80 x 80 a workgroup of seven rows looked at 560,
// 120 us a step more than without them.
constexpr int kFewSources = 4;

template <int ORDER, int V, bool XY>
__device__ __forceinline__ void fwd_e_group(const Grid& g, const float* ca, const float* ccurl, const float* cb,
                                            const CF3& Hf, const F3& E, const Cpml& cp, const float* tab, int has_cpml,
                                            const SourceBlocks& src, const HistWrite& hist, int sb, int se,
                                            const Group& q, float* s0, float* s1)
{
    const int sx = g.plane, sy = g.N[2], n2 = g.N[2];
    RowFace<V> fx, fy;
    if constexpr (!XY) {
        fx = row_face<V, true>(g, cp, tab, has_cpml, 0, q);
        fy = row_face<V, true>(g, cp, tab, has_cpml, 1, q);
    }
    const fv<V> hx = ldv<V>(Hf.c[0], q.m), hy = ldv<V>(Hf.c[1], q.m);
    fv<V> e[3] = {ldv<V>(E.c[0], q.m), ldv<V>(E.c[1], q.m), ldv<V>(E.c[2], q.m)};
    const fv<V> u0 = ldv<V>(ca, q.m), u1 = ldv<V>(ccurl, q.m);
    fv<V> cbv = 0.0f;
    if constexpr (!XY) cbv = ldv<V>(cb, q.m);
    const bool lx = q.i >= 1, ly = q.j >= 1;
    stv<V>(s0, (unsigned)q.k, hx, q.dup);
    stv<V>(s1, (unsigned)q.k, hy, q.dup);
    const fv<V> dzy = diff_row<ORDER, V, false, XY>(Hf.c[2], q.m, sy, q.j, g.N[1], ly);
    const fv<V> dzx = diff_row<ORDER, V, false, XY>(Hf.c[2], q.m, sx, q.i, g.N[0], lx);
    const fv<V> dyx = diff_row<ORDER, V, false, XY>(Hf.c[1], q.m, sx, q.i, g.N[0], lx);
    const fv<V> dxy = diff_row<ORDER, V, false, XY>(Hf.c[0], q.m, sy, q.j, g.N[1], ly);
    __syncthreads();
    const fv<V> dyz = diff_z<ORDER, V, false>(hy, s1, q, n2), dxz = diff_z<ORDER, V, false>(hx, s0, q, n2);
    const fv<V> uy = axis_coeffs<V>(g, u1, 1), uz = axis_coeffs<V>(g, u1, 2);
    const bool up[3] = {XY || row_updated<true>(g, 0, q.i, q.j), XY || row_updated<true>(g, 1, q.i, q.j),
                        XY || row_updated<true>(g, 2, q.i, q.j)};
    const fv<V> v0 = u0 * e[0] + uy * dzy - uz * dyz, v1 = u0 * e[1] + uz * dxz - u1 * dzx,
                v2 = u0 * e[2] + u1 * dyx - uy * dxy;
    if (XY && q.zplain) {
        e[0] = v0;
        e[1] = v1;
        e[2] = v2;
    } else {
        e[0] = pick_z<V, true>(up[0], q.k, n2, v0, e[0]);
        e[1] = pick_z<V, true>(up[1], q.k, n2, v1, e[1]);
        e[2] = pick_z<V, false>(up[2], q.k, n2, v2, e[2]);
    }
    if constexpr (!XY) {
        // x faces: (Ey, Hz), (Ez, Hy); y faces: (Ex, Hz), (Ez, Hx)
        row_face_apply<V, true>(g, 0, q, fx, cbv, dzx, dyx, e[1], e[2]);
        row_face_apply<V, true>(g, 1, q, fy, cbv, dzy, dxy, e[0], e[2]);
    }
    // z faces: (Ex, Hy), (Ey, Hx)
    if (!q.zplain && has_cpml) {
        const ZFace<V> zf = z_face<V, true>(g, cp, tab, cb, q);
        if (zf.any) z_face_apply<V, true>(g, q, zf, dyz, dxz, e[0], e[1]);
    }
    // sources and the history load cb, and the history ca and the old values,
    // again rather than keep them in registers all along
    unsigned m = q.m;
    asm volatile("" : "+v"(m));
    auto add = [&](const int2& ent) {
        const unsigned at = (unsigned)ent.x - q.m;
        if (at < (unsigned)V) {
            const fv<V> cbv = ldv<V>(cb, m);
            const float scale = src.wave[(long long)ent.y * src.nt + src.it] * src.dl / src.vol;
#pragma unroll
            for (int y = 0; y < V; ++y)
#pragma unroll
                for (int t = 0; t < 3; ++t)
                    if (at == (unsigned)y && t == src.comp) e[t][y] -= cbv[y] * scale;
        }
    };
    if (se - sb <= kFewSources) {
        for (int x = sb; x < se; ++x) add(src.entries[x]);
    } else {
        int x = sb, end = se;  // the first source on the group's cells or beyond them
        while (x < end) {
            const int mid = (x + end) >> 1;
            if ((unsigned)src.entries[mid].x < q.m) x = mid + 1;
            else end = mid;
        }
        for (; x < se; ++x) {
            const int2 ent = src.entries[x];
            if ((unsigned)ent.x >= q.m + V) break;
            add(ent);
        }
    }
    if (hist.active && q.i >= hist.box.x0 && q.i < hist.box.x0 + hist.box.nx && q.j >= hist.box.y0 &&
        q.j < hist.box.y0 + hist.box.ny) {
        const int z = q.k - hist.box.z0;
        const long long base = (long long)q.s * hist.box.cells +
                               ((long long)(q.i - hist.box.x0) * hist.box.ny + (q.j - hist.box.y0)) * hist.box.nz + z;
        const bool whole = q.dup == 0 && z >= 0 && z + V <= hist.box.nz;
        bool own[V];
#pragma unroll
        for (int y = 0; y < V; ++y) own[y] = y >= q.dup && z + y >= 0 && z + y < hist.box.nz;
        fv<V> cbv = 0.0f, cav = 0.0f;
        if (hist.save_r) {
            cbv = ldv<V>(cb, m);
            cav = ldv<V>(ca, m);
        }
#pragma unroll
        for (int comp = 0; comp < 3; ++comp) {
            if (hist.mode != 3 && comp != 2) continue;
            const int ci = hist.mode == 3 ? comp : 0;
            const fv<V> old = ldv<V>(E.c[comp], m);
            if (hist.save_e)
                store_hist_group<V>(hist.e_base, ci * hist.e_cstride + base, old, hist.e_kind, whole, own);
            if (hist.save_r) {
                fv<V> rhs;
#pragma unroll
                for (int y = 0; y < V; ++y) {
                    const bool u = up[comp] && q.k + y < n2 - 1 && (comp == 2 || q.k + y > 0);
                    const float a = u ? cav[y] : 1.0f;
                    rhs[y] = cbv[y] != 0.0f ? (e[comp][y] - a * old[y]) / cbv[y] : 0.0f;
                }
                store_hist_group<V>(hist.r_base, ci * hist.r_cstride + base, rhs, hist.r_kind, whole, own);
            }
        }
    }
    stv<V>(E.c[0], q.m, e[0], q.dup);
    stv<V>(E.c[1], q.m, e[1], q.dup);
    stv<V>(E.c[2], q.m, e[2], q.dup);
}

template <int ORDER, int V>
__global__ __launch_bounds__(kRowMaxThreads) void k_row_fwd_e(Grid g, const float* ca, const float* ccurl, const float* cb,
                                                   CF3 Hf, F3 E, Cpml cp, const float* tab, int has_cpml,
                                                   SourceBlocks src, HistWrite hist, RowReceivers rx, RowMap rm)
{
    extern __shared__ __align__(16) float sw[];
    int i, j0, nj, row;
    const int kind = row_block(rm, blockIdx.x, i, j0, nj);
    if (kind < 0) return;
    const int live = live_threads(kind == 1 ? rm.plain : rm.edge);
    if ((int)threadIdx.x >= live) return;
    const int blin = blockIdx.x + gridDim.x * blockIdx.y;
    int sb = 0, se = 0;
    if (src.count > 0) {
        sb = src.block_off[blin];
        se = src.block_off[blin + 1];
    }
    const long long so = (long long)blockIdx.y * g.cells;
    const CF3 Hs = shot_of(Hf, so);
    const F3 Es = shot_of(E, so);
    Group q;
    if (kind == 1) {
        thread_group<V>(g, rm, rm.plain, i, j0, nj, q, row);
        float* s0 = sw + row * rm.plain.gpr * V;
        fwd_e_group<ORDER, V, true>(g, ca, ccurl, cb, Hs, Es, cp, tab, has_cpml, src, hist, sb, se, q, s0,
                                    s0 + rm.lds);
    } else {
        thread_group<V / 2>(g, rm, rm.edge, i, j0, nj, q, row);
        float* s0 = sw + row * rm.edge.gpr * (V / 2);
        fwd_e_group<ORDER, V / 2, false>(g, ca, ccurl, cb, Hs, Es, cp, tab, has_cpml, src, hist, sb, se, q, s0,
                                         s0 + rm.lds);
    }
    if (rx.count > 0) {
        // receivers on cells of this workgroup, read back once it has stored them
        const int b0 = rx.off[blin], b1 = rx.off[blin + 1];
        if (b0 == b1) return;
        __syncthreads();
        const float* f = E.c[rx.comp] + (long long)blockIdx.y * g.cells;
        for (int x = b0 + (int)threadIdx.x; x < b1; x += live) {
            const int2 ent = rx.ent[x];
            rx.out[((long long)blockIdx.y * rx.nt + src.it) * rx.nrx + ent.y] = f[ent.x];
        }
    }
}

// ---------------------------------------------------------------------------
// Adjoint half steps (deepgpr_cpu.c:509-527, 1153-1239, 1332-1410)
// ---------------------------------------------------------------------------
// EL: the transposed electric step, lambda_H[u] += sum over a != u of
// D-^T W(u, a); otherwise the transposed magnetic step, lambda_E[u] =
// (ca) lambda_E[u] + sum of D+^T W(u, a). The channel weight W(u, a) of a cell
// is the CPML term of its faces on axis a (old auxiliaries) plus the curl
// term +-cu lambda[t], t the third axis, where component t is updated.

// The curl term of channel (u, a) enters with +cu (otherwise with -cu).
template <bool EL>
__device__ __forceinline__ bool channel_plus(int u, int a)
{
    const int t = 3 - u - a;
    const int t1 = t == 2 ? 0 : t + 1;
    return (a == t1) == EL;
}

// Offset of the r-th tap (r = 1 .. R) of the transposed stencil: the taps that
// are added and those that are subtracted.
template <bool EL>
__device__ __forceinline__ constexpr int tap_off(int r, bool added)
{
    return EL ? (added ? 1 - r : r) : (added ? -r : r - 1);
}

// One term of a transposed stencil with coefficient kc.
template <int ORDER, typename T>
__device__ __forceinline__ void add_tap(T& acc, float kc, const T& w, bool plus)
{
    if constexpr (ORDER <= 2) {
        if (plus) acc += w;
        else acc -= w;
    } else {
        if (plus) acc += kc * w;
        else acc -= kc * w;
    }
}

// Channels (u1, a) and (u2, a) of axis a (0 or 1) of cells in plain rows, with
// l1 and l2 the lambda components u1 < u2 (channel (u1, a) reads l2 and the
// other way round); o1, o2, ku: their values and the coefficient at the cells.
template <int ORDER, int V, bool EL>
__device__ __forceinline__ void gather_plain(const Grid& g, int a, const float* l1, const float* l2, const float* cu,
                                             unsigned m, int st, int u1, int u2, const fv<V>& o1, const fv<V>& o2,
                                             const fv<V>& ku, fv<V>& g1, fv<V>& g2)
{
    constexpr int R = Radius<ORDER>::value;
    const bool p1 = channel_plus<EL>(u1, a), p2 = channel_plus<EL>(u2, a);
    fv<V> kk[2 * R], x1[2 * R], x2[2 * R];
#pragma unroll
    for (int t = 0; t < 2 * R; ++t) {
        const int off = tap_off<EL>(t / 2 + 1, t % 2 == 0);
        const ptrdiff_t o = (ptrdiff_t)off * st;
        kk[t] = off == 0 ? ku : ldv<V>(cu + o, m);
        x1[t] = off == 0 ? o2 : ldv<V>(l2 + o, m);
        x2[t] = off == 0 ? o1 : ldv<V>(l1 + o, m);
    }
    g1 = 0.0f;
    g2 = 0.0f;
#pragma unroll
    for (int t = 0; t < 2 * R; ++t) {
        const float kc = stencil_c(R, t / 2 + 1);
        const fv<V> k = axis_coeffs<V>(g, kk[t], a);
        add_tap<ORDER>(g1, kc, k * x1[t], (t % 2 == 0) == p1);
        add_tap<ORDER>(g2, kc, k * x2[t], (t % 2 == 0) == p2);
    }
}

// The same in any row: clamped transposed stencils, cells that are not updated
// and CPML terms.
template <int ORDER, int V, bool EL>
__device__ __forceinline__ void gather_edge(const Grid& g, int a, const float* l1, const float* l2, const float* cu,
                                            const float* upd, const Cpml& cp, const float* tab, int has_cpml,
                                            const Group& q, int st, int u1, int u2, fv<V>& g1, fv<V>& g2)
{
    constexpr int R = Radius<ORDER>::value;
    const int c[3] = {q.i, q.j, q.k};
    const int n = g.N[a];
    const bool p1 = channel_plus<EL>(u1, a), p2 = channel_plus<EL>(u2, a);
    const int w1 = face_source(a, 0) == u1 ? 0 : 1, w2 = 1 - w1;
    // every load of the axis first: a tap outside the stencil reads the cell,
    // one outside the face an element of it that is not used
    const int ca = a == 0 ? q.i : q.j;
    const Side sd = side_of<EL>(g, a, ca);
    const bool face = has_cpml && sd.p > 0;
    const float* T = axis_table(g, tab, a);
    fv<V> kk[2 * R], x1[2 * R], x2[2 * R], uc[2 * R], b1[2 * R], b2[2 * R];
    float ra1[2 * R], rf[2 * R];
    int n1 = 0, n2 = 0;
#pragma unroll
    for (int t = 0; t < 2 * R; ++t) {
        const int r = t / 2 + 1, off = tap_off<EL>(r, t % 2 == 0), ct = ca + off;
        const int rs = EL ? fit_bwd_sel(ct, n, R) : fit_fwd_sel(ct, n, R);
        const bool ok = ct >= 0 && ct < n && r <= rs;
        const unsigned mt = q.m + (unsigned)((ok ? off : 0) * st);
        kk[t] = ldv<V>(cu, mt);
        x1[t] = ldv<V>(l2, mt);
        x2[t] = ldv<V>(l1, mt);
        uc[t] = b1[t] = b2[t] = 0.0f;
        ra1[t] = rf[t] = 0.0f;
        if (face) {
            const int cf = min(max(ct, sd.lo), sd.hi);
            uc[t] = ldv<V>(upd, mt);
            ra1[t] = T[cf];
            rf[t] = T[3 * n + cf];
            const float* r1 = psi_row<EL>(g, cp.psi, a, w1, sd, sd.at(cf), q.i, q.j, q.s, n1);
            const float* r2 = psi_row<EL>(g, cp.psi, a, w2, sd, sd.at(cf), q.i, q.j, q.s, n2);
            b1[t] = ldn<V>(r1 + q.k, n1 - q.k);
            b2[t] = ldn<V>(r2 + q.k, n2 - q.k);
        }
    }
    // component updated, apart from the coordinate on axis a: channel (u1, a)
    // targets component u2, channel (u2, a) component u1
    bool up1[V], up2[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const int z = q.k + e;
        const int c1 = u1 == 2 ? z : c[u1], c2 = u2 == 2 ? z : c[u2];
        const bool i1 = c1 < g.N[u1] - 1, i2 = c2 < g.N[u2] - 1;
        up1[e] = i1 && i2 && (EL ? c1 > 0 : c2 > 0);
        up2[e] = i1 && i2 && (EL ? c2 > 0 : c1 > 0);
    }
    const float inv = 1.0f / g.d[a];
    const float s1 = EL ? e_face_sign(a, w1) : h_face_sign(a, w1), s2 = EL ? e_face_sign(a, w2) : h_face_sign(a, w2);
    g1 = 0.0f;
    g2 = 0.0f;
#pragma unroll
    for (int t = 0; t < 2 * R; ++t) {
        const int r = t / 2 + 1, off = tap_off<EL>(r, t % 2 == 0), ct = ca + off;
        const int rs = EL ? fit_bwd_sel(ct, n, R) : fit_fwd_sel(ct, n, R);
        const bool ok = ct >= 0 && ct < n && r <= rs;  // order 2 has no radius test: r is 1
        const bool in = face && sd.in(ct), along = EL ? ct > 0 && ct < n - 1 : ct < n - 1;
        const fv<V> k = axis_coeffs<V>(g, kk[t], a);
        const fv<V> y1 = 0.0f + (s1 * uc[t] * ra1[t] * x1[t] - rf[t] * b1[t]) * inv;
        const fv<V> y2 = 0.0f + (s2 * uc[t] * ra1[t] * x2[t] - rf[t] * b2[t]) * inv;
        fv<V> v1, v2;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            v1[e] = in && q.k + e < n1 ? y1[e] : 0.0f;
            v2[e] = in && q.k + e < n2 ? y2[e] : 0.0f;
        }
        const fv<V> z1 = p1 ? v1 + k * x1[t] : v1 - k * x1[t], z2 = p2 ? v2 + k * x2[t] : v2 - k * x2[t];
        const float kc = stencil_c(ORDER <= 2 ? 1 : rs, r);
        fv<V> m1 = g1, m2 = g2, c1, c2;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            c1[e] = up1[e] && along ? z1[e] : v1[e];
            c2[e] = up2[e] && along ? z2[e] : v2[e];
        }
        add_tap<ORDER>(m1, kc, c1, t % 2 == 0);
        add_tap<ORDER>(m2, kc, c2, t % 2 == 0);
        g1 = pick<V>(ok, m1, g1);
        g2 = pick<V>(ok, m2, g2);
    }
}

// The auxiliaries of the face on axis a (0 or 1) advance at their own cells.
template <int V, bool EL>
__device__ __forceinline__ void psi_advance(const Grid& g, int a, const fv<V> (&lam)[3], const float* upd,
                                            const Cpml& cp, const PsiOut& out, const float* tab, int has_cpml,
                                            const Group& gr)
{
    const int c = a == 0 ? gr.i : gr.j, n = g.N[a];
    const Side sd = side_of<EL>(g, a, c);
    if (!has_cpml || !sd.in(c)) return;
    const float* T = axis_table(g, tab, a) + c;
    const float rb = T[n], re = T[2 * n];
    const fv<V> uc = ldv<V>(upd, gr.m);
    fv<V> old[2];
    int len[2];
#pragma unroll
    for (int w = 0; w < 2; ++w)
        old[w] = ldn<V>(psi_row<EL>(g, cp.psi, a, w, sd, sd.at(c), gr.i, gr.j, gr.s, len[w]) + gr.k, len[w] - gr.k);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const float sign = EL ? e_face_sign(a, w) : h_face_sign(a, w);
        float* to = psi_row<EL>(g, out.psi, a, w, sd, sd.at(c), gr.i, gr.j, gr.s, len[w]) + gr.k;
        stn<V>(to, sign * uc * rb * lam[face_target(a, w)] + re * old[w], gr.dup, len[w] - gr.k);
    }
}

// Channels (x, z) and (y, z): the weights of the group's own cells (w0, w1,
// with the z-CPML terms, whose auxiliaries have advanced by now) and, in s0 and
// s1, those of the row, which its moved-back last group takes for the cells of
// the group before it (row_own_element).
template <int ORDER, int V, bool EL>
__device__ __forceinline__ void gather_z(const Group& q, int n, const float* s0, const float* s1, const fv<V>& w0,
                                         const fv<V>& w1, fv<V>& g0, fv<V>& g1)
{
    constexpr int R = Radius<ORDER>::value;
    constexpr int L = EL ? R - 1 : R, U = EL ? R : R - 1;
    float a0[V + L + U], a1[V + L + U];
#pragma unroll
    for (int e = 0; e < L; ++e) {
        const int x = max(q.k - L + e, 0);
        a0[e] = s0[x];
        a1[e] = s1[x];
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
        a0[L + e] = w0[e];
        a1[L + e] = w1[e];
    }
    if (q.dup > 0) {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (!row_own_element(e, q.dup, V)) {
                a0[L + e] = s0[q.k + e];
                a1[L + e] = s1[q.k + e];
            }
    }
#pragma unroll
    for (int e = 0; e < U; ++e) {
        const int x = min(q.k + V + e, n - 1);
        a0[L + V + e] = s0[x];
        a1[L + V + e] = s1[x];
    }
    if (q.k >= 2 * R - 1 && q.k + V - 1 <= n - 2 * R) {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
            for (int t = 0; t < 2 * R; ++t) {
                const int at = L + e + tap_off<EL>(t / 2 + 1, t % 2 == 0);
                add_tap<ORDER>(x0, stencil_c(R, t / 2 + 1), a0[at], t % 2 == 0);
                add_tap<ORDER>(x1, stencil_c(R, t / 2 + 1), a1[at], t % 2 == 0);
            }
            g0[e] = x0;
            g1[e] = x1;
        }
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
            for (int t = 0; t < 2 * R; ++t) {
                const int r = t / 2 + 1, off = tap_off<EL>(r, t % 2 == 0), ct = q.k + e + off;
                const int rs = EL ? fit_bwd_sel(ct, n, R) : fit_fwd_sel(ct, n, R);
                const bool ok = ct >= 0 && ct < n && r <= rs;
                const float kc = stencil_c(ORDER <= 2 ? 1 : rs, r);
                float y0 = x0, y1 = x1;
                add_tap<ORDER>(y0, kc, a0[L + e + off], t % 2 == 0);
                add_tap<ORDER>(y1, kc, a1[L + e + off], t % 2 == 0);
                x0 = ok ? y0 : x0;
                x1 = ok ? y1 : x1;
            }
            g0[e] = x0;
            g1[e] = x1;
        }
    }
}

// The z-CPML terms of the group's own channel weights, and its auxiliaries
// advanced in place: the terms of cells that another thread owns may come from
// advanced ones and are not used (row_own_element).
template <int V, bool EL>
__device__ __forceinline__ void z_weights(const Grid& g, const Group& gr, const ZFace<V>& zf, const fv<V>& lx,
                                          const fv<V>& ly, fv<V>& w0, fv<V>& w1)
{
    const float inv = 1.0f / g.d[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        // w = 0: target x, source y (channel (y, z)); w = 1: target y, source x
        const float sign = EL ? e_face_sign(2, w) : h_face_sign(2, w);
        const fv<V>& lt = w == 0 ? lx : ly;
        fv<V>& wt = w == 0 ? w1 : w0;
        const fv<V> term = 0.0f + (sign * zf.upd * zf.ra1 * lt - zf.rf * zf.phi[w]) * inv;
#pragma unroll
        for (int e = 0; e < V; ++e) wt[e] = z_has(zf, w, gr.k + e) ? term[e] : 0.0f;
        if (zf.on[w]) z_store<V>(zf, zf.row[w], sign * zf.upd * zf.rb * lt + zf.re * zf.phi[w], gr);
    }
}

template <int ORDER, int V, bool XY, bool EL>
__device__ __forceinline__ void adj_group(const Grid& g, const float* cu, const float* upd, const float* ca,
                                          const F3& lam, const F3& out, const Cpml& cp, const PsiOut& po,
                                          const float* tab, int has_cpml, const Group& q, bool px, bool py, float* s0, float* s1)
{
    const int sx = g.plane, sy = g.N[2], n2 = g.N[2];
    const fv<V> l[3] = {ldv<V>(lam.c[0], q.m), ldv<V>(lam.c[1], q.m), ldv<V>(lam.c[2], q.m)};
    const fv<V> ku = ldv<V>(cu, q.m);
    // the z-channel weights of the own cells, shared with the row
    fv<V> w0 = 0.0f, w1 = 0.0f;
    if (!q.zplain && has_cpml) {
        const ZFace<V> zf = z_face<V, EL>(g, cp, tab, upd, q);
        if (zf.any) z_weights<V, EL>(g, q, zf, l[0], l[1], w0, w1);
    }
    {
        const fv<V> kz = axis_coeffs<V>(g, ku, 2);
        const fv<V> a0 = channel_plus<EL>(0, 2) ? w0 + kz * l[1] : w0 - kz * l[1];
        const fv<V> a1 = channel_plus<EL>(1, 2) ? w1 + kz * l[0] : w1 - kz * l[0];
        // channel (x, z) targets y, channel (y, z) targets x
        if (XY && q.zplain) {
            w0 = a0;
            w1 = a1;
        } else {
            w0 = pick_z<V, EL>(XY || row_updated<EL>(g, 1, q.i, q.j), q.k, n2, a0, w0);
            w1 = pick_z<V, EL>(XY || row_updated<EL>(g, 0, q.i, q.j), q.k, n2, a1, w1);
        }
    }
    stv<V>(s0, (unsigned)q.k, w0, q.dup);
    stv<V>(s1, (unsigned)q.k, w1, q.dup);
    fv<V> x1, x2, y0, y2, z0, z1;  // channels (component, axis)
    if constexpr (XY) {
        gather_plain<ORDER, V, EL>(g, 0, lam.c[1], lam.c[2], cu, q.m, sx, 1, 2, l[1], l[2], ku, x1, x2);
        gather_plain<ORDER, V, EL>(g, 1, lam.c[0], lam.c[2], cu, q.m, sy, 0, 2, l[0], l[2], ku, y0, y2);
    } else {
        if (px) gather_plain<ORDER, V, EL>(g, 0, lam.c[1], lam.c[2], cu, q.m, sx, 1, 2, l[1], l[2], ku, x1, x2);
        else gather_edge<ORDER, V, EL>(g, 0, lam.c[1], lam.c[2], cu, upd, cp, tab, has_cpml, q, sx, 1, 2, x1, x2);
        if (py) gather_plain<ORDER, V, EL>(g, 1, lam.c[0], lam.c[2], cu, q.m, sy, 0, 2, l[0], l[2], ku, y0, y2);
        else gather_edge<ORDER, V, EL>(g, 1, lam.c[0], lam.c[2], cu, upd, cp, tab, has_cpml, q, sy, 0, 2, y0, y2);
        psi_advance<V, EL>(g, 0, l, upd, cp, po, tab, has_cpml, q);
        psi_advance<V, EL>(g, 1, l, upd, cp, po, tab, has_cpml, q);
    }
    // A plain gather takes every tap as updated. Where the own coordinates say
    // that component 3 - u - a is not, all taps of channel (u, a) are zero.
    const fv<V> none = 0.0f;
    const bool ends = XY ? !q.zplain : true;
    if (px && ends) {
        const bool jo = XY || (q.j < g.N[1] - 1 && (EL ? q.j > 0 : true)), ji = XY || (q.j < g.N[1] - 1 && (EL ? true : q.j > 0));
        x1 = pick_z<V, !EL>(jo, q.k, n2, x1, none);
        x2 = pick_z<V, EL>(ji, q.k, n2, x2, none);
    }
    if (py && ends) {
        const bool io = XY || (q.i < g.N[0] - 1 && (EL ? q.i > 0 : true)), ii = XY || (q.i < g.N[0] - 1 && (EL ? true : q.i > 0));
        y0 = pick_z<V, !EL>(io, q.k, n2, y0, none);
        y2 = pick_z<V, EL>(ii, q.k, n2, y2, none);
    }
    // loaded here, not before the gathers: 16 registers less all along
    unsigned m = q.m;
    asm volatile("" : "+v"(m));
    fv<V> o[3] = {ldv<V>(out.c[0], m), ldv<V>(out.c[1], m), ldv<V>(out.c[2], m)};
    fv<V> cav = 0.0f;
    if (!EL) cav = ldv<V>(ca, m);
    __syncthreads();
    gather_z<ORDER, V, EL>(q, n2, s0, s1, w0, w1, z0, z1);
    if (!EL) {
        if (XY && q.zplain) {
            o[0] = cav * o[0];
            o[1] = cav * o[1];
            o[2] = cav * o[2];
        } else {
            o[0] = pick_z<V, true>(XY || row_updated<true>(g, 0, q.i, q.j), q.k, n2, cav * o[0], o[0]);
            o[1] = pick_z<V, true>(XY || row_updated<true>(g, 1, q.i, q.j), q.k, n2, cav * o[1], o[1]);
            o[2] = pick_z<V, false>(XY || row_updated<true>(g, 2, q.i, q.j), q.k, n2, cav * o[2], o[2]);
        }
    }
    stv<V>(out.c[0], q.m, o[0] + y0 + z0, q.dup);
    stv<V>(out.c[1], q.m, o[1] + x1 + z1, q.dup);
    stv<V>(out.c[2], q.m, o[2] + x2 + y2, q.dup);
}

template <int ORDER, int V, bool EL>
__global__ __launch_bounds__(kRowMaxThreads) void k_row_adj(Grid g, const float* cu, const float* upd, const float* ca, F3 lam,
                                                 F3 out, Cpml cp, PsiOut po, const float* tab, int has_cpml,
                                                 RowAdjReceivers rx, RowMap rm)
{
    extern __shared__ __align__(16) float sw[];  // two channels of the workgroup's rows
    int i, j0, nj, row;
    const int kind = row_block(rm, blockIdx.x, i, j0, nj);
    if (kind < 0) return;
    const int live = live_threads(kind == 1 ? rm.plain : rm.edge);
    if ((int)threadIdx.x >= live) return;
    const long long so = (long long)blockIdx.y * g.cells;
    const F3 ls = shot_of(lam, so), os = shot_of(out, so);
    Group q;
    if (kind == 1) {
        thread_group<V>(g, rm, rm.plain, i, j0, nj, q, row);
        float* s0 = sw + row * rm.plain.gpr * V;
        adj_group<ORDER, V, true, EL>(g, cu, upd, ca, ls, os, cp, po, tab, has_cpml, q, true, true, s0, s0 + rm.lds);
    } else {
        const bool px = i >= rm.xlo && i <= rm.xhi, py = j0 >= rm.ylo && j0 + nj - 1 <= rm.yhi;
        thread_group<V / 2>(g, rm, rm.edge, i, j0, nj, q, row);
        float* s0 = sw + row * rm.edge.gpr * (V / 2);
        adj_group<ORDER, V / 2, false, EL>(g, cu, upd, ca, ls, os, cp, po, tab, has_cpml, q, px, py, s0, s0 + rm.lds);
    }
    if (!EL && rx.count > 0) {
        // receivers^T of the next (earlier) step on cells of this workgroup,
        // once it has stored them; coincident receivers add in index order
        const int blin = blockIdx.x + gridDim.x * blockIdx.y;
        const int b0 = rx.off[blin], b1 = rx.off[blin + 1];
        if (b0 == b1) return;
        __syncthreads();
        float* f = out.c[rx.comp] + so;
        for (int x = b0 + (int)threadIdx.x; x < b1; x += live) {
            const int4 grp = rx.grp[x];  // cell, first member, members
            float acc = f[grp.x];
            for (int y = grp.y; y < grp.y + grp.z; ++y)
                acc += rx.dgrad[((long long)blockIdx.y * rx.nt + rx.it) * rx.nrx + rx.member[y]];
            f[grp.x] = acc;
        }
    }
}

// The profiles by cell (axis_table): electric, then magnetic.
__global__ __launch_bounds__(256) void k_profile_tables(Grid g, Cpml cpe, Cpml cph, float* tab)
{
    const int a = blockIdx.y, n = g.N[a], c = (int)(blockIdx.x * 256 + threadIdx.x);
    if (c >= n) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const int q = f / 2 == a ? face_q(g, h == 0, f, c) : -1;
            if (q < 0) continue;
            const float* R = h == 0 ? cpe.coef[f] : cph.coef[f];
            const int pp = g.pml[f];
            v[0] = R[q] - 1.0f;
            v[1] = R[pp + q];
            v[2] = R[2 * pp + q];
            v[3] = R[3 * pp + q];
        }
        float* T = tab + h * 4 * (g.N[0] + g.N[1] + g.N[2]) + 4 * (a == 0 ? 0 : (a == 1 ? g.N[0] : g.N[0] + g.N[1]));
#pragma unroll
        for (int x = 0; x < 4; ++x) T[x * n + c] = v[x];
    }
}

__global__ __launch_bounds__(256) void k_copy_spans(CopySpans sp)
{
    const int q = blockIdx.y;
    for (long long n = (long long)blockIdx.x * 256 + threadIdx.x; n < sp.n[q]; n += (long long)gridDim.x * 256)
        sp.to[q][n] = sp.from[q][n];
}

// ---------------------------------------------------------------------------
// Launches
// ---------------------------------------------------------------------------
unsigned row_lds(const RowMap& rm) { return 2u * (unsigned)rm.lds * (unsigned)sizeof(float); }

}  // namespace

RowMap row_map(const Grid& g, int order)
{
    return make_row_map(g.N, g.pml, order / 2, kRowCells, kRowThreads);
}

void launch_copy_spans(const CopySpans& sp, hipStream_t st)
{
    if (sp.count > 0) hipLaunchKernelGGL(k_copy_spans, dim3(128, (unsigned)sp.count), dim3(256), 0, st, sp);
}

void launch_profile_tables(const Grid& g, const Cpml& cpe, const Cpml& cph, float* tab, hipStream_t st)
{
    const int n = std::max(g.N[0], std::max(g.N[1], g.N[2]));
    hipLaunchKernelGGL(k_profile_tables, dim3((unsigned)((n + 255) / 256), 3), dim3(256), 0, st, g, cpe, cph, tab);
}

void launch_row_fwd_h(int order, const Grid& g, const RowMap& rm, const StepArgs& a, hipStream_t st)
{
    const dim3 grid((unsigned)rm.total, (unsigned)g.nshot), block((unsigned)rm.threads);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, block, row_lds(rm), st, g, a.hcurl, a.hrhs, a.Ec, a.H, a.cph, a.tab_h, a.has_cpml, rm);
    };
    if (order == 4) go(k_row_fwd_h<4, kRowCells>);
    else go(k_row_fwd_h<2, kRowCells>);
}

void launch_row_fwd_e(int order, const Grid& g, const RowMap& rm, const StepArgs& a, const RowReceivers& rx,
                      hipStream_t st)
{
    const dim3 grid((unsigned)rm.total, (unsigned)g.nshot), block((unsigned)rm.threads);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, block, row_lds(rm), st, g, a.ca, a.ccurl, a.cb, a.Hc, a.E, a.cpe, a.tab_e, a.has_cpml,
                           a.src, a.hist, rx, rm);
    };
    if (order == 4) go(k_row_fwd_e<4, kRowCells>);
    else go(k_row_fwd_e<2, kRowCells>);
}

void launch_row_adj(int order, bool electric, const Grid& g, const RowMap& rm, const AdjArgs& a, const PsiOut& po,
                    const RowAdjReceivers& rx, hipStream_t st)
{
    const dim3 grid((unsigned)rm.total, (unsigned)g.nshot), block((unsigned)rm.threads);
    const unsigned lds = row_lds(rm);
    auto go = [&](auto kern_e, auto kern_h) {
        if (electric)
            hipLaunchKernelGGL(kern_e, grid, block, lds, st, g, a.ccurl, a.cb, a.ca, a.lE, a.lH, a.cpe, po, a.tab_e,
                               a.has_cpml, rx, rm);
        else
            hipLaunchKernelGGL(kern_h, grid, block, lds, st, g, a.hcurl, a.hrhs, a.ca, a.lH, a.lE, a.cph, po, a.tab_h,
                               a.has_cpml, rx, rm);
    };
    if (order == 4) go(k_row_adj<4, kRowCells, true>, k_row_adj<4, kRowCells, false>);
    else go(k_row_adj<2, kRowCells, true>, k_row_adj<2, kRowCells, false>);
}

}  // namespace dgx
