// Several 2D-TM time steps in one launch, forward and adjoint.
//
// A solve of a few shots is a chain of thousands of small launches, each of
// which loads a tile, takes one step and stores it: the step's time is launch
// and memory latency. Here a workgroup keeps a tile in registers for T steps: a
// wavefront holds KR rows, one lane a column, a row difference comes from the
// wavefront's own registers (and, at its first and last rows, from its
// neighbours through LDS), a column difference from the neighbouring lanes. The
// margin of the tile is advanced redundantly. Every value uses the expression
// of the one-step kernels (dgx_tm2d_fused.hip), so both give the same bits.
//
// What bounds it: instructions. A wavefront alone on its SIMD issues one in
// four cycles or more, so the steps of a small solve cost what one strip's
// instructions cost, and a solve that fills the chip pays them for the margin
// too. Hence: the grid spacings' quotients by a product and two fused
// multiply-adds (div_all), one branch a face kind for a whole strip, row
// conditions as bits of scalar masks, loads and stores from scalar bases with
// 32-bit offsets, arguments read again where they are used instead of kept in
// (spilled) scalar registers. The same kernel with a division per cell, a
// branch per row and face, and all arguments in registers took 18.8 us for one
// step of 121 x 121 (order 2, CPML 10) and 2.5 us for each further one; this
// one takes 7.0 and 1.2.
#include <algorithm>
#include <type_traits>

#include "dgx_device.h"
#include "dgx_internal.h"

namespace dgx {

namespace {

// The value of the next / previous lane (0 beyond the wavefront's ends; those
// columns are in the margin of the tile).
__device__ __forceinline__ float lane_next(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));  // wave_shl:1
}
__device__ __forceinline__ float lane_prev(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));  // wave_shr:1
}

struct Cpml4 {
    float ra1, rb, re, rf;
};

// The face of an axis on one side: its cells [lo, hi] (none: lo > hi), profile
// index hi - c or c - lo, profile and auxiliary arrays.
struct StripFace {
    bool high;
    int p, lo, hi;
    __device__ __forceinline__ bool in(int c) const { return c >= lo && c <= hi; }
    // a valid index for any c, the cell's own inside the face
    __device__ __forceinline__ int at(int c) const { return min(max(high ? c - lo : hi - c, 0), max(p - 1, 0)); }
};

template <typename T>
__device__ __forceinline__ T choose(bool c, T a, T b)
{
    return c ? a : b;
}

template <typename G>
__device__ __forceinline__ StripFace strip_face(const G& g, bool electric, int axis, bool high)
{
    StripFace o;
    const int n = axis == 0 ? g.NX : g.NY;
    o.high = high;
    o.p = g.has_cpml ? choose(high, g.pml[2 * axis + 1], g.pml[2 * axis]) : 0;
    o.lo = high ? n - 1 - o.p : (electric ? 1 : 0);
    o.hi = o.p > 0 ? (high ? n - 2 : (electric ? o.p : o.p - 1)) : -1;
    return o;
}

__device__ __forceinline__ Cpml4 cpml_profile(const float* R, int p, int q)
{
    return {R[q] - 1.0f, R[p + q], R[2 * p + q], R[3 * p + q]};
}

template <typename G>
__device__ __forceinline__ float axis_k(const G& g, float c1, int a)
{
    if (a == 0 || g.d[a] == g.d[0]) return c1;
    return c1 * g.d[0] / g.d[a];
}

// A row mask, hidden from the optimiser in every step: tests of its bits stay
// scalar tests of one register instead of dozens of conditions kept across the
// step loop.
__device__ __forceinline__ unsigned rows_now(unsigned m)
{
    asm volatile("" : "+s"(m));
    return m;
}
// the rows i0 .. i0 + kr - 1 that lie in [lo, hi]
__device__ __forceinline__ unsigned row_range(int i0, int kr, int lo, int hi)
{
    const int a = min(max(lo - i0, 0), kr), b = min(max(hi + 1 - i0, 0), kr);
    return (unsigned)__builtin_amdgcn_readfirstlane((int)(((1u << b) - 1u) & ~((1u << a) - 1u)));
}
__device__ __forceinline__ bool row_of(unsigned m, int q) { return (m >> q) & 1u; }

// The staggered difference from its tap differences d[r - 1] (r = 1 .. R);
// clamped: fitted radius 1.
template <int ORDER>
__device__ __forceinline__ float diff_taps(const float (&d)[Radius<ORDER>::value], bool clamped)
{
    if constexpr (ORDER <= 2) {
        return d[0];
    } else {
        static_assert(ORDER == 4, "radius 2");
        float acc = 0.0f;
        acc += stencil_c(2, 1) * d[0];
        acc += stencil_c(2, 2) * d[1];
        const float one = 0.0f + stencil_c(1, 1) * d[0];
        return clamped ? one : acc;
    }
}

// The transposed difference along a row: w holds UP rows (or columns) before
// the KR of this strip and DN after, c1 / c2 their weights in the differences
// that read them with one and two cells' reach (fitted radius: c2 = 0).
// acc += c1 w[first] - c1 w[second] (+ c2 w[first - 1] - c2 w[second + 1]).
template <int ORDER>
__device__ __forceinline__ float tap1(float w, bool clamped)
{
    if constexpr (ORDER <= 2) return w;
    return (clamped ? stencil_c(1, 1) : stencil_c(2, 1)) * w;
}
__device__ __forceinline__ float tap2(float w, bool clamped)
{
    const float t = stencil_c(2, 2) * w;
    return clamped ? 0.0f : t;
}

// A load or store from a wave-uniform base and a 32-bit byte offset a lane.
__device__ __forceinline__ float ld(const float* base, unsigned off)
{
    return *(const float*)((const char*)base + off);
}
__device__ __forceinline__ void put(float* base, unsigned off, float v)
{
    *(float*)((char*)base + off) = v;
}

// History elements: a wave-uniform frame and a 32-bit element index a lane.
template <int KIND>
__device__ __forceinline__ void put_hist(void* base, unsigned idx, float v)
{
    if constexpr (KIND == kF32) *(float*)((char*)base + 4u * idx) = v;
    else *(uint16_t*)((char*)base + 2u * idx) = KIND == kF16 ? f32_to_f16_bits(v) : f32_to_bf16_bits(v);
}
template <int KIND>
__device__ __forceinline__ float get_hist(const void* base, unsigned idx)
{
    if constexpr (KIND == kF32) return *(const float*)((const char*)base + 4u * idx);
    const uint16_t b = *(const uint16_t*)((const char*)base + 2u * idx);
    return KIND == kF16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b);
}
// f with the storage kind as a constant
template <typename F>
__device__ __forceinline__ void with_kind(int kind, F f)
{
    if (kind == kF32) f(std::integral_constant<int, kF32>());
    else if (kind == kF16) f(std::integral_constant<int, kF16>());
    else f(std::integral_constant<int, kBF16>());
}

template <int ORDER, int KR, int NW, int T>
struct Strip {
    static constexpr int R = Radius<ORDER>::value;
    static constexpr int H = T * (2 * R - 1);
    static constexpr int SR = KR * NW;
    static constexpr int OR = SR - 2 * H;
    static constexpr int OC = 64 - 2 * H;
    static_assert(OR > 0 && OC > 0 && KR >= R, "strip shape");
};

// Sources of a wavefront up to which it takes one after the other, with scalar
// loads (0.3 us a source and step). More are taken by the lanes that hold their
// cells, each finding its own by bisection: 20 x 20 sources on 200 x 200 (order 2,
// forward), 75 us a step one after the other, 7 this way. The branches that points
// need are laid out of the way of the other wavefronts (adjoint of 441 x 241 x 20
// shots, two steps: 70.6 and 69.0 us).
constexpr int kFewPoints = 4;

// The first of the wavefront's entries (in lane order) of this lane or a later one.
__device__ __forceinline__ int lane_first(const int2* ent, int beg, int end, int lane)
{
    while (beg < end) {
        const int mid = (beg + end) >> 1;
        if ((ent[mid].x & 63) < lane) beg = mid + 1;
        else end = mid;
    }
    return beg;
}

// f(row of the strip, point) for the entries [beg, end) of this wavefront on cells
// of this lane, in input order.
template <int KR, typename F>
__device__ __forceinline__ void lane_points(const int2* ent, int beg, int end, int w, int lane, F f)
{
    if (end - beg <= kFewPoints) {
        for (int x = beg; x < end; ++x) {
            const int2 e = ent[x];
            f((e.x & 63) == lane ? (e.x >> 6) - w * KR : -1, e.y);
        }
    } else {
        for (int x = lane_first(ent, beg, end, lane); x < end; ++x) {
            const int2 e = ent[x];
            if ((e.x & 63) != lane) break;
            f((e.x >> 6) - w * KR, e.y);
        }
    }
}

// Rows -(R - 1) .. KR + R - 1 (FWD) or -R .. KR + R - 2 of this wavefront's
// strip of v: the rows of its neighbours through LDS. Two barriers' worth of
// steps may be in flight, so forward and backward exchanges use separate
// buffers. first / last: the buffers' rows of every wavefront.
template <int KR, int NW, int UP, int DN>
__device__ __forceinline__ void exchange(const float (&v)[KR], float (*first)[DN > 0 ? DN : 1][64],
                                         float (*last)[UP > 0 ? UP : 1][64], int w, int lane,
                                         float (&out)[KR + UP + DN])
{
#pragma unroll
    for (int r = 0; r < DN; ++r) first[w][r][lane] = v[r];
#pragma unroll
    for (int r = 0; r < UP; ++r) last[w][r][lane] = v[KR - UP + r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < UP; ++r) out[r] = w > 0 ? last[w - 1][r][lane] : 0.0f;
#pragma unroll
    for (int r = 0; r < KR; ++r) out[UP + r] = v[r];
#pragma unroll
    for (int r = 0; r < DN; ++r) out[UP + KR + r] = w + 1 < NW ? first[w + 1][r][lane] : 0.0f;
}

}  // namespace

// ---------------------------------------------------------------------------
// Forward: nsub (at most T) steps from it0
// ---------------------------------------------------------------------------
// One barrier per half step (its first and last rows through LDS) and one more
// where the tile owns a receiver. A source is added by every wavefront that stages
// its cell, a receiver read by the tile that owns it.
// The arguments are read where they are used: what only the stores or a listed
// source need is not kept in scalar registers over the steps.
typedef const __attribute__((address_space(4))) StripArgs* StripArgsPtr;
typedef const __attribute__((address_space(4))) StripAdjArgs* StripAdjArgsPtr;
template <typename P>
__device__ __forceinline__ P again(P a)
{
    asm volatile("" : "+s"(a));
    return a;
}

// Tile (ti, tj) of shot s, steps it0 .. it0 + nsub - 1; frame: the first history
// frame not yet written; par: which copy of the state holds step it0.
template <int ORDER, int KR, int NW, int T>
__device__ __forceinline__ void strip_fwd(StripArgsPtr args, int ti, int tj, int s, int it0, int nsub, int frame,
                                          int par)
{
    const auto& g = args->g;
    const auto& f = args->f;
    const auto& pp = args->pp;
    const auto& sm = args->sm;
    const auto& hist = args->hist;
    const Spacing sx{args->sx.d, args->sx.y, args->sx.big}, sy{args->sy.d, args->sy.y, args->sy.big};
    using St = Strip<ORDER, KR, NW, T>;
    constexpr int R = St::R, H = St::H, SR = St::SR;
    const int tile = ti * sm.ntj + tj;
    __shared__ float e_first[NW][R][64], e_last[NW][R > 1 ? R - 1 : 1][64];
    __shared__ float h_first[NW][R > 1 ? R - 1 : 1][64], h_last[NW][R][64];
    __shared__ float s_cx[SR][8];  // x-face profiles of the rows: H, then E
    __shared__ float s_ez[SR * 64];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i0 = ti * St::OR - H + w * KR, gj = tj * St::OC - H + lane;  // first row of the strip, column
    const bool col = gj >= 0 && gj < g.NY;
    const bool col_in = gj > 0 && gj < g.NY - 1;
    const bool own_col = col && lane >= H && lane < 64 - H;
    const long long sb = (long long)s * g.plane;
    const int lt = tile + sm.tiles * s;

    const int cj = min(max(gj, 0), g.NY - 1);

    float ez[KR], hx[KR], hy[KR], ca[KR], cc[KR], cb[KR], hc[KR], hr[KR];
    float pxe[KR], pye[KR], pxh[KR], pyh[KR];
    const float *gez = pp.Ez[par] + sb, *ghx = pp.Hx[par] + sb, *ghy = pp.Hy[par] + sb;
#pragma unroll
    for (int q = 0; q < KR; ++q) {
        const unsigned p = 4u * (unsigned)(min(max(i0 + q, 0), g.NX - 1) * g.NY + cj);
        ez[q] = ld(gez, p);
        hx[q] = ld(ghx, p);
        hy[q] = ld(ghy, p);
        ca[q] = ld(f.ca, p);
        cc[q] = ld(f.ccurl, p);
        cb[q] = ld(f.cb, p);
        hc[q] = ld(f.hcurl, p);
        hr[q] = pxe[q] = pye[q] = pxh[q] = pyh[q] = 0.0f;
    }
    // Faces: those of y on this lane's side, those of x on the strip's side (a
    // strip reaches into one of the two, strip_applies). Loads are unconditional
    // where an address is valid (rows and columns outside the grid read its edge
    // and are never used), so that they are all in flight together.
    const bool yhigh = 2 * gj > g.NY, xhigh = 2 * i0 + KR > g.NX;
    const StripFace fyh = strip_face(g, false, 1, yhigh), fye = strip_face(g, true, 1, yhigh);
    const StripFace fxh = strip_face(g, false, 0, xhigh), fxe = strip_face(g, true, 0, xhigh);
    const bool yh = col && fyh.in(gj), ye = col && fye.in(gj);
    const bool any_yh = __any(yh), any_ye = __any(ye);
    const bool any_xh = row_range(i0, KR, fxh.lo, fxh.hi) != 0, any_xe = row_range(i0, KR, fxe.lo, fxe.hi) != 0;
    Cpml4 cyh{}, cye{};
    if (any_xh || any_yh) {
#pragma unroll
        for (int q = 0; q < KR; ++q) hr[q] = ld(f.hrhs, 4u * (unsigned)(min(max(i0 + q, 0), g.NX - 1) * g.NY + cj));
    }
    if (any_xh) {
        const float* psi = choose(xhigh, pp.psi_h[par][1], pp.psi_h[par][0]) + (long long)s * fxh.p * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q) pxh[q] = ld(psi, 4u * (unsigned)(fxh.at(i0 + q) * g.NY + cj));
    }
    if (any_xe) {
        const float* psi = choose(xhigh, pp.psi_e[par][1], pp.psi_e[par][0]) + (long long)s * (fxe.p + 1) * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q) pxe[q] = ld(psi, 4u * (unsigned)(fxe.at(i0 + q) * g.NY + cj));
    }
    if (yh) {
        const float* psi = choose(yhigh, pp.psi_h[par][3], pp.psi_h[par][2]) + (long long)s * g.NX * fyh.p + fyh.at(gj);
#pragma unroll
        for (int q = 0; q < KR; ++q) pyh[q] = psi[min(max(i0 + q, 0), g.NX - 1) * fyh.p];
        cyh = cpml_profile(choose(yhigh, f.coef_h[3], f.coef_h[2]), fyh.p, fyh.at(gj));
    }
    if (ye) {
        const int depth = fye.p + 1;
        const float* psi = choose(yhigh, pp.psi_e[par][3], pp.psi_e[par][2]) + (long long)s * g.NX * depth + fye.at(gj);
#pragma unroll
        for (int q = 0; q < KR; ++q) pye[q] = psi[min(max(i0 + q, 0), g.NX - 1) * depth];
        cye = cpml_profile(choose(yhigh, f.coef_e[3], f.coef_e[2]), fye.p, fye.at(gj));
    }
    if (lane < 2 * KR && (any_xh || any_xe)) {  // x profiles of the strip's rows, by the strip itself
        const int q = lane >> 1;
        const bool el = lane & 1;
        const StripFace& fc = el ? fxe : fxh;
        Cpml4 c{};
        if (fc.in(i0 + q))
            c = cpml_profile(el ? choose(xhigh, f.coef_e[1], f.coef_e[0]) : choose(xhigh, f.coef_h[1], f.coef_h[0]),
                             fc.p, fc.at(i0 + q));
        float* o = s_cx[w * KR + q] + (el ? 4 : 0);
        o[0] = c.ra1;
        o[1] = c.rb;
        o[2] = c.re;
        o[3] = c.rf;
    }
    int sbeg = 0, send = 0, rbeg = 0, rend = 0;
    if (args->src.count > 0) {
        sbeg = args->src.block_off[lt * NW + w];
        send = args->src.block_off[lt * NW + w + 1];
    }
    if (args->rx.count > 0) {
        rbeg = args->rx.off[lt];
        rend = args->rx.off[lt + 1];
    }
    // conditions of the strip's rows, one bit each
    const unsigned m_in = row_range(i0, KR, 1, g.NX - 2);  // Hx and Ez updated
    const unsigned m_hy = row_range(i0, KR, 0, g.NX - 2);
    const unsigned m_cf = ~row_range(i0, KR, R - 1, g.NX - 1 - R), m_cb = ~row_range(i0, KR, R, g.NX - R);
    const unsigned m_xh = row_range(i0, KR, fxh.lo, fxh.hi), m_xe = row_range(i0, KR, fxe.lo, fxe.hi);
    const unsigned m_own = row_range(i0, KR, ti * St::OR, min((ti + 1) * St::OR, g.NX) - 1);
    const unsigned m_box = m_own & row_range(i0, KR, hist.box.x0, hist.box.x0 + hist.box.nx - 1);
    const bool cf_col = fit_fwd_sel(gj, g.NY, R) < R, cb_col = fit_bwd_sel(gj, g.NY, R) < R;
    const bool hx_col = gj >= 0 && gj < g.NY - 1;
    const bool box_col = own_col && gj >= hist.box.y0 && gj < hist.box.y0 + hist.box.ny;
    const bool listed = rend > rbeg;
    const bool save = hist.on;
    int next = frame * hist.S;  // the next saved step
    for (int sub = 0; sub < nsub; ++sub) {
        const int it = it0 + sub;
        // magnetic half step
        {
            constexpr int UP = R - 1, DN = R;
            float e[KR + UP + DN];
            exchange<KR, NW, UP, DN>(ez, e_first, e_last, w, lane, e);
            const unsigned inr = rows_now(m_in), hyr = rows_now(m_hy), cf = rows_now(m_cf), xr = rows_now(m_xh);
            float dEx[KR], dEy[KR];
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                float dx[R], dy[R];
#pragma unroll
                for (int r = 1; r <= R; ++r) dx[r - 1] = e[UP + q + r] - e[UP + q - r + 1];
                float nx = ez[q], pv = ez[q];
#pragma unroll
                for (int r = 1; r <= R; ++r) {
                    nx = lane_next(nx);
                    dy[r - 1] = nx - pv;
                    if (r < R) pv = lane_prev(pv);
                }
                dEx[q] = diff_taps<ORDER>(dx, row_of(cf, q));
                dEy[q] = diff_taps<ORDER>(dy, cf_col);
                const float u1 = hc[q], uy = axis_k(g, u1, 1);
                // the derivatives along z are zero: - uz * 0 and + uz * 0
                const float ny = hy[q] + u1 * dEx[q], nh = hx[q] - uy * dEy[q] + 0.0f;
                hy[q] = row_of(hyr, q) && col_in ? ny : hy[q];
                hx[q] = row_of(inr, q) && hx_col ? nh : hx[q];
            }
            if (any_xh) {
                float der[KR];
                div_all<KR>(dEx, sx, der);
#pragma unroll
                for (int q = 0; q < KR; ++q)
                    if (row_of(xr, q)) {
                        const float* c = s_cx[w * KR + q];
                        hy[q] += hr[q] * (c[0] * der[q] + c[1] * pxh[q]);
                        pxh[q] = c[2] * pxh[q] - c[3] * der[q];
                    }
            }
            if (any_yh) {
                float der[KR];
                div_all<KR>(dEy, sy, der);
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    const float nh = hx[q] - hr[q] * (cyh.ra1 * der[q] + cyh.rb * pyh[q]);
                    hx[q] = yh ? nh : hx[q];
                    pyh[q] = cyh.re * pyh[q] - cyh.rf * der[q];
                }
            }
        }
        // electric half step
        {
            constexpr int UP = R, DN = R - 1;
            float h[KR + UP + DN], eold[KR];
            exchange<KR, NW, UP, DN>(hy, h_first, h_last, w, lane, h);
            if (listed) {
                if (sub > 0) {  // receivers of the step before: every row of s_ez is there since the first barrier
                    const auto& rx = again(args)->rx;
                    for (int x = rbeg + (int)threadIdx.x; x < rend; x += NW * 64) {
                        const int2 ent = rx.ent[x];
                        rx.out[((long long)s * rx.nt + it - 1) * rx.nrx + ent.y] = s_ez[ent.x];
                    }
                }
                __syncthreads();
            }
            const unsigned er = rows_now(m_in), cbk = rows_now(m_cb), xr = rows_now(m_xe);
            float dHx[KR], dHy[KR];
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                float dx[R], dy[R];
#pragma unroll
                for (int r = 1; r <= R; ++r) dx[r - 1] = h[UP + q + r - 1] - h[UP + q - r];
                float nx = hx[q], pv = hx[q];
#pragma unroll
                for (int r = 1; r <= R; ++r) {
                    pv = lane_prev(pv);
                    dy[r - 1] = nx - pv;
                    if (r < R) nx = lane_next(nx);
                }
                dHy[q] = diff_taps<ORDER>(dx, row_of(cbk, q));
                dHx[q] = diff_taps<ORDER>(dy, cb_col);
                const float u1 = cc[q], uy = axis_k(g, u1, 1);
                eold[q] = ez[q];
                const float ne = ca[q] * ez[q] + u1 * dHy[q] - uy * dHx[q];
                ez[q] = row_of(er, q) && col_in ? ne : ez[q];
            }
            if (any_xe) {
                float der[KR];
                div_all<KR>(dHy, sx, der);
#pragma unroll
                for (int q = 0; q < KR; ++q)
                    if (row_of(xr, q)) {
                        const float* c = s_cx[w * KR + q] + 4;
                        ez[q] += cb[q] * (c[0] * der[q] + c[1] * pxe[q]);
                        pxe[q] = c[2] * pxe[q] - c[3] * der[q];
                    }
            }
            if (any_ye) {
                float der[KR];
                div_all<KR>(dHx, sy, der);
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    const float ne = ez[q] - cb[q] * (cye.ra1 * der[q] + cye.rb * pye[q]);
                    ez[q] = ye ? ne : ez[q];
                    pye[q] = cye.re * pye[q] - cye.rf * der[q];
                }
            }
            if (__builtin_expect(send > sbeg, 0)) {
                const auto& src = again(args)->src;
                lane_points<KR>(src.entries, sbeg, send, w, lane, [&](int row, int point) {
                    const float scale = src.wave[(long long)point * src.nt + it] * src.dl / src.vol;
#pragma unroll
                    for (int q = 0; q < KR; ++q)
                        if (row == q) ez[q] -= cb[q] * scale;
                });
            }
            if (save && it == next) {
                const auto& hist = again(args)->hist;
                const unsigned br = rows_now(m_box), ur = rows_now(m_in);
                const int comps = hist.mode == 3 ? 3 : 1;
                const int ny = hist.box.ny;
                const unsigned at = (unsigned)((i0 - hist.box.x0) * ny + (gj - hist.box.y0));
                const long long f0 = (long long)frame * hist.snap + (long long)s * hist.box.cells;
                ++frame;
                next += hist.S;
                with_kind(hist.kind, [&](auto kind) {
                    constexpr int K = decltype(kind)::value;
                    constexpr int EB = K == kF32 ? 4 : 2;
                    char* eb = (char*)hist.e + f0 * EB;
                    char* rb = (char*)hist.r + f0 * EB;
                    if (box_col) {
#pragma unroll 1
                        for (int ci = 0; ci + 1 < comps; ++ci) {  // Ex and Ey are identically zero here
#pragma unroll
                            for (int q = 0; q < KR; ++q) {
                                if (!row_of(br, q)) continue;
                                if (hist.e) put_hist<K>(eb, at + q * ny, 0.0f);
                                if (hist.r) put_hist<K>(rb, at + q * ny, cb[q] == cb[q] ? 0.0f : cb[q]);
                            }
                            eb += hist.cstride * EB;
                            rb += hist.cstride * EB;
                        }
#pragma unroll
                        for (int q = 0; q < KR; ++q) {
                            if (!row_of(br, q)) continue;
                            if (hist.e) put_hist<K>(eb, at + q * ny, eold[q]);
                            if (hist.r) {
                                const float a = row_of(ur, q) && col_in ? ca[q] : 1.0f;
                                put_hist<K>(rb, at + q * ny, cb[q] != 0.0f ? (ez[q] - a * eold[q]) / cb[q] : 0.0f);
                            }
                        }
                    }
                });
            }
            if (listed)
#pragma unroll
                for (int q = 0; q < KR; ++q) s_ez[(w * KR + q) * 64 + lane] = ez[q];
        }
    }
    if (rend > rbeg) {
        __syncthreads();
        const auto& rx = again(args)->rx;
        for (int x = rbeg + (int)threadIdx.x; x < rend; x += NW * 64) {
            const int2 ent = rx.ent[x];
            rx.out[((long long)s * rx.nt + it0 + nsub - 1) * rx.nrx + ent.y] = s_ez[ent.x];
        }
    }
    // the addresses are formed again here, not kept in registers since the loads
    int ib = i0, jb = gj;
    asm volatile("" : "+s"(ib), "+v"(jb));
    if (!own_col) return;
    {
    const auto& pp = again(args)->pp;
    const auto& g = again(args)->g;
    float *oez = pp.Ez[par ^ 1] + sb, *ohx = pp.Hx[par ^ 1] + sb, *ohy = pp.Hy[par ^ 1] + sb;
#pragma unroll
    for (int q = 0; q < KR; ++q) {
        if (!row_of(m_own, q)) continue;
        const unsigned p = 4u * (unsigned)((ib + q) * g.NY + jb);
        put(oez, p, ez[q]);
        put(ohx, p, hx[q]);
        put(ohy, p, hy[q]);
    }
    if (any_xh) {
        float* psi = choose(xhigh, pp.psi_h[par ^ 1][1], pp.psi_h[par ^ 1][0]) + (long long)s * fxh.p * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own & m_xh, q)) put(psi, 4u * (unsigned)(fxh.at(ib + q) * g.NY + jb), pxh[q]);
    }
    if (any_xe) {
        float* psi = choose(xhigh, pp.psi_e[par ^ 1][1], pp.psi_e[par ^ 1][0]) + (long long)s * (fxe.p + 1) * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own & m_xe, q)) put(psi, 4u * (unsigned)(fxe.at(ib + q) * g.NY + jb), pxe[q]);
    }
    if (yh) {
        float* psi = choose(yhigh, pp.psi_h[par ^ 1][3], pp.psi_h[par ^ 1][2]) + (long long)s * g.NX * fyh.p + fyh.at(jb);
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own, q)) psi[(ib + q) * fyh.p] = pyh[q];
    }
    if (ye) {
        const int depth = fye.p + 1;
        float* psi = choose(yhigh, pp.psi_e[par ^ 1][3], pp.psi_e[par ^ 1][2]) + (long long)s * g.NX * depth + fye.at(jb);
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own, q)) psi[(ib + q) * depth] = pye[q];
    }
    }
}

template <int ORDER, int KR, int NW, int T>
__global__ __launch_bounds__(NW * 64) void k_tm_strip_fwd(StripArgs a)
{
    strip_fwd<ORDER, KR, NW, T>((StripArgsPtr)__builtin_amdgcn_kernarg_segment_ptr(), blockIdx.y, blockIdx.x,
                                blockIdx.z, a.it0, a.nsub, a.frame, 0);
}

// ---------------------------------------------------------------------------
// Adjoint: nsub (at most T) steps downwards from it0
// ---------------------------------------------------------------------------
// Bound as the forward kernel is; 128 registers a lane let two workgroups of 512
// threads share a compute unit, so what is read once a step (the factors of the
// material terms, the y profiles) lies in LDS: 137 and more registers and
// factors in them took 47 us for two steps of 342 x 264 x 5 shots (order 4, BF16
// history), 119 registers 36, and the larger tile of shape 2 22 us, against 44
// in the one-step kernel. 121 x 121, one shot, order 2, FP32 history: 21.5 us
// for 8 steps, one-step kernel 61.
// As the forward kernel, with the transposed half steps: lambda_E's channel
// weights are exchanged and gathered into lambda_H, then lambda_H's into
// lambda_E. Receivers are added by the wavefronts that stage their cells, each
// in its own rows of s_lz. The material terms of a saved step go to one buffer
// a saved step of the launch (summed over shots afterwards) or, with DIRECT (one
// shot), into the sums themselves, which the launch keeps in registers.
// LDS of one wavefront is read in the order it was written; this keeps the
// compiler to it where lanes read what other lanes wrote.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Tile (ti, tj) of shot s, steps it0 .. it0 - nsub + 1; ts: the newest saved
// step's frame.
// += in the cache, without waiting for the value: one rounded addition, in order
// with this thread's earlier ones to the same address.
__device__ __forceinline__ void add_owned(double* p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void add_owned(float* p, float v) { *p += v; }

template <int ORDER, int KR, int NW, int T, bool DIRECT, typename ACC>
__device__ __forceinline__ void strip_adj(StripAdjArgsPtr args, int ti, int tj, int s, int it0, int nsub, int ts,
                                          int par)
{
    using St = Strip<ORDER, KR, NW, T>;
    constexpr int R = St::R, H = St::H, SR = St::SR;
    const auto& g = args->g;
    const auto& f = args->f;
    const auto& pp = args->pp;
    const auto& sm = args->sm;
    const int tile = ti * sm.ntj + tj;
    __shared__ float e_first[NW][R][64], e_last[NW][R > 1 ? R - 1 : 1][64];
    __shared__ float h_first[NW][R > 1 ? R - 1 : 1][64], h_last[NW][R][64];
    __shared__ float s_cx[SR][8];  // x-face profiles of the rows: H, then E
    __shared__ float s_lz[SR * 64];
    __shared__ float4 s_cy[2][64];  // y-face profiles of the columns: H, then E
    __shared__ float4 s_mat[SR * 64];  // factors of the material terms (a cell's own thread writes and reads them)
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i0 = ti * St::OR - H + w * KR, gj = tj * St::OC - H + lane;  // first row of the strip, column
    const bool col = gj >= 0 && gj < g.NY;
    const bool col_in = gj > 0 && gj < g.NY - 1;
    const bool own_col = col && lane >= H && lane < 64 - H;
    const long long sb = (long long)s * g.plane;
    const int lt = tile + sm.tiles * s;

    const int cj = min(max(gj, 0), g.NY - 1);

    float lz[KR], lx[KR], ly[KR], ca[KR], cc[KR], cb[KR], hc[KR], hr[KR];
    float pxe[KR], pye[KR], pxh[KR], pyh[KR];
    const float *gez = pp.Ez[par] + sb, *ghx = pp.Hx[par] + sb, *ghy = pp.Hy[par] + sb;
#pragma unroll
    for (int q = 0; q < KR; ++q) {
        const unsigned p = 4u * (unsigned)(min(max(i0 + q, 0), g.NX - 1) * g.NY + cj);
        lz[q] = ld(gez, p);
        lx[q] = ld(ghx, p);
        ly[q] = ld(ghy, p);
        ca[q] = ld(f.ca, p);
        cc[q] = ld(f.ccurl, p);
        cb[q] = ld(f.cb, p);
        hc[q] = ld(f.hcurl, p);
        hr[q] = pxe[q] = pye[q] = pxh[q] = pyh[q] = 0.0f;
    }
    const bool yhigh = 2 * gj > g.NY, xhigh = 2 * i0 + KR > g.NX;
    const StripFace fyh = strip_face(g, false, 1, yhigh), fye = strip_face(g, true, 1, yhigh);
    const StripFace fxh = strip_face(g, false, 0, xhigh), fxe = strip_face(g, true, 0, xhigh);
    const bool yh = col && fyh.in(gj), ye = col && fye.in(gj);
    const bool any_yh = __any(yh), any_ye = __any(ye);
    const bool any_xh = row_range(i0, KR, fxh.lo, fxh.hi) != 0, any_xe = row_range(i0, KR, fxe.lo, fxe.hi) != 0;
    if (any_xh || any_yh) {
#pragma unroll
        for (int q = 0; q < KR; ++q) hr[q] = ld(f.hrhs, 4u * (unsigned)(min(max(i0 + q, 0), g.NX - 1) * g.NY + cj));
    }
    if (any_xh) {
        const float* psi = choose(xhigh, pp.psi_h[par][1], pp.psi_h[par][0]) + (long long)s * fxh.p * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q) pxh[q] = ld(psi, 4u * (unsigned)(fxh.at(i0 + q) * g.NY + cj));
    }
    if (any_xe) {
        const float* psi = choose(xhigh, pp.psi_e[par][1], pp.psi_e[par][0]) + (long long)s * (fxe.p + 1) * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q) pxe[q] = ld(psi, 4u * (unsigned)(fxe.at(i0 + q) * g.NY + cj));
    }
    if (yh) {
        const float* psi = choose(yhigh, pp.psi_h[par][3], pp.psi_h[par][2]) + (long long)s * g.NX * fyh.p + fyh.at(gj);
#pragma unroll
        for (int q = 0; q < KR; ++q) pyh[q] = psi[min(max(i0 + q, 0), g.NX - 1) * fyh.p];
        if (w == 0) {
            const Cpml4 c = cpml_profile(choose(yhigh, f.coef_h[3], f.coef_h[2]), fyh.p, fyh.at(gj));
            s_cy[0][lane] = make_float4(c.ra1, c.rb, c.re, c.rf);
        }
    }
    if (ye) {
        const int depth = fye.p + 1;
        const float* psi = choose(yhigh, pp.psi_e[par][3], pp.psi_e[par][2]) + (long long)s * g.NX * depth + fye.at(gj);
#pragma unroll
        for (int q = 0; q < KR; ++q) pye[q] = psi[min(max(i0 + q, 0), g.NX - 1) * depth];
        if (w == 0) {
            const Cpml4 c = cpml_profile(choose(yhigh, f.coef_e[3], f.coef_e[2]), fye.p, fye.at(gj));
            s_cy[1][lane] = make_float4(c.ra1, c.rb, c.re, c.rf);
        }
    }
    if (lane < 2 * KR && (any_xh || any_xe)) {  // x profiles of the strip's rows, by the strip itself
        const int q = lane >> 1;
        const bool el = lane & 1;
        const StripFace& fc = el ? fxe : fxh;
        Cpml4 c{};
        if (fc.in(i0 + q))
            c = cpml_profile(el ? choose(xhigh, f.coef_e[1], f.coef_e[0]) : choose(xhigh, f.coef_h[1], f.coef_h[0]),
                             fc.p, fc.at(i0 + q));
        float* o = s_cx[w * KR + q] + (el ? 4 : 0);
        o[0] = c.ra1;
        o[1] = c.rb;
        o[2] = c.re;
        o[3] = c.rf;
    }
    const float invx = args->inv[0], invy = args->inv[1];
    int sbeg = 0, send = 0, rbeg = 0, rend = 0;
    if (args->src.count > 0) {
        sbeg = args->src.block_off[lt * NW + w];
        send = args->src.block_off[lt * NW + w + 1];
    }
    if (args->rx.count > 0) {
        rbeg = args->rx.off[lt * NW + w];
        rend = args->rx.off[lt * NW + w + 1];
    }
    // the first 64 receiver cells of the wavefront: a lane's own one, its data a step ahead
    int4 mine = make_int4(-1, 0, 0, 0);
    int first = 0;
    float ahead = 0.0f;
    if (rbeg + lane < rend) {
        mine = args->rx.grp[rbeg + lane];
        first = args->rx.member[mine.y];
        ahead = args->rx.dgrad[((long long)s * args->rx.nt + it0) * args->rx.nrx + first];
    }
    const bool any_rx = rend > rbeg;

    // conditions of the strip's rows, one bit each; m_cb and m_cf start with the rows before it
    const unsigned m_in = row_range(i0, KR, 1, g.NX - 2);
    const unsigned m_hy = row_range(i0, KR, 0, g.NX - 2);
    const unsigned m_cb = ~row_range(i0 - (R - 1), KR + 2 * R - 1, R, g.NX - R);
    const unsigned m_cf = ~row_range(i0 - R, KR + 2 * R - 1, R - 1, g.NX - 1 - R);
    const unsigned m_xh = row_range(i0, KR, fxh.lo, fxh.hi), m_xe = row_range(i0, KR, fxe.lo, fxe.hi);
    const unsigned m_own = row_range(i0, KR, ti * St::OR, min((ti + 1) * St::OR, g.NX) - 1);
    const bool cf_col = fit_fwd_sel(gj, g.NY, R) < R, cb_col = fit_bwd_sel(gj, g.NY, R) < R;
    const bool hx_col = gj >= 0 && gj < g.NY - 1;

    // material terms: factors of each cell (none: all zero), the sums of one shot
    const auto& box = args->mg.box;
    const bool mat = args->mg.on;
    const unsigned m_box = mat ? m_own & row_range(i0, KR, box.x0, box.x0 + box.nx - 1) : 0u;
    const bool box_col = own_col && gj >= box.y0 && gj < box.y0 + box.ny;
    unsigned active = 0;
    // FP64 sums of four rows would be 16 registers: they are added in memory, by
    // the one thread that owns the cell
    constexpr bool ATOMIC = DIRECT && KR > 2 && sizeof(ACC) == 8, REGS = DIRECT && !ATOMIC;
    ACC ge[REGS ? KR : 1], gs[REGS ? KR : 1];
    const int S = args->mg.S;
    int next = mat ? ts * S : -1;
    if (mat) {
        const float dt = args->mg.dt;
#pragma unroll
        for (int q = 0; q < KR; ++q) {
            if (!row_of(m_box, q) || !box_col) continue;
            const int gi = i0 + q;
            const float sig = args->mg.sig[(long long)gi * g.NY * 2 + (long long)gj * 2];  // full-layout material index
            active |= sig <= kPecSigma ? 1u << q : 0u;
            s_mat[(w * KR + q) * 64 + lane] =
                make_float4(kEps0 * (1.0f - ca[q]) * cb[q] / dt, -kEps0 * cb[q] * cb[q] / dt,
                            -0.5f * (1.0f + ca[q]) * cb[q], -0.5f * cb[q] * cb[q]);
            if constexpr (REGS) {
                const long long o = (long long)gi * (g.NY - 1) + gj;
                ge[q] = args->mg.want_eps ? ((const ACC*)args->mg.geps)[o] : (ACC)0;
                gs[q] = args->mg.want_sig ? ((const ACC*)args->mg.gsig)[o] : (ACC)0;
            }
        }
    }

    __syncthreads();  // s_cy
    int slot = 0;
    for (int sub = 0; sub < nsub; ++sub) {
        const int it = it0 - sub;
        const bool save = it == next;
        float m_e[KR], m_s[KR];
        if (save && m_box) {
            const auto& mg = again(args)->mg;
            const int ny = mg.box.ny;
            const unsigned at = (unsigned)((i0 - mg.box.x0) * ny + (gj - mg.box.y0));
            const bool last = mg.e_only && ts + 1 >= mg.nt_saved;
            const void* sec = !mg.e_only || last ? mg.r : mg.e;
            const long long s0 = (long long)s * mg.box.cells;
            const long long e0 = (long long)ts * mg.snap + mg.eoff + s0;
            const long long s1 = s0 + (last ? mg.roff : (long long)(mg.e_only ? ts + 1 : ts) * mg.snap + mg.eoff);
            with_kind(mg.kind, [&](auto kind) {
                constexpr int K = decltype(kind)::value;
                constexpr int EB = K == kF32 ? 4 : 2;
                const char *eb = (const char*)mg.e + e0 * EB, *sb1 = (const char*)sec + s1 * EB;
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    m_e[q] = m_s[q] = 0.0f;
                    if (row_of(m_box, q) && box_col) {
                        m_e[q] = get_hist<K>(eb, at + q * ny);
                        m_s[q] = get_hist<K>(sb1, at + q * ny);
                    }
                }
            });
        }
        // receivers^T
        if (__builtin_expect(any_rx, 0)) {
            const auto& rx = again(args)->rx;
#pragma unroll
            for (int q = 0; q < KR; ++q) s_lz[(w * KR + q) * 64 + lane] = lz[q];
            wave_lds_order();
            const long long at = ((long long)s * rx.nt + it) * rx.nrx;
            if (mine.x >= 0) {
                float acc = s_lz[mine.x] + ahead;
                for (int m = 1; m < mine.z; ++m) acc += rx.dgrad[at + rx.member[mine.y + m]];
                s_lz[mine.x] = acc;
                if (sub + 1 < nsub) ahead = rx.dgrad[at - rx.nrx + first];
            }
            for (int x = rbeg + 64 + lane; x < rend; x += 64) {
                const int4 e = rx.grp[x];
                float acc = s_lz[e.x];
                for (int m = 0; m < e.z; ++m) acc += rx.dgrad[at + rx.member[e.y + m]];
                s_lz[e.x] = acc;
            }
            wave_lds_order();
#pragma unroll
            for (int q = 0; q < KR; ++q) lz[q] = s_lz[(w * KR + q) * 64 + lane];
        }
        // source^T: one value per (step, shot, source), summed over shots later
        if (__builtin_expect(send > sbeg, 0)) {
            const auto& a = *again(args);
            lane_points<KR>(a.src.entries, sbeg, send, w, lane, [&](int row, int point) {
#pragma unroll
                for (int q = 0; q < KR; ++q)
                    if (row == q)
                        a.mg.src_vals[((long long)it * a.g.nshot + s) * a.mg.nsrc + point] = -cb[q] * a.mg.geo * lz[q];
            });
        }
        // (electric half step)^T
        {
            constexpr int UP = R - 1, DN = R;
            const unsigned inr = rows_now(m_in), cbk = rows_now(m_cb), xr = rows_now(m_xe);
            float wx[KR], wy[KR];
#pragma unroll
            for (int q = 0; q < KR; ++q) wx[q] = wy[q] = 0.0f;
            if (any_xe) {
#pragma unroll
                for (int q = 0; q < KR; ++q)
                    if (row_of(xr, q)) {
                        const float* c = s_cx[w * KR + q] + 4;
                        wx[q] = (cb[q] * c[0] * lz[q] - c[3] * pxe[q]) * invx;
                        pxe[q] = cb[q] * c[1] * lz[q] + c[2] * pxe[q];
                    }
            }
            if (any_ye) {
                const float4 c = s_cy[1][lane];
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    const float t = (-cb[q] * c.x * lz[q] - c.w * pye[q]) * invy;
                    wy[q] = ye ? t : 0.0f;
                    pye[q] = -cb[q] * c.y * lz[q] + c.z * pye[q];
                }
            }
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                const bool up = row_of(inr, q) && col_in;
                const float u1 = cc[q], uy = axis_k(g, u1, 1);
                wx[q] = up ? wx[q] + u1 * lz[q] : wx[q];
                wy[q] = up ? wy[q] - uy * lz[q] : wy[q];
            }
            float e[KR + UP + DN];
            exchange<KR, NW, UP, DN>(wx, e_first, e_last, w, lane, e);
            float e1[KR + UP + DN], e2[R > 1 ? KR + UP + DN : 1];
#pragma unroll
            for (int q = 0; q < KR + UP + DN; ++q) {
                e1[q] = tap1<ORDER>(e[q], row_of(cbk, q));
                if constexpr (R > 1) e2[q] = tap2(e[q], row_of(cbk, q));
            }
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                float acc = 0.0f + e1[UP + q] - e1[UP + q + 1];
                if constexpr (R > 1) {
                    acc += e2[UP + q - 1];
                    acc -= e2[UP + q + 2];
                }
                ly[q] = (ly[q] + acc) + 0.0f;
                const float y1 = tap1<ORDER>(wy[q], cb_col);
                acc = 0.0f + y1 - lane_next(y1);
                if constexpr (R > 1) {
                    const float y2 = tap2(wy[q], cb_col);
                    acc += lane_prev(y2);
                    acc -= lane_next(lane_next(y2));
                }
                lx[q] = (lx[q] + acc) + 0.0f;
            }
        }
        // (magnetic half step)^T
        {
            constexpr int UP = R, DN = R - 1;
            const unsigned inr = rows_now(m_in), hyr = rows_now(m_hy), cf = rows_now(m_cf), xr = rows_now(m_xh);
            float vx[KR], vy[KR];
#pragma unroll
            for (int q = 0; q < KR; ++q) vx[q] = vy[q] = 0.0f;
            if (any_xh) {
#pragma unroll
                for (int q = 0; q < KR; ++q)
                    if (row_of(xr, q)) {
                        const float* c = s_cx[w * KR + q];
                        vx[q] = (hr[q] * c[0] * ly[q] - c[3] * pxh[q]) * invx;
                        pxh[q] = hr[q] * c[1] * ly[q] + c[2] * pxh[q];
                    }
            }
            if (any_yh) {
                const float4 c = s_cy[0][lane];
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    const float t = (-hr[q] * c.x * lx[q] - c.w * pyh[q]) * invy;
                    vy[q] = yh ? t : 0.0f;
                    pyh[q] = -hr[q] * c.y * lx[q] + c.z * pyh[q];
                }
            }
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                const float u1 = hc[q], uy = axis_k(g, u1, 1);
                vx[q] = row_of(hyr, q) && col_in ? vx[q] + u1 * ly[q] : vx[q];
                vy[q] = row_of(inr, q) && hx_col ? vy[q] - uy * lx[q] : vy[q];
            }
            float h[KR + UP + DN];
            exchange<KR, NW, UP, DN>(vx, h_first, h_last, w, lane, h);
            // the material terms here: the history's loads had the half steps to arrive
            if (save && m_box) {
                const auto& mg = again(args)->mg;
                const float wgt = (float)min(S, mg.nt - it);
                const int ny = mg.box.ny;
                const unsigned at = 4u * (unsigned)((i0 - mg.box.x0) * ny + (gj - mg.box.y0));
                float* te = nullptr;  // this shot's eps and sigma terms
                float* ts1 = nullptr;
                if constexpr (!DIRECT) {
                    te = mg.terms + (long long)slot * mg.terms_len + (long long)s * mg.box.cells;
                    ts1 = te + (long long)g.nshot * mg.box.cells;
                }
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    if (!row_of(m_box, q) || !box_col) continue;
                    const bool up = row_of(inr, q) && col_in;
                    float l = lz[q], rhs = m_s[q];
                    if (mg.e_only) {
                        const float a = up ? ca[q] : 1.0f;
                        rhs = cb[q] != 0.0f ? (m_s[q] - a * m_e[q]) / cb[q] : 0.0f;
                    }
                    if (m_e[q] == 0.0f && rhs == 0.0f) l = 0.0f;
                    const float gca = up ? l * m_e[q] * wgt : 0.0f;
                    const float gcb = l * rhs * wgt;
                    const bool on = (active >> q) & 1u;
                    const long long o = (long long)(i0 + q) * (g.NY - 1) + gj;
                    const float4 d = s_mat[(w * KR + q) * 64 + lane];
                    if (mg.want_eps) {
                        const float t = on ? gca * d.x + gcb * d.y : 0.0f;
                        if constexpr (REGS) ge[q] += (ACC)0 + (ACC)t;
                        else if constexpr (ATOMIC) add_owned((ACC*)mg.geps + o, (ACC)0 + (ACC)t);
                        else put(te, at + 4u * (unsigned)(q * ny), t);
                    }
                    if (mg.want_sig) {
                        const float t = on ? gca * d.z + gcb * d.w : 0.0f;
                        if constexpr (REGS) gs[q] += (ACC)0 + (ACC)t;
                        else if constexpr (ATOMIC) add_owned((ACC*)mg.gsig + o, (ACC)0 + (ACC)t);
                        else put(ts1, at + 4u * (unsigned)(q * ny), t);
                    }
                }
            }
            if (save) {
                ++slot;
                --ts;
                next -= S;
            }
            float h1[KR + UP + DN], h2[R > 1 ? KR + UP + DN : 1];
#pragma unroll
            for (int q = 0; q < KR + UP + DN; ++q) {
                h1[q] = tap1<ORDER>(h[q], row_of(cf, q));
                if constexpr (R > 1) h2[q] = tap2(h[q], row_of(cf, q));
            }
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                const float scaled = ca[q] * lz[q];
                float acc = row_of(inr, q) && col_in ? scaled : lz[q];
                float gx = 0.0f + h1[UP + q - 1] - h1[UP + q];
                if constexpr (R > 1) {
                    gx += h2[UP + q - 2];
                    gx -= h2[UP + q + 1];
                }
                acc += gx;
                const float y1 = tap1<ORDER>(vy[q], cf_col);
                float gy = 0.0f + lane_prev(y1) - y1;
                if constexpr (R > 1) {
                    const float y2 = tap2(vy[q], cf_col);
                    gy += lane_prev(lane_prev(y2));
                    gy -= lane_next(y2);
                }
                lz[q] = acc + gy;
            }
        }
    }
    // the addresses are formed again here, not kept in registers since the loads
    int ib = i0, jb = gj;
    asm volatile("" : "+s"(ib), "+v"(jb));
    if (!own_col) return;
    {
        const auto& pp = again(args)->pp;
        const auto& g = again(args)->g;
        float *oez = pp.Ez[par ^ 1] + sb, *ohx = pp.Hx[par ^ 1] + sb, *ohy = pp.Hy[par ^ 1] + sb;
#pragma unroll
        for (int q = 0; q < KR; ++q) {
            if (!row_of(m_own, q)) continue;
            const unsigned p = 4u * (unsigned)((ib + q) * g.NY + jb);
            put(oez, p, lz[q]);
            put(ohx, p, lx[q]);
            put(ohy, p, ly[q]);
        }
        if constexpr (REGS) {
            const auto& mg = again(args)->mg;
            if (box_col) {
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    if (!row_of(m_box, q)) continue;
                    const long long o = (long long)(ib + q) * (g.NY - 1) + jb;
                    if (mg.want_eps) ((ACC*)mg.geps)[o] = ge[q];
                    if (mg.want_sig) ((ACC*)mg.gsig)[o] = gs[q];
                }
            }
        }
        if (any_xh) {
            float* psi = choose(xhigh, pp.psi_h[par ^ 1][1], pp.psi_h[par ^ 1][0]) + (long long)s * fxh.p * g.NY;
#pragma unroll
            for (int q = 0; q < KR; ++q)
                if (row_of(m_own & m_xh, q)) put(psi, 4u * (unsigned)(fxh.at(ib + q) * g.NY + jb), pxh[q]);
        }
        if (any_xe) {
            float* psi = choose(xhigh, pp.psi_e[par ^ 1][1], pp.psi_e[par ^ 1][0]) + (long long)s * (fxe.p + 1) * g.NY;
#pragma unroll
            for (int q = 0; q < KR; ++q)
                if (row_of(m_own & m_xe, q)) put(psi, 4u * (unsigned)(fxe.at(ib + q) * g.NY + jb), pxe[q]);
        }
        if (yh) {
            float* psi = choose(yhigh, pp.psi_h[par ^ 1][3], pp.psi_h[par ^ 1][2]) + (long long)s * g.NX * fyh.p + fyh.at(jb);
#pragma unroll
            for (int q = 0; q < KR; ++q)
                if (row_of(m_own, q)) psi[(ib + q) * fyh.p] = pyh[q];
        }
        if (ye) {
            const int depth = fye.p + 1;
            float* psi = choose(yhigh, pp.psi_e[par ^ 1][3], pp.psi_e[par ^ 1][2]) + (long long)s * g.NX * depth + fye.at(jb);
#pragma unroll
            for (int q = 0; q < KR; ++q)
                if (row_of(m_own, q)) psi[(ib + q) * depth] = pye[q];
        }
    }
}

template <int ORDER, int KR, int NW, int T, bool DIRECT, typename ACC>
__global__ __launch_bounds__(NW * 64, 4) void k_tm_strip_adj(StripAdjArgs a)
{
    strip_adj<ORDER, KR, NW, T, DIRECT, ACC>((StripAdjArgsPtr)__builtin_amdgcn_kernarg_segment_ptr(), blockIdx.y,
                                             blockIdx.x, blockIdx.z, a.it0, a.nsub, a.frame, 0);
}

// ---------------------------------------------------------------------------
// Launches
// ---------------------------------------------------------------------------
namespace {
// KR x NW rows and T steps of each shape. A forward launch costs 5.4 us before
// its first step and 1.1 us (order 2, KR = 2) to 2 us (order 4, KR = 4) a step,
// so a small solve takes few rows a wavefront, 16 wavefronts and many steps; one
// that fills the chip is bound by the instructions of its wavefronts, the
// margin's included, and takes more rows and, at order 4 (margin 3 a step),
// fewer steps. Measured forward step times without a history, in us, of the
// shape 0 / 1 / 2 against the one-step kernel:
//   121 x 121 order 2, CPML 10    1 shot   1.8 / 2.4 / -      5.0
//   121 x 121 order 4, CPML 10    1 shot   3.3 / 4.8 / -      5.8
//   121 x 121 order 2             8 shots  2.0 / 2.5 / -
//   121 x 121 order 2            14 shots  3.2 / 2.9 / -
//   342 x 264 order 4, CPML 20    2 shots  -   / 5.0 / 5.7    9.7
//   342 x 264 order 4, CPML 20    5 shots  -   / 8.4 / 6.5   14.4
//   342 x 264 order 2, CPML 20    5 shots  -   / 4.1 / 2.9   11.9
//   441 x 241 order 4, CPML 20   20 shots  -   / 20.0 / 19.5 34.9
//   441 x 241 order 2, CPML 20   20 shots  18  / 9.0 / 8.8   29.7
// Other step counts for the last rows: order 4 with 3 steps 20.4, order 2 with
// 4 or 8 steps 10.4 and 11.5.
// Hence the rule of map_order: shape 0 as long as each of its workgroups (1024
// threads) has a compute unit to itself, shape 1 as long as its workgroups (512
// threads, two a compute unit) are all resident at once, then shape 2, whose
// larger tile has the smaller margin. Before them comes shape 3, which is shape 0
// with more steps a launch and a margin that leaves 8 rows of 32: where its
// workgroups have a compute unit each as well, the margin costs no time and the
// launches are fewer. 600 steps, forward and gradient in ms, one shot, shape 0
// and shape 3: order 2, 121 x 121, 2.01 and 4.30 against 1.87 and 3.99; order 4,
// 3.01 and 6.47 against 2.85 and 5.89; 221 x 221, order 2, 2.05 and 4.48 against
// 1.98 and 4.15, order 4, 3.06 and 6.62 against 2.80 and 5.99. 10 steps at order 2:
// 1.93 and 4.15.
template <int ORDER, int SIZE>
struct Shapes;
template <>
struct Shapes<2, 0> {
    static constexpr int KR = 2, NW = 16, T = 8;
};
template <>
struct Shapes<2, 1> {
    static constexpr int KR = 4, NW = 8, T = 6;
};
template <>
struct Shapes<2, 2> {
    static constexpr int KR = 4, NW = 16, T = 6;
};
template <>
struct Shapes<4, 0> {
    static constexpr int KR = 2, NW = 16, T = 3;
};
template <>
struct Shapes<4, 1> {
    static constexpr int KR = 4, NW = 8, T = 2;
};
template <>
struct Shapes<4, 2> {
    static constexpr int KR = 4, NW = 16, T = 2;
};
template <>
struct Shapes<2, 3> {
    static constexpr int KR = 2, NW = 16, T = 12;
};
template <>
struct Shapes<4, 3> {
    static constexpr int KR = 2, NW = 16, T = 4;
};
template <int ORDER, int SIZE>
StripShape shape_of()
{
    using P = Shapes<ORDER, SIZE>;
    return {SIZE, P::KR * P::NW, P::T * (2 * Radius<ORDER>::value - 1), P::T, P::NW};
}
template <int ORDER, int SIZE>
void launch_shape(const dim3& grid, const StripArgs& a, hipStream_t st)
{
    using P = Shapes<ORDER, SIZE>;
    hipLaunchKernelGGL((k_tm_strip_fwd<ORDER, P::KR, P::NW, P::T>), grid, dim3(P::NW * 64), 0, st, a);
}
template <int ORDER>
void launch_order(const dim3& grid, const StripArgs& a, hipStream_t st)
{
    if (a.sm.sh.size == 0) launch_shape<ORDER, 0>(grid, a, st);
    else if (a.sm.sh.size == 1) launch_shape<ORDER, 1>(grid, a, st);
    else if (a.sm.sh.size == 2) launch_shape<ORDER, 2>(grid, a, st);
    else launch_shape<ORDER, 3>(grid, a, st);
}
template <int ORDER>
StripMap map_order(const Tm2dGrid& g)
{
    const StripMap deep = make_strip_map(shape_of<ORDER, 3>(), g.NX, g.NY);
    if ((long long)deep.tiles * g.nshot <= 256) return deep;
    const StripMap small = make_strip_map(shape_of<ORDER, 0>(), g.NX, g.NY);
    if ((long long)small.tiles * g.nshot <= 256) return small;
    const StripMap mid = make_strip_map(shape_of<ORDER, 1>(), g.NX, g.NY);
    if ((long long)mid.tiles * g.nshot <= 512) return mid;
    return make_strip_map(shape_of<ORDER, 2>(), g.NX, g.NY);
}
}  // namespace

bool strip_applies(int order, const Tm2dGrid& g)
{
    // 32-bit byte offsets, and tiles along x and shots within a launch's 65535
    if (order > 4 || g.plane >= 1 << 30 || g.NX > 1 << 20 || g.nshot > 65535) return false;
    // no face reaches the middle of its axis, and no strip of rows both faces
    return g.NX - g.pml[0] - g.pml[1] >= 12 && g.NY - g.pml[2] - g.pml[3] >= 4 && 2 * g.pml[0] + 9 < g.NX &&
           2 * g.pml[1] + 9 < g.NX && 2 * g.pml[2] + 2 < g.NY && 2 * g.pml[3] + 2 < g.NY;
}

StripMap strip_map(int order, const Tm2dGrid& g) { return order == 4 ? map_order<4>(g) : map_order<2>(g); }

void launch_tm_strip_fwd(int order, const Tm2dGrid& g, const Tm2dFields& f, const TmPingPong& pp, const StripMap& sm,
                         const SourceBlocks& src, const TmReceiversFwd& rx, const StripHist& hist, int it0, int nsub,
                         hipStream_t st)
{
    const dim3 grid((unsigned)sm.ntj, (unsigned)sm.nti, (unsigned)g.nshot);
    const StripArgs a{g, f, pp, sm, src, rx, hist, make_spacing(g.d[0]), make_spacing(g.d[1]), it0, nsub,
                       (it0 + hist.S - 1) / std::max(hist.S, 1)};
    order == 4 ? launch_order<4>(grid, a, st) : launch_order<2>(grid, a, st);
}

namespace {
template <int ORDER, int SIZE>
void launch_adj_shape(const dim3& grid, const StripAdjArgs& a, bool fp64, hipStream_t st)
{
    using P = Shapes<ORDER, SIZE>;
    constexpr int KR = P::KR, NW = P::NW, T = P::T;
    const dim3 block(NW * 64);
    const bool direct = a.mg.on && a.g.nshot == 1;
    if (!direct) hipLaunchKernelGGL((k_tm_strip_adj<ORDER, KR, NW, T, false, float>), grid, block, 0, st, a);
    else if (fp64) hipLaunchKernelGGL((k_tm_strip_adj<ORDER, KR, NW, T, true, double>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_tm_strip_adj<ORDER, KR, NW, T, true, float>), grid, block, 0, st, a);
}
template <int ORDER>
void launch_adj_order(const dim3& grid, const StripAdjArgs& a, bool fp64, hipStream_t st)
{
    if (a.sm.sh.size == 0) launch_adj_shape<ORDER, 0>(grid, a, fp64, st);
    else if (a.sm.sh.size == 1) launch_adj_shape<ORDER, 1>(grid, a, fp64, st);
    else if (a.sm.sh.size == 2) launch_adj_shape<ORDER, 2>(grid, a, fp64, st);
    else launch_adj_shape<ORDER, 3>(grid, a, fp64, st);
}
}  // namespace

void launch_tm_strip_adj(int order, const Tm2dGrid& g, const Tm2dFields& f, const TmPingPong& pp, const StripMap& sm,
                         const SourceBlocks& src, const TmReceiversAdj& rx, const StripGrad& mg, int it0, int nsub,
                         bool fp64, hipStream_t st)
{
    const dim3 grid((unsigned)sm.ntj, (unsigned)sm.nti, (unsigned)g.nshot);
    const StripAdjArgs a{g, f, pp, sm, src, rx, mg, {1.0f / g.d[0], 1.0f / g.d[1]}, it0, nsub,
                          it0 / std::max(mg.S, 1)};
    order == 4 ? launch_adj_order<4>(grid, a, fp64, st) : launch_adj_order<2>(grid, a, fp64, st);
}

// ---------------------------------------------------------------------------
// Batches: one launch advances every one-shot instance of one order and phase
// ---------------------------------------------------------------------------
// A batch fills the chip with its instances, so they take shape 2. Twelve
// gradients of 148 to 404 cells a side, orders 2 and 4 by halves: a step of the
// one-step kernels takes 12 (forward) and 24 us (adjoint) at order 4, 10 and 21
// at order 2, one launch after the other; these take 15.7 us for 2 steps of both
// phases at order 4 and 27 for 6 at order 2. With a launch a phase each took
// 14 to 16 and 23 to 27.
namespace {
template <int ORDER>
using BatchShape = Shapes<ORDER, 2>;

// Instance of workgroup b by bisection of the prefix sums; b becomes its tile.
__device__ __forceinline__ int batch_instance(const int* __restrict__ prefix, int ninst, int& b)
{
    int lo = 0, hi = ninst - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (prefix[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    const int k = __builtin_amdgcn_readfirstlane(lo);
    b = __builtin_amdgcn_readfirstlane(b - prefix[k]);
    return k;
}

// Both phases in one launch, adjoint workgroups (the longer ones) first:
// apart, each left half of the compute units idle.
template <int ORDER>
__global__ __launch_bounds__(BatchShape<ORDER>::NW * 64, 4) void k_tm_strip_batch(StripBatchSlot fwd,
                                                                                  StripBatchSlot adj, int gstep,
                                                                                  int launch, int nsub)
{
    using P = BatchShape<ORDER>;
    // XCD x takes the x-th contiguous chunk of workgroups
    int b = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    if (b < adj.total) {
        const int k = batch_instance(adj.prefix, adj.ninst, b);
        const StripBatchInst& I = adj.insts[k];
        const int ti = b / I.adj.sm.ntj, it0 = I.nt - 1 - (gstep - I.start);
        strip_adj<ORDER, P::KR, P::NW, P::T, true, double>((StripAdjArgsPtr)&I.adj, ti, b - ti * I.adj.sm.ntj, 0, it0,
                                                           nsub, it0, (launch - I.launch) & 1);
    } else {
        b -= adj.total;
        if (b >= fwd.total) return;
        const int k = batch_instance(fwd.prefix, fwd.ninst, b);
        const StripBatchInst& I = fwd.insts[k];
        const int ti = b / I.fwd.sm.ntj, it0 = gstep - I.start;
        strip_fwd<ORDER, P::KR, P::NW, P::T>((StripArgsPtr)&I.fwd, ti, b - ti * I.fwd.sm.ntj, 0, it0, nsub, it0,
                                             (launch - I.launch) & 1);
    }
}
}  // namespace

StripMap strip_batch_map(int order, const Tm2dGrid& g)
{
    return make_strip_map(order == 4 ? shape_of<4, 2>() : shape_of<2, 2>(), g.NX, g.NY);
}

int strip_batch_steps(int order) { return order == 4 ? BatchShape<4>::T : BatchShape<2>::T; }

void launch_tm_strip_batch(int order, const StripBatchSlot& fwd, const StripBatchSlot& adj, int gstep, int launch,
                           int nsub, hipStream_t st)
{
    const int total = fwd.total + adj.total;
    if (total <= 0) return;
    const dim3 grid((unsigned)((total + 7) / 8 * 8));
    if (order == 4)
        hipLaunchKernelGGL(k_tm_strip_batch<4>, grid, dim3(BatchShape<4>::NW * 64), 0, st, fwd, adj, gstep, launch,
                           nsub);
    else
        hipLaunchKernelGGL(k_tm_strip_batch<2>, grid, dim3(BatchShape<2>::NW * 64), 0, st, fwd, adj, gstep, launch,
                           nsub);
}

}  // namespace dgx
