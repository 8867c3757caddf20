// Several 2D-TM time steps in one launch.
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

__device__ __forceinline__ StripFace strip_face(const Tm2dGrid& g, bool electric, int axis, bool high)
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

__device__ __forceinline__ float axis_k(const Tm2dGrid& g, float c1, int a)
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

// A load or store from a wave-uniform base and a 32-bit byte offset a lane.
__device__ __forceinline__ float ld(const float* base, unsigned off)
{
    return *(const float*)((const char*)base + off);
}
__device__ __forceinline__ void put(float* base, unsigned off, float v)
{
    *(float*)((char*)base + off) = v;
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
// where the tile owns a receiver. A source is added by every tile that stages
// its cell, a receiver read by the tile that owns it.
struct StripArgs {
    Tm2dGrid g;
    Tm2dFields f;
    TmPingPong pp;
    StripMap sm;
    SourceBlocks src;
    TmReceiversFwd rx;
    StripHist hist;
    Spacing sx, sy;
    int it0, nsub;
};

// The kernel's arguments, read where they are used: what only the stores or a
// listed source need is not kept in scalar registers over the steps.
typedef const __attribute__((address_space(4))) StripArgs* StripArgsPtr;
__device__ __forceinline__ StripArgsPtr args_now()
{
    StripArgsPtr a = (StripArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return a;
}

template <int ORDER, int KR, int NW, int T>
__global__ __launch_bounds__(NW * 64) void k_tm_strip_fwd(StripArgs args)
{
    const Tm2dGrid& g = args.g;
    const Tm2dFields& f = args.f;
    const TmPingPong& pp = args.pp;
    const StripMap& sm = args.sm;
    const StripHist& hist = args.hist;
    const Spacing &sx = args.sx, &sy = args.sy;
    const int it0 = args.it0, nsub = args.nsub;
    using St = Strip<ORDER, KR, NW, T>;
    constexpr int R = St::R, H = St::H, SR = St::SR;
    const int tile = blockIdx.x;
    const int s = blockIdx.y;
    __shared__ float e_first[NW][R][64], e_last[NW][R > 1 ? R - 1 : 1][64];
    __shared__ float h_first[NW][R > 1 ? R - 1 : 1][64], h_last[NW][R][64];
    __shared__ float s_cx[SR][8];  // x-face profiles of the rows: H, then E
    __shared__ float s_ez[SR * 64];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int ti = tile / sm.ntj, tj = tile - ti * sm.ntj;
    const int i0 = ti * St::OR - H + w * KR, gj = tj * St::OC - H + lane;  // first row of the strip, column
    const bool col = gj >= 0 && gj < g.NY;
    const bool col_in = gj > 0 && gj < g.NY - 1;
    const bool own_col = col && lane >= H && lane < 64 - H;
    const long long sb = (long long)s * g.plane;
    const int lt = tile + sm.tiles * s;

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
    const int cj = min(max(gj, 0), g.NY - 1);

    float ez[KR], hx[KR], hy[KR], ca[KR], cc[KR], cb[KR], hc[KR], hr[KR];
    float pxe[KR], pye[KR], pxh[KR], pyh[KR];
    const float *gez = pp.Ez[0] + sb, *ghx = pp.Hx[0] + sb, *ghy = pp.Hy[0] + sb;
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
    Cpml4 cyh{}, cye{};
    if (any_xh || any_yh) {
#pragma unroll
        for (int q = 0; q < KR; ++q) hr[q] = ld(f.hrhs, 4u * (unsigned)(min(max(i0 + q, 0), g.NX - 1) * g.NY + cj));
    }
    if (any_xh) {
        const float* psi = choose(xhigh, pp.psi_h[0][1], pp.psi_h[0][0]) + (long long)s * fxh.p * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q) pxh[q] = ld(psi, 4u * (unsigned)(fxh.at(i0 + q) * g.NY + cj));
    }
    if (any_xe) {
        const float* psi = choose(xhigh, pp.psi_e[0][1], pp.psi_e[0][0]) + (long long)s * (fxe.p + 1) * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q) pxe[q] = ld(psi, 4u * (unsigned)(fxe.at(i0 + q) * g.NY + cj));
    }
    if (yh) {
        const float* psi = choose(yhigh, pp.psi_h[0][3], pp.psi_h[0][2]) + (long long)s * g.NX * fyh.p + fyh.at(gj);
#pragma unroll
        for (int q = 0; q < KR; ++q) pyh[q] = psi[min(max(i0 + q, 0), g.NX - 1) * fyh.p];
        cyh = cpml_profile(choose(yhigh, f.coef_h[3], f.coef_h[2]), fyh.p, fyh.at(gj));
    }
    if (ye) {
        const int depth = fye.p + 1;
        const float* psi = choose(yhigh, pp.psi_e[0][3], pp.psi_e[0][2]) + (long long)s * g.NX * depth + fye.at(gj);
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
    if (args.src.count > 0) {
        sbeg = args.src.block_off[lt];
        send = args.src.block_off[lt + 1];
    }
    if (args.rx.count > 0) {
        rbeg = args.rx.off[lt];
        rend = args.rx.off[lt + 1];
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
    int frame = it0 / hist.S, next = frame * hist.S;  // the next saved step
    if (next < it0) {
        ++frame;
        next += hist.S;
    }
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
                    const auto& rx = args_now()->rx;
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
            for (int x = sbeg; x < send; ++x) {
                const auto& src = args_now()->src;
                const int2 ent = src.entries[x];
                const int row = ent.x >> 6;
                if (row / KR != w) continue;
                const float scale = src.wave[(long long)ent.y * src.nt + it] * src.dl / src.vol;
#pragma unroll
                for (int q = 0; q < KR; ++q)
                    if (row - w * KR == q && (ent.x & 63) == lane) ez[q] -= cb[q] * scale;
            }
            if (save && it == next) {
                const auto& hist = args_now()->hist;
                long long at = (long long)frame * hist.snap + (long long)s * hist.box.cells +
                               (long long)(i0 - hist.box.x0) * hist.box.ny + (gj - hist.box.y0);
                ++frame;
                next += hist.S;
                const unsigned br = rows_now(m_box), ur = rows_now(m_in);
                const int comps = hist.mode == 3 ? 3 : 1;
                if (comps == 1 && hist.kind == kF32 && !hist.r) {
                    float* to = (float*)hist.e + at;
                    asm volatile("" : "+v"(to));  // one running address, not one per row
#pragma unroll
                    for (int q = 0; q < KR; ++q) {
                        if (row_of(br, q) && box_col) *to = eold[q];
                        to += hist.box.ny;
                    }
                } else
#pragma unroll
                for (int q = 0; q < KR; ++q) {
                    asm volatile("" : "+v"(at));  // one running index, not one per row
                    const long long row_at = at;
                    at += hist.box.ny;
                    if (!row_of(br, q) || !box_col) continue;
#pragma unroll 1
                    for (int ci = 0; ci < comps; ++ci) {
                        const bool is_ez = ci == comps - 1;  // Ex and Ey are identically zero here
                        const float eo = is_ez ? eold[q] : 0.0f, en = is_ez ? ez[q] : 0.0f;
                        const float a = is_ez && row_of(ur, q) && col_in ? ca[q] : 1.0f;
                        if (hist.e) store_hist(hist.e, ci * hist.cstride + row_at, eo, hist.kind);
                        if (hist.r)
                            store_hist(hist.r, ci * hist.cstride + row_at, cb[q] != 0.0f ? (en - a * eo) / cb[q] : 0.0f,
                                       hist.kind);
                    }
                }
            }
            if (listed)
#pragma unroll
                for (int q = 0; q < KR; ++q) s_ez[(w * KR + q) * 64 + lane] = ez[q];
        }
    }
    if (rend > rbeg) {
        __syncthreads();
        const auto& rx = args_now()->rx;
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
    const auto& pp = args_now()->pp;
    const auto& g = args_now()->g;
    float *oez = pp.Ez[1] + sb, *ohx = pp.Hx[1] + sb, *ohy = pp.Hy[1] + sb;
#pragma unroll
    for (int q = 0; q < KR; ++q) {
        if (!row_of(m_own, q)) continue;
        const unsigned p = 4u * (unsigned)((ib + q) * g.NY + jb);
        put(oez, p, ez[q]);
        put(ohx, p, hx[q]);
        put(ohy, p, hy[q]);
    }
    if (any_xh) {
        float* psi = choose(xhigh, pp.psi_h[1][1], pp.psi_h[1][0]) + (long long)s * fxh.p * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own & m_xh, q)) put(psi, 4u * (unsigned)(fxh.at(ib + q) * g.NY + jb), pxh[q]);
    }
    if (any_xe) {
        float* psi = choose(xhigh, pp.psi_e[1][1], pp.psi_e[1][0]) + (long long)s * (fxe.p + 1) * g.NY;
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own & m_xe, q)) put(psi, 4u * (unsigned)(fxe.at(ib + q) * g.NY + jb), pxe[q]);
    }
    if (yh) {
        float* psi = choose(yhigh, pp.psi_h[1][3], pp.psi_h[1][2]) + (long long)s * g.NX * fyh.p + fyh.at(jb);
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own, q)) psi[(ib + q) * fyh.p] = pyh[q];
    }
    if (ye) {
        const int depth = fye.p + 1;
        float* psi = choose(yhigh, pp.psi_e[1][3], pp.psi_e[1][2]) + (long long)s * g.NX * depth + fye.at(jb);
#pragma unroll
        for (int q = 0; q < KR; ++q)
            if (row_of(m_own, q)) psi[(ib + q) * depth] = pye[q];
    }
    }
}

// ---------------------------------------------------------------------------
// Launches
// ---------------------------------------------------------------------------
namespace {
// KR x NW rows and T steps of each shape. A launch costs 6 to 7 us before its
// first step and 1.1 us (order 2, KR = 2) to 1.8 us (order 4, KR = 4) a step, so
// a small solve takes few rows a wavefront, 16 wavefronts and many steps; one
// that fills the chip is bound by the instructions of the margin's cells, and
// takes more rows and fewer steps. Measured a step, in us, small / large shape:
// 121 x 121 order 2, 1 shot 1.9 / 2.4, 8 shots 2.0 / 2.5, 14 shots 3.2 / 2.9,
// 40 shots 6.3 / 4.8; order 4, 1 shot 3.3 / 4.8, 8 shots 3.6 / 5.0, 20 shots
// 7.8 / 6.6; 441 x 241, 20 shots, order 2 18 / 9.3, order 4 39 / 21. The
// one-step kernels take 5.0 to 7.5 (order 2), 5.8 to 8.8 (order 4) and, for the
// large grid, 30 and 35 us.
template <int ORDER, bool SMALL>
struct Shapes;
template <>
struct Shapes<2, true> {
    static constexpr int KR = 2, NW = 16, T = 8;
};
template <>
struct Shapes<2, false> {
    static constexpr int KR = 4, NW = 8, T = 6;
};
template <>
struct Shapes<4, true> {
    static constexpr int KR = 2, NW = 16, T = 3;
};
template <>
struct Shapes<4, false> {
    static constexpr int KR = 4, NW = 8, T = 2;
};
template <int ORDER, bool SMALL>
StripShape shape_of()
{
    using P = Shapes<ORDER, SMALL>;
    return {P::KR * P::NW, P::T * (2 * Radius<ORDER>::value - 1), P::T};
}
template <int ORDER, bool SMALL>
void launch_shape(const dim3& grid, const StripArgs& a, hipStream_t st)
{
    using P = Shapes<ORDER, SMALL>;
    hipLaunchKernelGGL((k_tm_strip_fwd<ORDER, P::KR, P::NW, P::T>), grid, dim3(P::NW * 64), 0, st, a);
}
}  // namespace

bool strip_applies(int order, const Tm2dGrid& g)
{
    if (order > 4 || g.plane >= 1 << 30) return false;  // 32-bit byte offsets
    // no face reaches the middle of its axis, and no strip of rows both faces
    return g.NX - g.pml[0] - g.pml[1] >= 12 && g.NY - g.pml[2] - g.pml[3] >= 4 && 2 * g.pml[0] + 9 < g.NX &&
           2 * g.pml[1] + 9 < g.NX && 2 * g.pml[2] + 2 < g.NY && 2 * g.pml[3] + 2 < g.NY;
}

// The small shapes as long as each of their workgroups (of 1024 threads, one a
// compute unit) has a compute unit to itself.
StripMap strip_map(int order, const Tm2dGrid& g)
{
    const StripMap small = make_strip_map(order == 4 ? shape_of<4, true>() : shape_of<2, true>(), g.NX, g.NY);
    if ((long long)small.tiles * g.nshot <= 256) return small;
    return make_strip_map(order == 4 ? shape_of<4, false>() : shape_of<2, false>(), g.NX, g.NY);
}

void launch_tm_strip_fwd(int order, const Tm2dGrid& g, const Tm2dFields& f, const TmPingPong& pp, const StripMap& sm,
                         const SourceBlocks& src, const TmReceiversFwd& rx, const StripHist& hist, int it0, int nsub,
                         hipStream_t st)
{
    const dim3 grid((unsigned)sm.tiles, (unsigned)g.nshot);
    const StripArgs a{g, f, pp, sm, src, rx, hist, make_spacing(g.d[0]), make_spacing(g.d[1]), it0, nsub};
    const bool small = sm.sh.steps == (order == 4 ? Shapes<4, true>::T : Shapes<2, true>::T);
    if (order == 4)
        small ? launch_shape<4, true>(grid, a, st) : launch_shape<4, false>(grid, a, st);
    else
        small ? launch_shape<2, true>(grid, a, st) : launch_shape<2, false>(grid, a, st);
}

}  // namespace dgx
