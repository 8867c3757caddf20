// Block -> cell mapping of the row sweeps (dgx_rows.hip), shared by the
// kernels, the host launch code and a host-only test.
//
// A workgroup owns some consecutive rows of one x-plane of one shot, over
// their whole z extent; its threads take the rows one after another in groups
// of consecutive cells. The last group of a row is moved back to end with the
// row: its first cells belong to the group before it. There are two kinds of
// workgroups: plain ones, whose rows lie in the plain ranges of x and y, with
// groups of V cells, and edge ones with groups of V / 2 cells (their code holds
// more values a cell). The first threads of a workgroup take the groups at the
// ends of its rows, so that one or two wavefronts run the z-CPML and the z-edge
// code and the others skip it.
#pragma once

#include "dgx_sweep.h"

namespace dgx {

struct RowKind {
    int gpr;   // groups of a row
    int rb;    // rows of a workgroup
    int ends;  // groups of a row that reach out of the plain z-range
    int low;   // of these, the ones at its start
    Div div_ends, div_mid;  // / ends, / (gpr - ends), or / 1
};

struct RowMap {
    RowKind plain, edge;
    int V;               // cells of a plain group
    int threads;         // threads of a workgroup (a multiple of 64)
    int lds;             // floats of one row buffer of a workgroup
    int n0, n1, n2;      // the grid
    int xlo, xhi, ylo, yhi, zlo, zhi;  // plain ranges (inclusive)
    int ne, nm;          // edge and plain workgroups of an inner plane (i in [xlo, xhi])
    int nylo;            // of the ne, those of rows below ylo
    int bo, bi;          // workgroups of an outer / inner plane, padded to multiples of 8
    int to, ti;          // of all outer / inner planes
    int ratio;           // bundles of 8 inner workgroups after one of outer ones
    int total;           // workgroups of a shot
    Div div_bo, div_bi, div_group;  // / bo, / bi, / (8 (1 + ratio))
};

// Plain range along one axis of n cells with CPML widths plo and phi: cells
// whose stencils, and the transposed stencils of the adjoint, are full-width,
// see no CPML term of this axis and read only updated cells.
DGX_HD void row_plain_range(int n, int plo, int phi, int R, int& lo, int& hi)
{
    lo = 2 * R - 1;
    if (plo > 0 && plo + R > lo) lo = plo + R;
    hi = n - 2 * R;
    if (n - 2 - R < hi) hi = n - 2 - R;
    if (phi > 0 && n - 2 - phi - R < hi) hi = n - 2 - phi - R;
}

// The face of an axis of n cells that a thread of the row sweeps looks at: the
// one on the side of its cell c (along z, of its first cell).
DGX_HD bool row_high_side(int c, int n) { return 2 * c > n; }

// Cells beyond its own for which a thread relies on that face: the taps of the
// adjoint along x and y (radius 2 at order 4), and the others of its group along z.
constexpr int kRowReach = 3;

// A face of width p, on the low or the high side of an axis of n cells, that is
// in no thread's reach on the other side: its cells are 0 .. p or n - 1 - p .. n - 2.
inline bool row_face_fits(int n, int p, bool high)
{
    if (p <= 0) return true;
    const int last_low = n / 2;  // the last cell for which row_high_side is false
    return high ? last_low + kRowReach < n - 1 - p : last_low + 1 - kRowReach > p;
}

// The row sweeps take solves of order 2 and 4 on grids with a plain interior
// that is worth it: at least 65536 cells plain for every order, in rows of at
// least 32 of them and at most 1024 cells (a row fits a workgroup of 512
// threads), and a field array of a shot below 4 GiB (32-bit offsets). An
// order-8 cell has so many taps that its values fill the registers of a
// thread (us per step on an MI355X, row sweeps / one thread per cell: forward
// 118 / 100, adjoint 199 / 152 on 138 x 120 x 152 fields).
//
// Rows of more than 512 cells need workgroups of 5 to 8 wavefronts, a row or two
// each, and fewer of those share a compute unit. Forward and adjoint, us a step,
// rows / one thread per cell, fields of 111 x 111 (CPML 10: 62 % of the rows
// plain), 151 x 151 (CPML 30: 31 %) and 61 x 61 (CPML 10: 39 %) rows:
//   order 4   501 cells   172 / 181   217 / 304    389 / 575   534 / 840     63 /  79    85 / 117
//   order 4   521         241 / 189   326 / 318    562 / 596   831 / 860     90 /  80   137 / 120
//   order 4   701         293 / 249   378 / 414    648 / 762   912 / 1078    99 / 101   146 / 163
//   order 2   521         177 / 165   225 / 259    395 / 550   568 / 792     66 /  74    92 / 110
//   order 2   701         220 / 215   278 / 342    475 / 702   682 / 988     76 /  93   112 / 145
// Hence: order 4 from 704 cells again, and a forward sweep only where fewer than
// half of the rows are plain.
inline bool row_sweep_applies(const int N[3], const int pml[6], int order, bool backward = true)
{
    if (order > 4) return false;
    long long cells = 1, rows = 1;
    for (int a = 0; a < 3; ++a) {
        int lo, hi;
        row_plain_range(N[a], pml[2 * a], pml[2 * a + 1], 4, lo, hi);
        if (hi < lo) return false;
        if (a == 2 && hi - lo + 1 < 32) return false;
        if (a == 2) rows = cells;
        cells *= hi - lo + 1;
        if (!row_face_fits(N[a], pml[2 * a], false) || !row_face_fits(N[a], pml[2 * a + 1], true)) return false;
    }
    if (N[2] > 512 && ((order == 4 && N[2] < 704) || (!backward && 2 * rows >= 1LL * N[0] * N[1]))) return false;
    return cells >= 65536 && N[2] <= 1024 && 1LL * N[0] * N[1] * N[2] < (1LL << 30);
}

// Rows of a workgroup: the count within max_threads that leaves the fewest
// lanes idle, the larger of nearly equal ones.
inline RowKind make_row_kind(int n2, int V, int max_threads)
{
    RowKind k{};
    k.gpr = (n2 + V - 1) / V;
    double best = 0.0;
    for (int rb = 1; rb <= 16; ++rb) {
        const int t = (rb * k.gpr + 63) / 64 * 64;
        if (rb > 1 && t > max_threads) break;
        const double use = (double)rb * k.gpr / t;
        if (use > best - 0.02) {
            best = use > best ? use : best;
            k.rb = rb;
        }
    }
    return k;
}

// Groups at the ends of a row: not wholly in the plain z-range.
inline void set_row_ends(RowKind& k, int V, int zlo, int zhi)
{
    const int low = (zlo + V - 1) / V, from = (zhi + 1) / V;  // groups below zlo; the first group beyond zhi
    k.low = low < k.gpr ? low : k.gpr;
    const int high = k.gpr - (from > k.low ? from : k.low);
    k.ends = k.low + (high > 0 ? high : 0);
    if (k.ends >= k.gpr) k.ends = k.low = 0;  // no others
    k.div_ends = make_div((unsigned)(k.ends > 0 ? k.ends : 1));
    k.div_mid = make_div((unsigned)(k.gpr > k.ends ? k.gpr - k.ends : 1));
}

inline RowMap make_row_map(const int N[3], const int pml[6], int R, int V, int max_threads)
{
    RowMap m{};
    m.V = V;
    m.n0 = N[0];
    m.n1 = N[1];
    m.n2 = N[2];
    row_plain_range(N[0], pml[0], pml[1], R, m.xlo, m.xhi);
    row_plain_range(N[1], pml[2], pml[3], R, m.ylo, m.yhi);
    row_plain_range(N[2], pml[4], pml[5], R, m.zlo, m.zhi);
    // A long row takes more than max_threads threads in edge groups, and the launch
    // has as many for every workgroup: the plain ones then hold rows for all of
    // them (two rows of 561 cells in 282 threads of 320, not one in 141).
    m.edge = make_row_kind(N[2], V / 2, max_threads);
    const int most = (m.edge.rb * m.edge.gpr + 63) / 64 * 64;
    m.plain = make_row_kind(N[2], V, most > max_threads ? most : max_threads);
    set_row_ends(m.plain, V, m.zlo, m.zhi);
    set_row_ends(m.edge, V / 2, m.zlo, m.zhi);
    const int tp = m.plain.rb * m.plain.gpr, te = m.edge.rb * m.edge.gpr;
    m.threads = ((tp > te ? tp : te) + 63) / 64 * 64;
    const int lp = tp * V, le = te * (V / 2);
    m.lds = ((lp > le ? lp : le) + 3) / 4 * 4;
    auto blocks = [](int rows, int rb) { return (rows + rb - 1) / rb; };
    auto pad8 = [](int n) { return (n + 7) / 8 * 8; };
    m.nylo = blocks(m.ylo, m.edge.rb);
    m.ne = m.nylo + blocks(m.n1 - 1 - m.yhi, m.edge.rb);
    m.nm = blocks(m.yhi - m.ylo + 1, m.plain.rb);
    m.bi = pad8(m.ne + m.nm);
    m.bo = pad8(blocks(m.n1, m.edge.rb));
    m.ti = m.bi * (m.xhi - m.xlo + 1);
    m.to = m.bo * (m.n0 - (m.xhi - m.xlo + 1));
    m.ratio = (m.ti + m.to / 2) / m.to;
    if (m.ratio < 1) m.ratio = 1;
    const int go = m.to / 8, gi = (m.ti / 8 + m.ratio - 1) / m.ratio;
    m.total = (go > gi ? go : gi) * 8 * (1 + m.ratio);
    m.div_bo = make_div((unsigned)m.bo);
    m.div_bi = make_div((unsigned)m.bi);
    m.div_group = make_div((unsigned)(8 * (1 + m.ratio)));
    return m;
}

// Workgroup b of a shot: its kind (1 plain, 0 edge, -1 none), plane, first row
// and row count. The outer planes' workgroups (CPML along x) are spread among
// the others, so that their longer chains run beside them. Workgroup b runs on
// XCD b mod 8, and so does the same row block of the next plane (bundles of 8,
// bo and bi multiples of 8): x-neighbours meet in one L2.
DGX_HD int row_block(const RowMap& m, int b, int& i, int& j0, int& nj)
{
    const int span = 8 * (1 + m.ratio);
    const int g = (int)div_q((unsigned)b, m.div_group), r = b - g * span;
    if (r < 8) {
        const int o = g * 8 + r;
        if (o >= m.to) return -1;
        const int pl = (int)div_q((unsigned)o, m.div_bo);
        i = pl < m.xlo ? pl : pl + (m.xhi - m.xlo + 1);
        j0 = (o - pl * m.bo) * m.edge.rb;
        nj = m.n1 - j0 < m.edge.rb ? m.n1 - j0 : m.edge.rb;
        return nj > 0 ? 0 : -1;
    }
    const int o = g * 8 * m.ratio + r - 8;
    if (o >= m.ti) return -1;
    const int pl = (int)div_q((unsigned)o, m.div_bi);
    const int p = o - pl * m.bi;
    i = m.xlo + pl;
    if (p < m.ne) {
        const bool low = p < m.nylo;
        j0 = low ? p * m.edge.rb : m.yhi + 1 + (p - m.nylo) * m.edge.rb;
        const int end = low ? m.ylo : m.n1;
        nj = end - j0 < m.edge.rb ? end - j0 : m.edge.rb;
        return 0;
    }
    j0 = m.ylo + (p - m.ne) * m.plain.rb;
    nj = m.yhi + 1 - j0 < m.plain.rb ? m.yhi + 1 - j0 : m.plain.rb;
    return nj > 0 ? 1 : -1;
}

// Thread t of a workgroup of nj rows (the ends of its rows first, then what lies
// between them, row by row): its row, the first cell k of its group of
// V cells and how many of the group's first cells belong to the group before
// it; false for an idle thread (row, k and dup are then those of a valid one).
DGX_HD bool row_thread(const RowMap& m, const RowKind& kd, int V, int t, int nj, int& row, int& k, int& dup)
{
    const int u = t - kd.rb * kd.ends;
    if (u < 0) {
        row = (int)div_q((unsigned)t, kd.div_ends);
        k = t - row * kd.ends;
        if (k >= kd.low) k += kd.gpr - kd.ends;
    } else {
        const int mid = kd.gpr - kd.ends;
        row = (int)div_q((unsigned)u, kd.div_mid);
        k = u - row * mid + kd.low;
    }
    k *= V;
    dup = 0;
    if (k > m.n2 - V) {
        dup = k - (m.n2 - V);
        k = m.n2 - V;
    }
    if (row < nj) return true;
    row = 0;
    return false;
}

// Whether element e of a group (its cell k + e) comes from the group's own
// registers in a z-stencil, not from the row buffer, which every owner fills
// before the barrier. The adjoint's z weights are formed from CPML auxiliaries
// that their owner advances in place, so a cell of the group before (e < dup)
// is right in the buffer alone: the thread before it may be in another
// wavefront and have advanced the auxiliary already.
DGX_HD bool row_own_element(int e, int dup, int V) { return e >= dup && e < V; }

// Workgroup of a shot that owns row (i, j).
inline int row_block_of(const RowMap& m, int i, int j)
{
    if (i < m.xlo || i > m.xhi) {
        const int pl = i < m.xlo ? i : i - (m.xhi - m.xlo + 1);
        const int o = pl * m.bo + j / m.edge.rb;
        return o / 8 * 8 * (1 + m.ratio) + o % 8;
    }
    const int p = j < m.ylo ? j / m.edge.rb
                            : (j > m.yhi ? m.nylo + (j - m.yhi - 1) / m.edge.rb : m.ne + (j - m.ylo) / m.plain.rb);
    const int o = (i - m.xlo) * m.bi + p;
    const int g = o / (8 * m.ratio);
    return g * 8 * (1 + m.ratio) + 8 + o - g * 8 * m.ratio;
}

}  // namespace dgx
