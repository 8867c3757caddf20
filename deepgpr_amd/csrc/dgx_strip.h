// Tiles of the 2D TM strip kernels (dgx_tm2d_strip.hip), shared by the kernels
// and the host code that builds their source and receiver lists.
//
// A workgroup stages SR = KR * NW rows x 64 columns of one shot (KR rows a
// wavefront, one lane a column) and advances them T steps. Each step the outer
// 2R - 1 rows and columns become unusable, so it owns the (SR - 2 H) x
// (64 - 2 H) cells inside a margin of H = T (2R - 1).
#pragma once

#include "dgx_sweep.h"

namespace dgx {

struct StripShape {
    int size;    // which of the shapes (dgx_tm2d_strip.hip)
    int rows;    // SR
    int halo;    // H
    int steps;   // T
    int waves;   // NW
};

struct StripMap {
    StripShape sh;
    int orow, ocol;      // owned rows and columns of a tile
    int nti, ntj, tiles;
};

inline StripMap make_strip_map(const StripShape& sh, int nx, int ny)
{
    StripMap m{};
    m.sh = sh;
    m.orow = sh.rows - 2 * sh.halo;
    m.ocol = 64 - 2 * sh.halo;
    m.nti = (nx + m.orow - 1) / m.orow;
    m.ntj = (ny + m.ocol - 1) / m.ocol;
    m.tiles = m.nti * m.ntj;
    return m;
}

// Tiles whose staged region holds row (or column) c: [first, last].
inline void strip_tiles(int c, int owned, int halo, int staged, int count, int& first, int& last)
{
    // staged region of tile t: [t owned - halo, t owned - halo + staged)
    first = (c + halo - staged + owned) / owned;
    if (c + halo - staged + 1 <= 0) first = 0;
    last = (c + halo) / owned;
    if (last > count - 1) last = count - 1;
}

// Wavefront of a tile that stages the cell with index `local`.
inline int strip_wave(const StripMap& m, int local) { return (local >> 6) / (m.sh.rows / m.sh.waves); }

// Staged index (row * 64 + column) of cell (i, j) in tile (ti, tj).
inline int strip_local(const StripMap& m, int ti, int tj, int i, int j)
{
    return (i - (ti * m.orow - m.sh.halo)) * 64 + (j - (tj * m.ocol - m.sh.halo));
}

}  // namespace dgx
