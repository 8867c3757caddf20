// Host check of the rule by which the row sweeps take grids with CPML faces
// (deepgpr_amd/csrc/dgx_rows.h), by brute force over the widths of a pair of
// faces: on every grid that row_sweep_applies takes, each cell that a thread
// treats (along x and y the cells its adjoint taps reach, along z the cells of
// its group) lies in no face but the one on the side that row_high_side names.
#include <cstdio>

#include "dgx_rows.h"

using namespace dgx;

static bool in_face(int c, int n, int p, bool high)
{
    if (p <= 0 || c < 0 || c >= n) return false;
    return high ? c >= n - 1 - p && c <= n - 2 : c <= p;  // electric and magnetic faces together
}

int main()
{
    int taken = 0, refused = 0;
    for (int axis = 0; axis < 3; ++axis)
        for (int n = 40; n <= 103; n += axis == 2 ? 7 : 3)
            for (int plo = 0; plo < n; ++plo)
                for (int phi = 0; phi < n; ++phi) {
                    int N[3] = {400, 400, 400}, pml[6] = {4, 4, 4, 4, 4, 4};
                    N[axis] = n;
                    pml[2 * axis] = plo;
                    pml[2 * axis + 1] = phi;
                    if (!row_sweep_applies(N, pml, 4)) {
                        ++refused;
                        continue;
                    }
                    ++taken;
                    for (int c = 0; c < n; ++c) {
                        const bool other = !row_high_side(c, n);
                        const int from = axis == 2 ? c : c - 2, to = axis == 2 ? c + 3 : c + 2;
                        for (int t = from; t <= to; ++t)
                            if (in_face(t, n, other ? phi : plo, other)) {
                                std::printf("FAILED axis %d of %d cells, faces %d and %d: cell %d reaches %d\n", axis, n,
                                            plo, phi, c, t);
                                return 1;
                            }
                    }
                }
    // ordinary widths are taken: a quarter of the axis each, and one wide face
    const int N[3] = {160, 160, 160}, quarter[6] = {40, 40, 40, 40, 40, 40}, wide[6] = {76, 4, 4, 75, 20, 20};
    if (!row_sweep_applies(N, quarter, 4) || !row_sweep_applies(N, wide, 4) || taken < 10000 || refused < 10000) {
        std::printf("FAILED: %d taken, %d refused\n", taken, refused);
        return 1;
    }
    std::printf("all checks passed (%d taken, %d refused)\n", taken, refused);
    return 0;
}
