// Host check of the z windows of the adjoint row sweeps
// (deepgpr_amd/csrc/dgx_rows.h): whichever wavefront of a workgroup runs first,
// no weight that a thread uses comes from a CPML auxiliary that its owner has
// already advanced. The workgroups are played wavefront by wavefront, first to
// last and last to first: every thread forms the weights of its group from the
// auxiliaries as they are, writes those it owns to the row buffer and advances
// the auxiliaries it owns; after the barrier it takes its window as
// row_own_element says. The grids have to hold some where taking every cell of
// the group from its own registers would be wrong.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "dgx_rows.h"

using namespace dgx;

// Weights of the workgroup's threads that come from advanced auxiliaries.
static long long stale(const RowMap& m, const RowKind& kd, int W, const int pml[2], bool down, bool all_own)
{
    const int n = m.n2, nj = kd.rb, waves = m.threads / 64;
    std::vector<char> advanced((size_t)nj * n, 0), buffer((size_t)nj * n, 0), regs((size_t)m.threads * W, 0);
    auto in_face = [&](int k) {
        return (pml[0] > 0 && k <= pml[0]) || (pml[1] > 0 && k >= n - 1 - pml[1] && k <= n - 2);
    };
    for (int x = 0; x < waves; ++x) {
        const int w = down ? waves - 1 - x : x;
        for (int pass = 0; pass < 2; ++pass)  // a wavefront loads, then stores
            for (int t = w * 64; t < w * 64 + 64; ++t) {
                int row, k, dup;
                if (!row_thread(m, kd, W, t, nj, row, k, dup)) continue;
                for (int e = 0; e < W; ++e) {
                    const size_t c = (size_t)row * n + k + e;
                    if (pass == 0) regs[(size_t)t * W + e] = advanced[c];
                    else if (e >= dup) {
                        buffer[c] = regs[(size_t)t * W + e];
                        advanced[c] = in_face(k + e);
                    }
                }
            }
    }
    long long bad = 0;
    for (int t = 0; t < m.threads; ++t) {
        int row, k, dup;
        if (!row_thread(m, kd, W, t, nj, row, k, dup)) continue;
        for (int e = 0; e < W; ++e)
            bad += all_own || row_own_element(e, dup, W) ? regs[(size_t)t * W + e] : buffer[(size_t)row * n + k + e];
    }
    return bad;
}

int main()
{
    std::mt19937 rng(11);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    const int fixed[][3] = {{142, 20, 2}, {91, 21, 2}, {63, 6, 1}, {86, 20, 2}, {67, 10, 1}};  // N2, CPML, radius
    int done = 0, reached = 0;
    for (int it = 0; it < 4000; ++it) {
        int N[3] = {pick(40, 80), pick(40, 80), pick(40, 260)};
        int pml[6];
        for (int f = 0; f < 6; ++f) pml[f] = pick(0, 3) ? pick(1, 22) : 0;
        int R = pick(1, 2);
        if (it < 5) {
            N[0] = N[1] = 60;
            N[2] = fixed[it][0];
            pml[0] = pml[1] = pml[2] = pml[3] = 4;
            pml[4] = pml[5] = fixed[it][1];
            R = fixed[it][2];
        }
        if (!row_sweep_applies(N, pml, 2 * R)) continue;
        const RowMap m = make_row_map(N, pml, R, 4, 256);
        bool split = false;
        for (int down = 0; down < 2; ++down)
            for (int kind = 0; kind < 2; ++kind) {
                const RowKind& kd = kind ? m.plain : m.edge;
                const int W = kind ? 4 : 2;
                if (stale(m, kd, W, pml + 4, down, false)) {
                    std::printf("FAILED grid %d x %d x %d CPML %d %d radius %d: weights from advanced auxiliaries\n",
                                N[0], N[1], N[2], pml[4], pml[5], R);
                    return 1;
                }
                split = split || stale(m, kd, W, pml + 4, down, true);
            }
        if (it < 5 && !split) {
            std::printf("FAILED grid %d x %d x %d CPML %d: its groups share wavefronts\n", N[0], N[1], N[2], pml[4]);
            return 1;
        }
        ++done;
        reached += split;
    }
    if (done < 100 || reached < 15) {
        std::printf("FAILED: %d grids, %d of them with the last groups of a row in two wavefronts\n", done, reached);
        return 1;
    }
    std::printf("all checks passed (%d grids, %d with the last groups of a row in two wavefronts)\n", done, reached);
    return 0;
}
