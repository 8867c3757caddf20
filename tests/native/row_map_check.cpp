// Host check of the row sweeps' block map (deepgpr_amd/csrc/dgx_rows.h): every
// cell is owned by exactly one thread, whole wavefronts, at most 512 threads,
// groups inside their row and the row buffers, plain workgroups in the plain
// ranges, the inverse used for the source and receiver lists, taps of the plain
// z-range inside the row and away from the faces, and row blocks on one XCD.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "dgx_rows.h"

using namespace dgx;

static int fail(const char* what, const int N[3], int a, int b)
{
    std::printf("FAILED %s: grid %d x %d x %d (%d, %d)\n", what, N[0], N[1], N[2], a, b);
    return 1;
}

static int check(const int N[3], const int pml[6], int R, int V)
{
    const RowMap m = make_row_map(N, pml, R, V, 256);
    if (m.threads > 512 || m.threads % 64) return fail("threads", N, m.threads, m.plain.rb);
    const int lo[3] = {m.xlo, m.ylo, m.zlo}, hi[3] = {m.xhi, m.yhi, m.zhi};
    for (int a = 0; a < 3; ++a)
        for (int c = lo[a]; c <= hi[a]; ++c) {
            if (c - R < 0 || c + R > N[a] - 2) return fail("taps outside the axis", N, c, R);
            if (pml[2 * a] > 0 && c - R < pml[2 * a]) return fail("taps in the low face", N, c, R);
            if (pml[2 * a + 1] > 0 && c + R > N[a] - 2 - pml[2 * a + 1]) return fail("taps in the high face", N, c, R);
            if (c < 2 * R - 1 || c > N[a] - 2 * R) return fail("clamped transposed stencil", N, c, R);
        }
    std::vector<unsigned char> seen((size_t)N[0] * N[1] * N[2], 0);
    for (int b = 0; b < m.total; ++b) {
        int i, j0, nj;
        const int kind = row_block(m, b, i, j0, nj);
        if (kind < 0) continue;
        const int W = kind == 1 ? V : V / 2;
        const RowKind& kd = kind == 1 ? m.plain : m.edge;
        if (i < 0 || i >= N[0] || j0 < 0 || nj < 1 || nj > kd.rb || j0 + nj > N[1]) return fail("block", N, i, j0);
        const bool px = i >= m.xlo && i <= m.xhi, py = j0 >= m.ylo && j0 + nj - 1 <= m.yhi;
        if ((kind == 1) != (px && py)) return fail("kind", N, i, j0);
        int next = i + 1;
        if (next < N[0] && (next >= m.xlo) == (i >= m.xlo) && (next > m.xhi) == (i > m.xhi) &&
            row_block_of(m, next, j0) % 8 != b % 8)
            return fail("XCD of a row", N, i, j0);
        for (int t = 0; t < m.threads; ++t) {
            int row, k, dup;
            const bool live = row_thread(m, kd, W, t, nj, row, k, dup);
            const int j = j0 + row;
            if (row < 0 || row >= nj || k < 0 || k + W > N[2] || dup < 0 || dup >= W) return fail("group", N, k, dup);
            if (row * kd.gpr * W + N[2] > m.lds) return fail("row buffer", N, row, m.lds);
            if (!live) continue;
            if (row_block_of(m, i, j) != b) return fail("inverse", N, i, j);
            for (int e = dup; e < W; ++e) seen[((size_t)i * N[1] + j) * N[2] + k + e] += 1;
        }
    }
    for (size_t n = 0; n < seen.size(); ++n)
        if (seen[n] != 1) return fail("coverage", N, (int)(n / N[2]), (int)(n % N[2]));
    return 0;
}

int main()
{
    std::mt19937 rng(7);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    int done = 0, bad = 0;
    for (int it = 0; it < 120 && !bad; ++it) {
        int N[3] = {pick(20, 80), pick(20, 80), it % 5 == 0 ? pick(300, 1024) : pick(40, 140)};
        int pml[6];
        for (int f = 0; f < 6; ++f) pml[f] = pick(0, 3) ? pick(1, 16) : 0;
        if (!row_sweep_applies(N, pml, 4)) continue;
        for (int R : {1, 2}) bad |= check(N, pml, R, 4);
        ++done;
    }
    // what the rule refuses: small interiors, short and long rows, order 8
    const int none[6] = {0, 0, 0, 0, 0, 0};
    const int small[3] = {30, 31, 32}, flat[3] = {400, 400, 2}, tall[3] = {64, 64, 1025}, good[3] = {64, 64, 64};
    if (row_sweep_applies(small, none, 4) || row_sweep_applies(flat, none, 4) || row_sweep_applies(tall, none, 4) ||
        !row_sweep_applies(good, none, 4) || row_sweep_applies(good, none, 8)) {
        std::printf("FAILED rule\n");
        bad = 1;
    }
    if (!bad && done >= 30) std::printf("all checks passed (%d grids)\n", done);
    return bad || done < 30;
}
