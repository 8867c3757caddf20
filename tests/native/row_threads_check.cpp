// Host check of the row sweeps' workgroups on long rows (deepgpr_amd/csrc/dgx_rows.h):
// where the groups of an edge row need more than 256 threads, the plain
// workgroups fill as many. And which long rows the sweeps take: order 4 from 704
// cells, forward sweeps where fewer than half of the rows are plain.
#include <cstdio>

#include "dgx_rows.h"

using namespace dgx;

int main()
{
    for (int order = 2; order <= 4; order += 2)
        for (int n = 513; n <= 1024; ++n) {
            const int N[3] = {100, 100, n}, pml[6] = {20, 20, 20, 20, 4, 4}, few[6] = {5, 5, 5, 5, 4, 4};
            const RowMap m = make_row_map(N, pml, order / 2, 4, 256);
            if (m.plain.rb * m.plain.gpr * 5 < m.threads * 3 || m.edge.rb * m.edge.gpr * 5 < m.threads * 3 ||
                m.threads > 512) {
                std::printf("FAILED rows of %d cells: %d and %d of %d threads\n", n, m.plain.rb * m.plain.gpr,
                            m.edge.rb * m.edge.gpr, m.threads);
                return 1;
            }
            const bool taken = order == 2 || n >= 704;
            if (row_sweep_applies(N, pml, order, true) != taken || row_sweep_applies(N, pml, order, false) != taken ||
                row_sweep_applies(N, few, order, true) != taken || row_sweep_applies(N, few, order, false)) {
                std::printf("FAILED rule for rows of %d cells, order %d\n", n, order);
                return 1;
            }
        }
    const int N[3] = {100, 100, 512}, few[6] = {5, 5, 5, 5, 4, 4};
    if (!row_sweep_applies(N, few, 4, false) || !row_sweep_applies(N, few, 4, true)) {
        std::printf("FAILED rule for rows of 512 cells\n");
        return 1;
    }
    std::printf("all checks passed\n");
    return 0;
}
