"""bench.py's bytes of a kernel launch: the kernels of the 3D row sweeps and of
the one-thread-per-cell sweeps share names, and the run's kernels tell them
apart. No GPU needed."""
import os
import sys
from types import SimpleNamespace

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

ARGS = SimpleNamespace(shots_per_call=2, rhs="auto", storage="float32", accumulator="float64")


def _workload(shape, pml):
    cells = 1
    for n in shape:
        cells *= n + 2 * pml
    return SimpleNamespace(physical_shape=shape, pml=pml, mode=3, sampling_interval=4, extended_cells=lambda: cells)


@pytest.mark.parametrize("ran,core", [(("adj_e", "adj_h"), {"adj_e": 40, "adj_h": 44}),
                                      (("adj_weights_e", "adj_e_w", "adj_h"), {"adj_weights_e": 40, "adj_e_w": 76,
                                                                              "adj_h": 52}),
                                      (("adj_weights_e", "adj_weights_h", "adj_e", "adj_h"),
                                       {"adj_weights_e": 40, "adj_weights_h": 40, "adj_e": 48, "adj_h": 52})])
def test_adjoint_bytes_follow_the_sweeps(ran, core):
    w = _workload((30, 20, 40), 0)
    for kernel, per_cell in core.items():
        got = bench.kernel_bytes(kernel, w, ARGS, ran=ran)
        assert got == per_cell * 2 * w.extended_cells() + 8 * 2 * _psi(kernel, ran, w), kernel


def _psi(kernel, ran, w):
    e, h = bench._psi_elems(w)
    if kernel.startswith("adj_weights") or "adj_weights_e" not in ran:
        return h if kernel.endswith("_h") else e
    return h if kernel == "adj_e_w" else 0


def test_sum_of_material_terms_reads_the_terms_it_holds():
    w = _workload((50, 60), 10)
    cells = w.extended_cells()
    one = bench.kernel_bytes("tm_grad_reduce", w, ARGS)
    held = bench.kernel_bytes("tm_grad_reduce", w, ARGS, 32.0, ("tm_strip_adj", "tm_grad_reduce"))
    assert one == 32 * cells + 8 * 2 * cells  # two FP64 accumulators read and written, two terms of two shots
    assert held == 32 * cells + 8 * 8 * 2 * cells  # eight saved steps' terms
