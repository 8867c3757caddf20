"""The row sweeps of 3D solves (deepgpr_amd/csrc/dgx_rows.hip) against the CPU
oracle, bit for bit: rows of every remainder by the group width, CPML widths
that cut groups, faces without CPML, unequal spacing, PEC cells, odd and even
step counts (the adjoint's second auxiliary copies), every history format and
box, sources and coincident receivers of every component on the outermost
cells, in the CPML and inside, and rows that fill a workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # (NX, NY, NZ, order, nt, nshot, S, storage, pml, component, kw)
    (58, 55, 64, 2, 7, 1, 1, "e_only", (5, 4, 3, 6, 4, 5), 2, {}),
    (57, 58, 65, 4, 8, 2, 2, "f32", (4, 5, 6, 3, 7, 3), 0, {}),
    (58, 56, 66, 4, 7, 1, 3, "bf16", (3, 0, 0, 4, 5, 0), 1, {"pec": True}),
    (56, 57, 67, 2, 8, 1, 2, "f16", (0, 5, 4, 0, 0, 6), 2, {"pec": True}),
    (56, 55, 69, 4, 7, 2, 2, "int8", (4, 4, 4, 4, 8, 8), 2, {}),
    (50, 56, 66, 4, 6, 1, 1, "physical", (0, 0, 0, 0, 0, 0), 1, {}),
    (52, 50, 70, 2, 7, 1, 1, "physical_forward", (3, 4, 2, 3, 5, 2), 2, {}),
    (46, 40, 519, 4, 5, 1, 1, "f32", (4, 3, 2, 3, 5, 9), 0, {}),
    (40, 38, 1021, 2, 4, 1, 1, "e_only", (4, 3, 2, 3, 5, 9), 2, {}),
]


def _storage(h, name):
    return {"f32": 0, "e_only": h.RHS_FROM_E, "f16": h.KIND_F16, "bf16": h.KIND_BF16,
            "int8": h.int8_storage_type((4, 4, 4)), "physical": h.PHYSICAL, "physical_forward": h.PHYSICAL}[name]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-o{c[3]}-{c[7]}")
def test_row_sweeps_match_oracle_bitwise(oracle_built, cuda_device, case):
    h = oracle_built
    NX, NY, NZ, order, nt, nshot, S, st, pml, comp, kw = case
    print(f"[gpu row sweeps] {case}", flush=True)
    p = h.make_problem(NX, NY, NZ, order=order, nt=nt, nshot=nshot, nsrc=3, nrx=8, seed=17, pml=pml,
                       d=(0.02, 0.017, 0.015), **kw)
    p.S = S
    p.storage_type = _storage(h, st)
    p.src_comp = p.rx_comp = comp
    last = nshot - 1
    p.src_loc[0, 0] = [NX // 2, NY // 2, 1]
    p.src_loc[last, 1] = [NX // 2 + 1, 1, NZ // 2]
    p.src_loc[0, 2] = p.src_loc[0, 0]
    spots = [[NX // 2, NY // 2, NZ // 2], [NX // 2, NY // 2, NZ // 2], [1, NY // 2, 3], [NX - 2, 2, NZ - 3],
             [NX // 3, NY - 2, NZ - 2], [0, 0, 0], [NX // 2, NY // 3, NZ - 5], [NX // 2, NY // 2, 2]]
    for s in range(nshot):
        for r, cell in enumerate(spots):
            p.rx_loc[s, r] = cell
    backward = st != "physical_forward"  # its gradient would lack the CPML's part
    p.save_model_history = int(backward)
    cpu = h.run_cpu(p, "oracle", backward=backward)
    gpu = h.run_gpu(p, backward=backward, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + (list(h.KEYS_BWD) if backward else []))
    assert not bad, bad
    assert np.array_equal(gpu["E_saved"], cpu["E_saved"])
    assert np.array_equal(gpu["R_saved"], cpu["R_saved"])


@pytest.mark.parametrize("shape,pml", [((64, 80, 96), (36, 4, 4, 4, 4, 4)), ((80, 66, 96), (4, 4, 5, 36, 4, 3)),
                                       ((70, 70, 100), (4, 4, 4, 4, 56, 3))])
def test_faces_beyond_the_middle_match_oracle(oracle_built, cuda_device, shape, pml):
    """A CPML that reaches past the middle of its axis."""
    h = oracle_built
    print(f"[gpu row sweeps] faces beyond the middle {shape} {pml}", flush=True)
    p = h.make_problem(*shape, order=2, nt=4, nshot=1, nsrc=2, nrx=4, seed=29, pml=pml, d=(0.02, 0.02, 0.02))
    p.src_loc[0, 0] = [shape[0] // 2, shape[1] // 2, shape[2] // 2]
    cpu = h.run_cpu(p, "oracle")
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad


@pytest.mark.parametrize("shape,order,pz,nt", [((60, 58, 142), 4, 20, 7), ((60, 60, 91), 4, 21, 6),
                                               ((60, 60, 63), 2, 6, 7), ((62, 60, 67), 2, 10, 6)])
def test_split_row_ends_match_oracle(oracle_built, cuda_device, shape, order, pz, nt):
    """Rows whose last two groups overlap and lie in two wavefronts of a workgroup (tests/native/row_window_check.cpp)."""
    h = oracle_built
    print(f"[gpu row sweeps] split row ends {shape} {order} {pz}", flush=True)
    p = h.make_problem(*shape, order=order, nt=nt, nshot=2, nsrc=2, nrx=6, seed=43, pml=(4, 4, 4, 4, pz, pz),
                       d=(0.02, 0.017, 0.015))
    for s in range(2):
        p.src_loc[s, 0] = [shape[0] // 2, shape[1] // 2, shape[2] - 4]
        for r in range(6):
            p.rx_loc[s, r] = [10 + 8 * r, 5 + 9 * r, shape[2] - 2 - r]
    cpu = h.run_cpu(p, "oracle")
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("shape,pml", [((80, 72, 84), (4, 38, 4, 4, 4, 4)), ((74, 81, 84), (4, 4, 38, 0, 3, 4)),
                                       ((72, 72, 84), (4, 4, 4, 4, 3, 40)), ((72, 72, 84), (4, 4, 4, 4, 5, 36)),
                                       ((81, 80, 90), (36, 3, 0, 35, 4, 4))])
def test_faces_close_to_the_middle_match_oracle(oracle_built, cuda_device, shape, pml, order):
    """A CPML that ends within a few cells of the middle of its axis, one side or the other of what row sweeps take."""
    h = oracle_built
    print(f"[gpu row sweeps] faces close to the middle {shape} {pml} {order}", flush=True)
    p = h.make_problem(*shape, order=order, nt=4, nshot=1, nsrc=2, nrx=4, seed=31, pml=pml, d=(0.02, 0.02, 0.02))
    p.src_loc[0, 0] = [shape[0] // 2, shape[1] // 2, shape[2] // 2]
    cpu = h.run_cpu(p, "oracle")
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad


@pytest.mark.parametrize("NZ,order,comp,nshot", [(66, 4, 1, 1), (71, 2, 2, 2), (68, 4, 0, 1)])
def test_many_sources_match_oracle(oracle_built, cuda_device, NZ, order, comp, nshot):
    """Sources on whole planes, in no order, several on one cell: more of a workgroup than every thread looks at."""
    h = oracle_built
    print(f"[gpu row sweeps] many sources {NZ} {order} {comp}", flush=True)
    p = h.make_problem(56, 54, NZ, order=order, nt=5, nshot=nshot, nsrc=1, nrx=5, seed=37, pml=(4, 3, 5, 4, 4, 6),
                       d=(0.02, 0.017, 0.015))
    cells = [(20, j, k) for j in range(0, 53, 2) for k in range(0, NZ - 1)] + [(i, 30, 33) for i in range(55)]
    cells += [(20, 16, 9)] * 7 + [(5, 5, NZ - 2)] * 3
    rng = np.random.default_rng(5)
    order_ = rng.permutation(len(cells))
    p.src_loc = np.array([[list(cells[k]) for k in order_] for _ in range(nshot)], np.int32)
    p.wave = rng.standard_normal((len(cells), 5)).astype(np.float32)
    p.src_comp = p.rx_comp = comp
    for s in range(nshot):
        for r in range(5):
            p.rx_loc[s, r] = [18 + r, 16, 8 + r]
    cpu = h.run_cpu(p, "oracle")
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad


@pytest.mark.parametrize("shape,order,pml", [((48, 46, 707), 4, (6, 5, 7, 4, 5, 9)), ((48, 46, 541), 2, (6, 5, 7, 4, 5, 9)),
                                             ((30, 33, 1022), 4, (4, 4, 4, 4, 6, 6)),
                                             ((60, 58, 541), 2, (3, 3, 2, 3, 5, 9)), ((56, 58, 706), 4, (3, 0, 2, 3, 5, 9))])
def test_long_rows_match_oracle(oracle_built, cuda_device, shape, order, pml):
    """Rows that need workgroups of more than 256 threads; on the last two grids in the adjoint alone."""
    h = oracle_built
    print(f"[gpu row sweeps] long rows {shape} {order}", flush=True)
    p = h.make_problem(*shape, order=order, nt=5, nshot=1, nsrc=2, nrx=4, seed=53, pml=pml, d=(0.02, 0.017, 0.015))
    p.src_loc[0, 0] = [shape[0] // 2, shape[1] // 2, shape[2] // 2]
    p.rx_loc[0, 0] = [shape[0] // 2, 1 + shape[1] // 2, shape[2] - 3]
    cpu = h.run_cpu(p, "oracle")
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad


@pytest.mark.parametrize("NZ,order", [(261, 4), (327, 2)])
def test_receivers_on_whole_rows_match_oracle(oracle_built, cuda_device, NZ, order):
    """More receivers on the rows of a workgroup than its live wavefronts have threads; some of its wavefronts idle."""
    h = oracle_built
    print(f"[gpu row sweeps] receivers on whole rows {NZ} {order}", flush=True)
    rows = [(1, 20), (20, 20), (20, 21), (20, 22), (21, 1), (41, 40)]
    cells = [(i, j, k) for i, j in rows for k in range(NZ)] + [(20, 20, 33)] * 3
    p = h.make_problem(44, 42, NZ, order=order, nt=4, nshot=1, nsrc=1, nrx=len(cells), seed=59, pml=(4, 3, 4, 5, 6, 4),
                       d=(0.02, 0.017, 0.015))
    p.src_loc[0, 0] = [20, 21, 40]
    p.rx_loc = np.array([cells], np.int32)
    cpu = h.run_cpu(p, "oracle")
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad
