"""The 2D Ez-TM strip kernels (deepgpr_amd/csrc/dgx_tm2d_strip.hip: several
steps a launch) against the CPU oracle, bit for bit: every shape (few
workgroups and many, one shot and several), grids smaller than a tile and with
owned ranges that end inside, at and just past a tile edge, step counts with
and without a remainder, unequal spacing and CPML widths, faces without CPML,
PEC cells, every history that the 2D path keeps, and sources and coincident
receivers in margins, on tile corners, in the CPML and on the grid's edges."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TM2D = 1 << 6
INACTIVE_PHI = (0, 3, 4, 7, 8, 11, 12, 15)
CASES = [
    # (NX, NY, order, nt, nshot, S, storage, mode, pml, d, pec)
    (14, 9, 2, 17, 1, 1, "e_only", 2, (1, 1, 1, 2), (0.02, 0.02), False),
    (19, 23, 4, 8, 2, 1, "f32", 3, (3, 2, 4, 3), (0.02, 0.013), True),
    (33, 49, 2, 8, 2, 3, "f32", 3, (4, 5, 0, 6), (0.017, 0.02), True),
    (48, 96, 2, 16, 1, 2, "bf16", 3, (0, 0, 0, 0), (0.02, 0.02), False),
    (64, 97, 2, 13, 3, 1, "f16", 2, (10, 9, 12, 11), (0.02, 0.02), True),
    (43, 93, 4, 10, 1, 2, "bf16", 2, (0, 6, 7, 0), (0.02, 0.017), False),
    (81, 104, 4, 7, 7, 1, "e_only", 2, (9, 10, 8, 10), (0.02, 0.02), False),
    (101, 157, 4, 7, 9, 3, "f32", 3, (5, 3, 6, 4), (0.02, 0.016), True),
    (61, 209, 2, 14, 14, 1, "e_only", 2, (10, 10, 10, 10), (0.02, 0.02), False),
    (100, 105, 2, 11, 17, 2, "bf16", 3, (6, 0, 5, 7), (0.018, 0.02), True),
    (61, 209, 4, 5, 26, 1, "bf16", 2, (6, 9, 10, 5), (0.02, 0.02), False),
    (64, 105, 2, 8, 43, 2, "f32", 3, (6, 9, 10, 5), (0.02, 0.019), True),
    (52, 62, 2, 9, 1, 1, "e_only", 3, (7, 6, 5, 8), (0.02, 0.02), False),
    (46, 38, 4, 7, 3, 1, "f16_e", 3, (6, 5, 7, 3), (0.02, 0.018), True),
    (61, 209, 2, 11, 7, 1, "e_only", 2, (10, 10, 9, 10), (0.02, 0.018), True),
    (81, 104, 4, 7, 9, 1, "f32", 3, (9, 10, 8, 10), (0.02, 0.02), False),
    (64, 81, 2, 25, 4, 1, "f32", 2, (10, 9, 12, 11), (0.02, 0.02), True),
    (41, 83, 4, 9, 6, 2, "bf16", 3, (3, 6, 7, 4), (0.02, 0.017), False),
    (300, 700, 2, 9, 1, 2, "f32", 3, (10, 7, 9, 10), (0.02, 0.02), True),
    (251, 731, 4, 5, 1, 1, "e_only", 2, (10, 7, 9, 10), (0.02, 0.021), False),
]


def _storage(h, name):
    return {"f32": 0, "e_only": h.RHS_FROM_E, "f16": h.KIND_F16, "bf16": h.KIND_BF16,
            "f16_e": h.KIND_F16 | h.RHS_FROM_E}[name]


def _problem(h, case):
    NX, NY, order, nt, nshot, S, st, mode, pml, d, pec = case
    p = h.make_problem(NX, NY, 2, order=order, nt=nt, nshot=nshot, nsrc=4, nrx=7, seed=31, pml=pml + (0, 0),
                       d=d + (0.02,), pec=pec)
    # the 2D TM contract: Ex, Ey, Hz and their CPML auxiliaries start at zero
    for arrs, idx in ((p.E0, (0, 1)), (p.H0, (2,)), (p.lam0, (0, 1, 5))):
        for k in idx:
            arrs[k] = np.zeros_like(arrs[k])
    for k in INACTIVE_PHI:
        p.phi0[k] = np.zeros_like(p.phi0[k])
        p.lam0[6 + k] = np.zeros_like(p.lam0[6 + k])
    p.mode, p.S = mode, S
    p.storage_type = _storage(h, st)
    for s in range(nshot):
        p.src_loc[s, 0] = [NX // 2, NY // 2, 0]
        p.src_loc[s, 1] = [min(16 + s % 3, NX - 2), min(47 + s % 2, NY - 2), 0]
        p.src_loc[s, 2] = p.src_loc[s, 0]
        p.src_loc[s, 3] = [1, NY - 2, 0]
        spots = [[NX // 2, NY // 2], [NX // 2, NY // 2], [0, 0], [NX - 2, 1], [min(20, NX - 2), min(52, NY - 2)],
                 [min(19, NX - 2), min(51, NY - 2)], [NX // 3, NY - 2]]
        for r, (i, j) in enumerate(spots):
            p.rx_loc[s, r] = [i, j, 0]
    return p


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}-o{c[2]}-n{c[4]}-{c[6]}")
def test_strips_match_oracle_bitwise(oracle_built, cuda_device, monkeypatch, case):
    h = oracle_built
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_TILE_ROWS", raising=False)
    print(f"[gpu strips] {case}", flush=True)
    p = _problem(h, case)
    cpu = h.run_cpu(p, "oracle")
    p.storage_type |= TM2D
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, h.KEYS_FWD + ("g_src", "g_eps", "g_sig"))
    assert not bad, bad
    for k in [2, 3, 4] + [6 + k for k in range(24) if k not in INACTIVE_PHI]:
        assert np.array_equal(gpu["L"][k], cpu["L"][k]), k
    assert np.array_equal(gpu["E_saved"], cpu["E_saved"])
    assert np.array_equal(gpu["R_saved"], cpu["R_saved"])



@pytest.mark.parametrize("case", [(19, 23, 2, 75, 2, 1, "f32", 2), (43, 57, 4, 71, 5, 2, "bf16", 3),
                                  (30, 41, 4, 40, 9, 1, "e_only", 2), (47, 38, 2, 101, 8, 3, "f16", 3)],
                         ids=lambda c: f"{c[0]}x{c[1]}-o{c[2]}-nt{c[3]}-n{c[4]}")
def test_held_material_terms_are_summed_in_order(oracle_built, cuda_device, monkeypatch, case):
    """Terms of several launches wait for one sum: more saved steps than the buffer holds, odd numbers of them left,
    shots below, at and above the eight that the sum loads at once."""
    h = oracle_built
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_TILE_ROWS", raising=False)
    print(f"[gpu strips] held terms {case}", flush=True)
    p = _problem(h, case + ((4, 3, 5, 4), (0.02, 0.018), True))
    cpu = h.run_cpu(p, "oracle")
    p.storage_type |= TM2D
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, h.KEYS_FWD + ("g_src", "g_eps", "g_sig"))
    assert not bad, bad


def _request(rid, shape, nt, order, nshot, gradient, seed):
    from deepgpr_amd.serving import SolveRequest
    gen = torch.Generator().manual_seed(seed)
    eps = 1.0 + 8.0 * torch.rand(shape, generator=gen)
    sig = 0.01 * torch.rand(shape, generator=gen)
    t = torch.arange(nt, dtype=torch.float32) * 3e-11
    a2 = (torch.pi * 4e8 * (t - 2.5e-9)) ** 2
    wave = ((1 - 2 * a2) * torch.exp(-a2)).reshape(1, nt, 1)
    src = torch.tensor([[[shape[0] // 2 - s, shape[1] // 2, 0]] for s in range(nshot)])
    rx = torch.tensor([[[5 + 3 * (r % 4), 2 + 5 * r, 0] for r in range(9)] for _ in range(nshot)])
    return SolveRequest(eps, sig, wave, src, rx, 0.02, 3e-11, fdtd_order=order, pmlthick=8, gradient=gradient,
                        rid=rid, options={"mode": 2, "wavefield_rhs_history": "reconstructed",
                                              "wavefield_storage_dtype": torch.bfloat16 if rid % 3 == 1
                                              else torch.float32})


def test_batch_of_strips_equals_one_step_launches(cuda_device, monkeypatch):
    """Instances that run several steps a launch beside some that cannot (order
    8, two shots), in both phases at once and with steps that end inside a
    launch: the bits of the same solves one at a time, one step a launch."""
    from deepgpr_amd import batch, serving
    shapes = [(60, 52), (91, 77), (52, 104), (110, 47), (48, 48), (75, 130)]
    reqs = [_request(k, shapes[k % 6], 37 + 8 * (k % 5), (2, 4, 4, 2, 8, 4, 2)[k % 7], 2 if k % 6 == 5 else 1,
                     k % 4 != 3, 900 + k) for k in range(13)]
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", "0")
    alone = serving.run_sequential(reqs, cuda_device)["results"]

    def batched(strips):
        monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", strips)
        with batch.BatchSolver(cuda_device) as solver:
            ids = {solver.add(r): r.rid for r in reqs[:7]}
            solver.step(40)  # joins while some are in their adjoint
            ids.update({solver.add(r): r.rid for r in reqs[7:]})
            solver.run(11)
            return {ids[n]: solver.result(n) for n in ids}

    for strips in ("1", "0"):
        print(f"[gpu strips] batch, strips {strips}", flush=True)
        got = batched(strips)
        for r in reqs:
            a = alone[r.rid]
            res = got[r.rid]
            assert torch.equal(res[0], a.receivers), (strips, r.rid)
            if r.gradient:
                assert torch.equal(res[1], a.grad_eps_r), (strips, r.rid)
                assert torch.equal(res[2], a.grad_sigma), (strips, r.rid)


@pytest.mark.parametrize("order", [2, 4])
def test_signs_of_zeros_equal_the_one_step_kernels(oracle_built, cuda_device, monkeypatch, order):
    """Fields and auxiliaries of zeros of either sign: quotients of -0 by the grid spacing keep their sign, so both
    kernels leave the same bits, those of the zeros included."""
    h = oracle_built
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_TILE_ROWS", raising=False)
    print(f"[gpu strips] signs of zeros, order {order}", flush=True)
    p = _problem(h, (57, 71, order, 3, 2, 1, "f32", 2, (9, 8, 7, 10), (0.02, 0.017), False))
    rng = np.random.default_rng(order)
    for arrs in (p.E0, p.H0, p.phi0):
        for k, a in enumerate(arrs):
            arrs[k] = np.where(rng.random(a.shape) < 0.5, np.float32(-0.0), np.float32(0.0))
    for arrs, idx in ((p.E0, (0, 1)), (p.H0, (2,)), (p.phi0, INACTIVE_PHI)):
        for k in idx:
            arrs[k] = np.zeros_like(arrs[k])
    p.wave = np.zeros_like(p.wave)
    p.storage_type |= TM2D
    strips = h.run_gpu(p, backward=False, api="dgx")
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", "0")
    steps = h.run_gpu(p, backward=False, api="dgx")
    for key in ("E", "H", "phi"):
        for k, (a, b) in enumerate(zip(strips[key], steps[key])):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (key, k)


@pytest.mark.parametrize("NX,NY,order,nt,nshot", [(45, 70, 2, 26, 1), (45, 70, 4, 9, 2), (61, 209, 2, 9, 14),
                                                  (50, 90, 2, 8, 48), (50, 90, 4, 5, 40)])
def test_many_points_match_oracle(oracle_built, cuda_device, monkeypatch, NX, NY, order, nt, nshot):
    """Sources on a block of cells and along both axes, several on one cell, and receivers on every second cell: more
    points of a wavefront than it takes one after the other, and more receiver cells than its lanes."""
    h = oracle_built
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_TILE_ROWS", raising=False)
    print(f"[gpu strips] many points {NX}x{NY} o{order} n{nshot}", flush=True)
    p = _problem(h, (NX, NY, order, nt, nshot, 1, "f32", 2, (5, 4, 6, 7), (0.02, 0.018), False))
    cells = [(i, j) for i in range(9, 21) for j in range(30, 50)] + [(17, j) for j in range(1, NY - 1, 3)]
    cells += [(i, 40) for i in range(1, NX - 1, 2)] + [(12, 33)] * 7 + [(30, 60)] * 6
    rx = [(i, j) for i in range(0, NX - 1) for j in range(i % 2, NY - 1, 2)] + [(12, 34)] * 3
    rng = np.random.default_rng(7)
    p.src_loc = np.array([[[(i + s) % (NX - 1), j, 0] for i, j in cells] for s in range(nshot)], np.int32)
    p.rx_loc = np.array([[[i, j, 0] for i, j in rx] for _ in range(nshot)], np.int32)
    p.wave = rng.standard_normal((len(cells), nt)).astype(np.float32)
    p.data_grad = (1e-3 * rng.standard_normal((nshot, nt, len(rx)))).astype(np.float32)
    cpu = h.run_cpu(p, "oracle")
    p.storage_type |= TM2D
    gpu = h.run_gpu(p, api="dgx")
    bad = h.bitwise_diff(gpu, cpu, h.KEYS_FWD + ("g_src", "g_eps", "g_sig"))
    assert not bad, bad
