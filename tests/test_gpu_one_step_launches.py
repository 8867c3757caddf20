"""The one-step 2D Ez-TM kernels under solves that by default run several steps
a launch: the tile tuner, the graphs of forward solves and the graphs of batches
still give the bits of the strip kernels (DEEPGPR_AMD_TM2D_STRIPS=0 keeps one
step a launch), and batches whose instances have one step a launch by
themselves (order 8, two shots) replay graphs by default."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.dirname(__file__))
from gpu_helpers import capture  # noqa: E402

pytestmark = pytest.mark.gpu


def _solve(dev, nx, ny, order, nshot, gradient):
    import deepgpr_amd as dg
    gen = torch.Generator().manual_seed(nx + order)
    nt = 75
    eps = (1.0 + 8.0 * torch.rand(nx, ny, generator=gen)).to(dev).requires_grad_(gradient)
    sig = (0.01 * torch.rand(nx, ny, generator=gen)).to(dev).requires_grad_(gradient)
    t = torch.arange(nt, dtype=torch.float32) * 3e-11
    a2 = (torch.pi * 4e8 * (t - 2.5e-9)) ** 2
    wave = ((1 - 2 * a2) * torch.exp(-a2)).reshape(1, nt, 1).to(dev)
    src = torch.tensor([[[20, 10 + 30 * s, 0]] for s in range(nshot)], device=dev)
    rx = torch.tensor([[[25, 5 + 9 * r, 0] for r in range(8)] for _ in range(nshot)], device=dev)
    kw = dict(dx=0.02, dt=3e-11, source_amplitudes=wave, source_location=src, receiver_location=rx, eps_r=eps,
              sigma=sig, fdtd_order=order, mode=2)
    if not gradient:
        with torch.no_grad():
            out = dg.compute(dev, save_wavefield_history=False, **kw)
        return [out[-1].clone()] + [t.clone() for t in out[1] + out[2]]
    out = dg.compute(dev, gradient_accumulator="float32", **kw)
    (out[-1] ** 2).sum().backward()
    return [out[-1].detach().clone(), eps.grad.clone(), sig.grad.clone()]


@pytest.mark.parametrize("nx,order,nshot", [(131, 2, 2), (137, 4, 3), (143, 8, 1)])
def test_tuner_of_the_one_step_kernels(cuda_device, monkeypatch, nx, order, nshot):
    from deepgpr_amd.native.loader import get_library
    print(f"[gpu one step] tuner, order {order}", flush=True)
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_TILE_ROWS", raising=False)
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_TUNE", raising=False)
    strips = _solve(cuda_device, nx, 118, order, nshot, True)  # several steps a launch at orders 2 and 4
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", "0")
    lib = get_library()
    lib.dgx_set_kernel_timing(1)
    calls = capture(monkeypatch)
    tuned = _solve(cuda_device, nx, 118, order, nshot, True)
    torch.cuda.synchronize()
    lib.dgx_set_kernel_timing(0)
    fin = calls[0][1]
    assert fin["storage_type"] & (1 << 6)  # the fused 2D Ez-TM path
    rows = lib.dgx_tm2d_tile_rows_tuned(fin["nx_fields"], fin["ny_fields"], fin["nshot"], order, 1)
    assert rows in (4, 8, 16), rows
    assert _launches(lib, "tm_step_fwd") == 75 and _launches(lib, "tm_strip_fwd") == 0
    for a, b in zip(strips, tuned):
        assert torch.equal(a, b)
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_TUNE", "0")
    for a, b in zip(_solve(cuda_device, nx, 118, order, nshot, True), tuned):
        assert torch.equal(a, b)


def _launches(lib, name):
    import ctypes
    for k in range(64):
        got = lib.dgx_kernel_name(k)
        if not got:
            break
        if got.decode() == name:
            ms, n = ctypes.c_double(), ctypes.c_longlong()
            lib.dgx_kernel_timing(k, ctypes.byref(ms), ctypes.byref(n))
            return n.value
    raise AssertionError(name)


@pytest.mark.parametrize("order", [2, 4])
def test_forward_graphs_of_the_one_step_kernels(cuda_device, monkeypatch, order):
    """75 steps: two replays of 32 steps and a remainder, against strips; three times, with eager work between."""
    print(f"[gpu one step] graphs, order {order}", flush=True)
    strips = _solve(cuda_device, 70, 90, order, 2, False)
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", "0")
    for rep in range(3):
        got = _solve(cuda_device, 70, 90, order, 2, False)
        scratch = torch.randn(1 << 16, device=cuda_device).cumsum(0)
        torch.cuda.synchronize()
        assert torch.isfinite(scratch).all()
        for a, b in zip(strips, got):
            assert torch.equal(a, b), rep
    assert strips[0].abs().max() > 0


def _requests(order, nshot, seed):
    from deepgpr_amd.serving import SolveRequest
    out = []
    for k in range(6):
        gen = torch.Generator().manual_seed(seed + k)
        shape, nt = ((60, 52), (91, 77), (52, 104))[k % 3], 70 + 11 * k
        eps = 1.0 + 8.0 * torch.rand(shape, generator=gen)
        sig = 0.01 * torch.rand(shape, generator=gen)
        t = torch.arange(nt, dtype=torch.float32) * 3e-11
        a2 = (torch.pi * 4e8 * (t - 2.5e-9)) ** 2
        wave = ((1 - 2 * a2) * torch.exp(-a2)).reshape(1, nt, 1)
        src = torch.tensor([[[shape[0] // 2 - s, shape[1] // 2, 0]] for s in range(nshot)])
        rx = torch.tensor([[[5 + 3 * (r % 4), 2 + 5 * r, 0] for r in range(9)] for _ in range(nshot)])
        out.append(SolveRequest(eps, sig, wave, src, rx, 0.02, 3e-11, fdtd_order=order, pmlthick=8, gradient=True,
                                rid=k, options={"mode": 2}))
    return out


@pytest.mark.parametrize("order,nshot,strips", [(2, 1, "0"), (4, 1, "0"), (4, 2, "1"), (8, 1, "1")])
def test_batch_graphs_of_the_one_step_kernels(cuda_device, monkeypatch, order, nshot, strips):
    from deepgpr_amd import batch, serving
    print(f"[gpu one step] batch graphs, order {order}, shots {nshot}", flush=True)
    reqs = _requests(order, nshot, 500)
    alone = serving.run_sequential(reqs, cuda_device)["results"]
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", strips)

    def batched(graphs):
        monkeypatch.setenv("DEEPGPR_AMD_BATCH_GRAPHS", graphs)
        with batch.BatchSolver(cuda_device) as solver:
            ids = {solver.add(r): r.rid for r in reqs[:4]}
            solver.step(64)  # whole graphs while no instance changes phase
            ids.update({solver.add(r): r.rid for r in reqs[4:]})  # joins rebuild the table
            solver.run(64)
            return {ids[n]: solver.result(n) for n in ids}

    for graphs in ("1", "0"):
        got = batched(graphs)
        for r in reqs:
            a = alone[r.rid]
            for x, y in zip(got[r.rid], (a.receivers, a.grad_eps_r, a.grad_sigma)):
                assert torch.equal(x, y), (graphs, r.rid)
