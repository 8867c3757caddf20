"""dgx_scratch_bytes of 2D gradients (host logic only, no GPU): the per-shot
material terms that the adjoint holds between its sums."""
import ctypes

import pytest
import torch

from deepgpr_amd.native.bridge import build_solve
from deepgpr_amd.native.loader import get_library

_T = torch.zeros(8)  # stands in for every array: only the sizes are read


def _scratch(nx, ny, nshot, order, nt=100, S=1, grad=1, pml=(0, 0, 0, 0, 0, 0)):
    args = dict(nx_fields=nx, ny_fields=ny, nz_fields=2, nshot=nshot, nt=nt, fdtd_order=order, pml=list(pml),
                dx=0.02, dy=0.02, dz=0.02, dt=1e-11, storage_type=1 << 6, source_component=2, receiver_component=2,
                sampling_interval=S, fwi_mode=2, nsource=1, nreceiver=1, save_model_history=1, accumulate_fp64=0,
                eps_r_requires_grad=grad, sigma_requires_grad=0, E=[_T] * 3, H=[_T] * 3, eps_r_pad=_T, sigma_pad=_T,
                mu_r_pad=_T, update_coeff=[_T] * 6, source_location=_T, source_waveform=_T, receiver_location=_T,
                receiver_data=_T, data_grad=_T, grad_eps_r=_T, grad_sigma=_T, grad_source=_T)
    lib = get_library()
    solve = build_solve(args)
    back = lib.dgx_scratch_bytes(ctypes.byref(solve), 1)
    assert back >= 0, lib.dgx_last_error()
    return back


@pytest.mark.parametrize("nx,ny,nshot,order,nt,S,saves", [
    (101, 121, 5, 4, 100, 1, 32),    # as many as one sum takes
    (101, 121, 5, 4, 100, 4, 25),    # as many as there are
    (101, 121, 5, 4, 3, 2, 2),       # at least two
    (343, 265, 5, 4, 400, 1, 9),     # what fits 32 MiB
    (442, 242, 20, 2, 400, 1, 2),    # more than 32 MiB already
    (101, 121, 1, 2, 100, 1, 0),     # one shot is summed in registers
    (101, 121, 5, 8, 100, 1, 2),     # one step a launch
    (101, 121, 1, 8, 100, 1, 2)])
def test_terms_of_a_2d_gradient(monkeypatch, nx, ny, nshot, order, nt, S, saves):
    monkeypatch.delenv("DEEPGPR_AMD_TM2D_STRIPS", raising=False)
    assert _scratch(nx, ny, nshot, order, nt, S) == saves * 2 * nshot * (nx - 1) * (ny - 1) * 4
    assert _scratch(nx, ny, nshot, order, nt, S, grad=0) == 0


def test_terms_of_the_one_step_kernels(monkeypatch):
    monkeypatch.setenv("DEEPGPR_AMD_TM2D_STRIPS", "0")
    assert _scratch(101, 121, 5, 4) == 2 * 2 * 5 * 100 * 120 * 4
