"""The one-pass value checks (deepgpr_amd/csrc/dgx_checks.hip) against the same
checks as torch reductions: sizes below, at and above a workgroup's share, both
integer widths, extremes at the first and last cell, NaN and infinities, and
coordinates on and outside the grid. Inputs that the kernel does not take keep
the torch reductions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(dev, shape, itype, seed):
    gen = torch.Generator().manual_seed(seed)
    er = (1.0 + 9.0 * torch.rand(shape, generator=gen)).to(dev)
    se = (0.1 * torch.rand(shape, generator=gen)).to(dev)
    mr = (0.5 + torch.rand(shape, generator=gen)).to(dev)
    wave = torch.randn((2, 37, 1), generator=gen).to(dev)
    top = torch.tensor(shape) - 1
    src = torch.stack([torch.zeros(3), top.float(), top.float() // 2]).long()[None].to(device=dev, dtype=itype)
    rx = torch.stack([top, top // 3])[None].to(device=dev, dtype=itype)
    return [er, se, mr, wave, src, rx]


def _both(m, monkeypatch, args):
    native = m._native_scalars(*args)
    with monkeypatch.context() as c:
        c.setattr(m, "_native_scalars", lambda *a: None)
        torch_way = m._device_scalars(*args)
    return native, torch_way


@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 3, 1), (16, 16, 1), (45, 47, 1), (33, 65, 131)])
@pytest.mark.parametrize("itype", [torch.int32, torch.int64])
def test_native_checks_equal_torch_reductions(cuda_device, monkeypatch, shape, itype):
    from deepgpr_amd.preprocessing import model_setup as m
    print(f"[gpu checks] {shape} {itype}", flush=True)
    args = _inputs(cuda_device, shape, itype, 5)
    args[0].view(-1)[-1], args[1].view(-1)[0], args[2].view(-1)[-1] = 0.25, -0.125, -2.0
    args[1].view(-1)[-1] = 7.0
    native, want = _both(m, monkeypatch, args)
    assert native == want
    for k, name in ((0, "finite_er"), (1, "finite_se"), (2, "finite_mr"), (3, "finite_wave")):
        for bad in (float("nan"), float("inf"), float("-inf")):
            broken = [t.clone() for t in args]
            broken[k].view(-1)[-1] = bad
            native, want = _both(m, monkeypatch, broken)
            assert native[name] == want[name] == 0.0, (name, bad)
            for other in ("finite_er", "finite_se", "finite_mr", "finite_wave", "inside_src", "inside_rx"):
                assert native[other] == want[other], (name, bad, other)
    for k, name in ((4, "inside_src"), (5, "inside_rx")):
        for axis in range(3):
            for bad in (-1, shape[axis]):
                broken = [t.clone() for t in args]
                broken[k][0, -1, axis] = bad
                native, want = _both(m, monkeypatch, broken)
                assert native == want and native[name] == 0.0, (name, axis, bad)


def test_other_inputs_keep_the_torch_reductions(cuda_device):
    from deepgpr_amd.preprocessing import model_setup as m
    args = _inputs(cuda_device, (8, 6, 1), torch.int32, 3)
    assert m._native_scalars(*args) is not None
    for k, t in ((4, args[4].float()), (5, args[5].to(torch.int16)), (0, args[0].transpose(0, 1)),
                 (0, args[0].double())):
        other = list(args)
        other[k] = t
        assert m._native_scalars(*other) is None
    assert m._native_scalars(*(t.cpu() for t in args)) is None
