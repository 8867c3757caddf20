"""INT8 histories in 4x4x4 tiles (four tiles along z a wavefront) against the CPU
oracle, byte for byte: tile counts along z of every remainder by four, boxes
that end inside a tile on each axis, E and R frames and several shots. Fields
with NaN, infinities and values too small for a scale, where the C oracle's
conversion is undefined, are checked against the codec written out in numpy:
the maximum in the pairing of a 64-wide tree, NaN stored as -127."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # (NX, NY, NZ, nshot, S, e_only, special values)
    (17, 13, 18, 1, 1, False, False),
    (14, 19, 22, 2, 2, False, True),
    (18, 14, 27, 1, 1, True, False),
    (13, 18, 33, 2, 1, True, True),
    (21, 16, 50, 1, 3, False, True),
    (15, 15, 66, 1, 1, False, False),
]


def _encode(v):
    """Payload and scales of one (nx, ny, nz) frame."""
    n = v.shape
    t = [(k + 3) // 4 for k in n]
    full = np.zeros([4 * k for k in t], np.float32)
    full[:n[0], :n[1], :n[2]] = v
    tiles = full.reshape(t[0], 4, t[1], 4, t[2], 4).transpose(0, 2, 4, 1, 3, 5).reshape(*t, 64)
    with np.errstate(all="ignore"):
        m = np.where(tiles < 0, -tiles, tiles)
        for stride in (32, 16, 8, 4, 2, 1):
            a, b = m[..., :stride], m[..., stride:2 * stride]
            m = np.where(b > a, b, a)
        peak = m[..., 0]
        scale = np.where(peak >= np.float32(1e-30), peak / np.float32(127), np.float32(1)).astype(np.float32)
        r = np.fmin(np.fmax(np.rint(tiles / scale[..., None]), -127), 127)
    q = r.astype(np.int8).reshape(*t, 4, 4, 4).transpose(0, 3, 1, 4, 2, 5).reshape(full.shape)
    return q[:n[0], :n[1], :n[2]], scale


def _check_first_frame(packed, e0, nshot, frames):
    """Frame 0 of a packed E history holds the initial field."""
    box = [k - 1 for k in e0[0].shape[1:]]
    cells, tiles = int(np.prod(box)), int(np.prod([(k + 3) // 4 for k in box]))
    payload = (3 * frames * nshot * cells + 3) // 4 * 4
    q = packed[:3 * frames * nshot * cells].view(np.int8).reshape(3, frames, nshot, *box)
    scale = packed[payload:payload + 4 * 3 * frames * nshot * tiles].view(np.float32).reshape(3, frames, nshot, tiles)
    for comp in range(3):
        for s in range(nshot):
            want, ws = _encode(e0[comp][s, :box[0], :box[1], :box[2]])
            assert np.array_equal(q[comp, 0, s], want), (comp, s)
            assert np.array_equal(scale[comp, 0, s], ws.reshape(-1)), (comp, s)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-n{c[3]}-S{c[4]}")
def test_int8_tiles_match_oracle(oracle_built, cuda_device, case):
    h = oracle_built
    NX, NY, NZ, nshot, S, e_only, special = case
    print(f"[gpu int8 tiles] {case}", flush=True)
    p = h.make_problem(NX, NY, NZ, order=2, nt=5, nshot=nshot, nsrc=2, nrx=3, seed=23, pml=(3, 2, 3, 3, 2, 3))
    p.mode, p.S = 3, S
    p.storage_type = h.int8_storage_type((4, 4, 4)) | (h.RHS_FROM_E if e_only else 0)
    if special:
        e = p.E0[2].reshape(nshot, NX, NY, NZ)
        e[0, 5, 6, 7] = np.nan
        e[-1, 9, 9, 4] = np.inf
        e[0, 1, 2, 13] = -np.inf
        e[-1, 8:12, 8:12, 8:12] = 1e-37
    gpu = h.run_gpu(p, backward=not special, api="dgx")
    _check_first_frame(np.ascontiguousarray(gpu["E_saved"]).view(np.uint8).reshape(-1),
                       [a.reshape(nshot, NX, NY, NZ) for a in p.E0], nshot, (p.nt + S - 1) // S)
    if special:
        return
    cpu = h.run_cpu(p, "oracle", backward=True)
    assert np.array_equal(gpu["E_saved"], cpu["E_saved"])
    assert np.array_equal(gpu["R_saved"], cpu["R_saved"])
    bad = h.bitwise_diff(gpu, cpu, list(h.KEYS_FWD) + list(h.KEYS_BWD))
    assert not bad, bad
