"""The matrix-core multiply-accumulate (k_mac: fp32 operands split into two
fp16 numbers, 8 frames per workgroup) at the sizes where its tiling has
remainders, against the FP64 oracle, and what its scaling promises exactly.

Tolerance 1e-6 relative L2: the transforms around the kernel round about 30
times in fp32 (2^-24 each, random: 3e-7) and the split keeps 23 bits of each
operand (2e-7)."""
import numpy as np
import pytest

from flfhip.psfmatrix import MemoryHMatrix
from oracle import projector as oproj

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _hm(N, sides, seed):
    rng = np.random.default_rng(seed)
    h = (N + 1) // 2
    return MemoryHMatrix([rng.random((h, h, s, s)).astype(np.float32) for s in sides],
                         [rng.random((h, h, s, s)).astype(np.float32) for s in sides])


def rel_l2(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


# pitches: 3 (fewer spectra than one K step), 5 (an odd number of spectra on
# non-square grids), 13, 19 (two chunks per orbit), 23 and 31 (several table
# batches per plane); frames: one, one short of a block, a block, one over
@pytest.mark.parametrize("N,Y,X,sides,T", [
    (3, 30, 30, [5, 9], 1), (3, 27, 36, [5, 9], 9), (5, 60, 60, [9, 15], 7), (5, 60, 75, [9, 15], 8),
    (13, 78, 78, [13, 27], 2), (13, 78, 91, [13, 27], 1), (15, 90, 90, [15, 31], 8), (15, 75, 105, [15, 31], 17),
    (19, 76, 76, [19, 21], 3), (19, 76, 95, [19, 21], 1), (23, 69, 69, [23], 2), (31, 62, 62, [15], 1),
    (31, 62, 93, [15], 2)])
def test_projections_match_oracle(N, Y, X, sides, T):
    from flfhip.projector import Projector_hip
    hm = _hm(N, sides, seed=N + T)
    rng = np.random.default_rng(N * T + X)
    nz = len(sides)
    vol = rng.random((nz, T, Y, X)).astype(np.float32)
    img = rng.random((T, Y, X)).astype(np.float32)
    proj = Projector_hip()
    print("N %d %dx%d T %d" % (N, Y, X, T), flush=True)
    fwd = proj.ForwardProjectACC(hm, vol, range(nz))
    bwd = proj.BackwardProjectACC(hm, img, range(nz))
    for t in {0, T // 2, T - 1}:
        ef = rel_l2(fwd[t], sum(oproj.project_special(vol[z, t], hm.Hcc(z, False)) for z in range(nz)))
        eb = max(rel_l2(bwd[z, t], oproj.project_special(img[t], hm.Hcc(z, True))) for z in range(nz))
        print("  frame %d forward %.2e backward %.2e" % (t, ef, eb), flush=True)
        assert ef < 1e-6 and eb < 1e-6


@pytest.mark.parametrize("Y,X", [(90, 90), (75, 105)])
def test_frames_and_scales_are_exact(Y, X):
    """A frame's result does not depend on the other frames of its block, bit
    for bit; a power of two times the input gives that power of two times the
    result; NaN and infinity stay in their frame."""
    from flfhip.projector import Projector_hip
    hm = _hm(15, [15, 31], seed=3)
    p = Projector_hip()
    p.prepare(hm, 1, Y, X, frames_capacity=9)
    p.set_option("fwd_split", 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    vol = torch.rand((2, 9, Y, X), generator=g, device="cuda")
    img = torch.rand((9, Y, X), generator=g, device="cuda")
    f, b = p.forward_device(hm, vol), p.backward_device(hm, img)
    for t in (0, 3, 8):
        v1, i1 = vol[:, t:t + 1].contiguous(), img[t:t + 1].contiguous()
        assert torch.equal(p.forward_device(hm, v1)[0], f[t])
        assert torch.equal(p.backward_device(hm, i1)[:, 0], b[:, t])
        for s in (2.0 ** 90, 2.0 ** -90):
            assert torch.equal(p.forward_device(hm, v1 * s)[0], f[t] * s)
            assert torch.equal(p.backward_device(hm, i1 * s)[:, 0], b[:, t] * s)
    bad = img.clone()
    bad[2, 5, 7] = float("nan")
    bad[4, 9, 1] = float("inf")
    got = p.backward_device(hm, bad)
    for t in range(9):
        if t in (2, 4):
            assert not bool(torch.isfinite(got[:, t]).any())
        else:
            assert torch.equal(got[:, t], b[:, t])
    assert not bool(p.forward_device(hm, torch.zeros_like(vol)).any())
