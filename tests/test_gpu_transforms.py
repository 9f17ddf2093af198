"""The transforms around the multiply-accumulate at the lengths where their
passes change: every radix and remainder of the reduced grids' workgroup-level
transforms, prime last passes, rows of several frames staged through LDS, even
and odd lengths; against the FP64 oracle.

Tolerance 1e-6 relative L2: about 30 fp32 roundings on the way of a value
(2^-24 each, random: 3e-7) and the multiply-accumulate's 23-bit operands
(2e-7)."""
import numpy as np
import pytest

from flfhip.psfmatrix import MemoryHMatrix
from oracle import projector as oproj

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _check(N, Y, X, sides, T):
    from flfhip.projector import Projector_hip
    rng = np.random.default_rng(N * 1000 + Y + 3 * X + T)
    h, nz = (N + 1) // 2, len(sides)
    hm = MemoryHMatrix([rng.random((h, h, s, s)).astype(np.float32) for s in sides],
                       [rng.random((h, h, s, s)).astype(np.float32) for s in sides])
    vol = rng.random((nz, T, Y, X)).astype(np.float32)
    img = rng.random((T, Y, X)).astype(np.float32)
    print("N %d %dx%d T %d" % (N, Y, X, T), flush=True)
    proj = Projector_hip()
    fwd = proj.ForwardProjectACC(hm, vol, range(nz))
    bwd = proj.BackwardProjectACC(hm, img, range(nz))

    def err(a, b):
        return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))

    for t in {0, T - 1}:
        assert err(fwd[t], sum(oproj.project_special(vol[z, t], hm.Hcc(z, False)) for z in range(nz))) < 1e-6
        for z in range(nz):
            assert err(bwd[z, t], oproj.project_special(img[t], hm.Hcc(z, True))) < 1e-6


# reduced lengths: with Nnum 3 and a PSF of 5, an image of 3 r - 4 has the grid 3 r
@pytest.mark.parametrize("rY,rX", [(r, r) for r in (3, 4, 5, 6, 9, 10, 12, 25, 27, 75, 81, 96, 108, 120, 125, 128)] +
                         [(96, 125), (128, 81), (120, 128), (128, 120), (3, 128), (135, 90)])
def test_reduced_lengths(rY, rX):
    _check(3, 3 * rY - 4, 3 * rX - 4, [5], 1)


@pytest.mark.parametrize("N", [7, 11, 17, 29])
@pytest.mark.parametrize("ny,nx,T", [(4, 4, 1), (4, 5, 3)])
def test_prime_passes(N, ny, nx, T):
    _check(N, N * ny - 8, N * nx - 8, [9], T)


# rows of several frames: 8, 2 x 4, 4 x 2 per workgroup, remainders, a block
# of one frame after a full one; even and odd row lengths in one projection
@pytest.mark.parametrize("Y,X", [(41, 371), (42, 370), (41, 356)])
@pytest.mark.parametrize("T", [2, 3, 4, 5, 8, 9, 11])
def test_staged_rows(Y, X, T):
    _check(3, Y, X, [5, 17], T)
