"""calc_T of a grid from the domain's corner, with and without the corner's own block.

The block is left out where the other blocks fill the chip exactly (256 CUs: a
512 x 512 grid with the tables of 16 x 16 cells, a 512 x 640 one with those of
4 x 4) and for integrations of less than four steps, which also take the points
in index order.  End points and fallback counts against the oracle, bit for bit
(cpab/gpu/calc_2Dto2D.cu:348-408)."""
import numpy as np
import pytest

from cpabdiffeo_amd import configs
from cpabdiffeo_amd.calcs import Calcs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows,cols", [(16, 512, 512), (16, 512, 448), (4, 512, 640), (4, 512, 512)])
@pytest.mark.parametrize("nT,nS", [(1, 5), (3, 40), (4, 40), (20, 10)])
def test_end_points_equal_the_oracle(gpu, orc, n, rows, cols, nT, nS):
    torch = gpu
    print("[gpu] corner room", n, rows, cols, nT, nS, flush=True)
    sp = configs.unit_space((n, n), "I")
    A = (sp.B @ np.random.default_rng(3).normal(size=sp.d)).reshape(sp.nC, 6)
    A /= np.abs(A).max()
    y, x = np.mgrid[0:rows, 0:cols]
    pts = np.ascontiguousarray(np.stack([x.ravel() / cols, y.ravel() / rows], 1))
    sA, T = orc.prep(2, A, 1, 1.0 / nT)
    want, nfb_w, _ = orc.calc_T(sp.tessellation.geom(), pts, T, sA, 1.0 / nT, nT, nS, probe=True)
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    out = torch.full(pts.shape, -7.0, dtype=torch.float64, device="cuda")
    nfb = torch.full((len(pts),), -7, dtype=torch.int32, device="cuda")
    Calcs(sp.nC, np.float64, 2, 2, "I").calc_T(None, None, dev(T), dev(sA), dev(pts), 1.0 / nT, nT, nS, out, 2, 2, sp.nCs,
                                               sp.incs, n_fallback=nfb)
    assert np.array_equal(out.cpu().numpy(), want)
    assert np.array_equal(nfb.cpu().numpy(), nfb_w)
