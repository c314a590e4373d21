"""calc_trajectory with more rows than the 256 MiB cache holds.

There a lane of a wave stays within 16 steps of the wave's last one, and a
wave's points all start together.  Just above that size, a point and two points
a lane, with points at rest (on walls), calm ones and ones that change
cell at most steps in each wave: every row against the oracle, bit for bit
(cpab/gpu/calc_2Dto2D.cu:499-556)."""
import numpy as np
import pytest

from cpabdiffeo_amd.calcs import Calcs
from test_gpu_simple_walls import tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,tess,nCs,extent,nT", [
    (1, "II", (8,), (1.0,), 240), (2, "I", (4, 4), (1.0, 1.0), 240), (2, "II", (5, 3), (640.0, 480.0), 240),
    (3, "I", (2, 2, 2), (1.0, 1.0, 1.0), 240), (1, "II", (8,), (1.0,), 60), (2, "I", (3, 5), (1.0, 1.0), 28)])
def test_rows_equal_the_oracle(gpu, orc, dim, tess, nCs, extent, nT):
    torch = gpu
    nS, dt = 3 if nT > 33 else 4, 1.0 / nT
    n = (256 << 20) // (8 * dim * nT) + 70
    print("[gpu] trajectory of", n, "points", dim, tess, nCs, flush=True)
    rng = np.random.default_rng(23)
    incs = [e / k for e, k in zip(extent, nCs)]
    nC = int(np.prod(nCs)) * (1 if tess == "II" else (4 if dim == 2 else 5))
    geom = {"dim": dim, "tess": 1 if tess == "I" else 2, "nCs": list(nCs), "incs": incs}
    A = tables(dim, nC, incs, extent, 3.0, rng)
    A[rng.random(nC) < 0.25] = 0.0
    sA, T = orc.prep(dim, A, 1, dt)
    pts = rng.random((n, dim))
    corners = rng.random(n) < 0.1
    pts[corners] = np.round(pts[corners])
    pts = np.ascontiguousarray(pts * np.array(extent))
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    traj = Calcs(nC, np.float64, dim, dim, tess).calc_trajectory(None, None, dev(T), dev(sA), dev(pts), dt, nT, nS, dim, dim,
                                                                list(nCs), incs)
    assert traj.numel() * 8 > 256 << 20
    want = orc.calc_trajectory(geom, pts, T, sA, dt, nT, nS)
    assert np.array_equal(traj.cpu().numpy(), want)
