"""calc_T_simple by stretches without a lookup and by substeps with one.

A wave goes on without lookups while all its points stay in the bounds of
their cells, and takes 3, 7, 15, 31 and then 63 substeps with a lookup each
after several stretches in a row that ended at once.  Grids whose points lie on the walls and
their edges (out of the bounds at every substep), points that change cell at
most substeps, calm ones, and mixed waves; counts of substeps around those of
the sequence.  End points against the oracle, bit for bit
(cpab/gpu/calc_2Dto2D.cu:412-445)."""
import numpy as np
import pytest

from cpabdiffeo_amd.calcs import Calcs

pytestmark = pytest.mark.gpu

CASES = [(1, "II", (8,), (1.0,)), (1, "II", (7,), (3.0,)), (2, "I", (4, 4), (1.0, 1.0)), (2, "I", (3, 5), (640.0, 480.0)),
         (2, "II", (4, 2), (1.0, 1.0)), (2, "II", (5, 3), (1.0, 1.0)), (3, "I", (2, 2, 2), (1.0, 1.0, 1.0)),
         (3, "I", (3, 2, 3), (96.0, 80.0, 64.0)), (3, "II", (3, 4, 2), (1.0, 1.0, 1.0))]
STEPS = [(1, 1), (1, 3), (3, 1), (1, 4), (7, 1), (2, 4), (3, 5), (8, 8), (11, 13), (30, 10)]


def tables(dim, nC, incs, extent, speed, rng):
    """A turn about the domain's centre and a velocity of its own in each cell, up to `speed` increments a unit time."""
    inc, ext = np.array(incs), np.array(extent)
    A = np.zeros((nC, dim, dim + 1))
    L = rng.normal(size=(dim, dim))
    A[:, :, :-1] = speed * 0.3 * (L - L.T) * inc[:, None] / ext[None, :]
    A[:, :, -1] = -A[:, :, :-1] @ (0.5 * ext) + speed * inc * rng.uniform(-1, 1, (nC, dim))
    return A.reshape(nC, -1)


def points(dim, extent, rng):
    m = {1: 130, 2: 12, 3: 6}[dim]
    g = np.stack([x.ravel() for x in np.meshgrid(*[np.linspace(0, 1, m)] * dim, indexing="ij")[::-1]], 1)
    r = rng.random((200, dim))
    mixed = np.where(rng.random((150, dim)) < 0.2, np.round(rng.random((150, dim))), rng.random((150, dim)))
    return np.ascontiguousarray(np.concatenate([g, r, mixed]) * np.array(extent))


@pytest.mark.parametrize("dim,tess,nCs,extent", CASES)
def test_end_points_equal_the_oracle(gpu, orc, dim, tess, nCs, extent):
    torch = gpu
    print("[gpu] calc_T_simple walls", dim, tess, nCs, extent, flush=True)
    rng = np.random.default_rng(17)
    incs = [e / n for e, n in zip(extent, nCs)]
    nC = int(np.prod(nCs)) * (1 if tess == "II" else (4 if dim == 2 else 5))
    geom = {"dim": dim, "tess": 1 if tess == "I" else 2, "nCs": list(nCs), "incs": incs}
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    calcs = Calcs(nC, np.float64, dim, dim, tess)
    pts = points(dim, extent, rng)
    p = dev(pts)
    for speed in (0.0, 0.05, 2.0, 20.0):  # increments a unit time: at rest, calm, some and many changes of cell
        A = tables(dim, nC, incs, extent, speed, rng)
        for nT, nS in STEPS:
            want = orc.calc_T_simple(geom, pts, A, 1.0 / nT, nT, nS)
            for n in (len(pts), 65, 1):
                out = torch.zeros((n, dim), dtype=torch.float64, device="cuda")
                calcs.calc_T_simple(None, None, dev(A), p[:n].contiguous(), 1.0 / nT, nT, nS, out, dim, dim, nCs, incs)
                assert np.array_equal(out.cpu().numpy(), want[:n]), (speed, nT, nS, n)
