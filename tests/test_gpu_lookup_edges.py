"""The lookup for increments that are not powers of two, where it can go wrong.

The cell of a point is decided there from an exact quotient and remainder and
from products with the rounded reciprocal of the increment; IEEE divisions are
only formed next to a decision.  The points here sit on and within a few ulps
of every multiple of the increment, on and next to the diagonals (the planes
of the tetrahedra), at the clamps and outside the domain, and at special
values; the cells must equal the oracle's exactly (cpab/gpu/calc_1Dto1D.cu:
62-65, calc_2Dto2D.cu:38-153, calc_3Dto3D.cu:43-137)."""
import numpy as np
import pytest

from cpabdiffeo_amd.calcs import Calcs

pytestmark = pytest.mark.gpu

SPECIAL = [0.0, -0.0, 5e-324, -5e-324, 1e-310, 1e-300, -1e-300, 1e-17, -1e-17, 1e17, -1e17, 1e300, -1e300, 1.7e308,
           -1.7e308, np.inf, -np.inf, np.nan]


def axis_values(n, inc, rng):
    """Multiples of inc and their neighbours, the clamp, points inside and outside."""
    v = []
    for k in list(range(-2, n + 3)) if n <= 12 else sorted({-1, 0, 1, 2, 3, n // 3, n // 2, n - 2, n - 1, n, n + 1}):
        x = k * inc
        v.append(x)
        lo = hi = x
        for _ in range(3):
            lo, hi = np.nextafter(lo, -np.inf), np.nextafter(hi, np.inf)
            v += [lo, hi]
    top = n * inc - 1e-10
    v += [top, np.nextafter(top, 0), np.nextafter(top, np.inf), 0.5 * inc, 1.5 * inc, inc / 3, inc * 1e-20]
    return np.array(v + list(rng.uniform(-0.5 * inc, (n + 0.5) * inc, 8)) + SPECIAL)


def points(dim, nCs, incs, rng):
    ax = [axis_values(n, i, rng) for n, i in zip(nCs, incs)]
    if dim == 3:  # the full product would be millions of points
        ax = [np.concatenate([a[-18:], rng.choice(a, 60, replace=True)]) for a in ax]
    grid = np.stack([g.ravel() for g in np.meshgrid(*ax, indexing="ij")], 1)
    near = []  # on the diagonals and planes, and an ulp or a few off
    u = np.concatenate([rng.uniform(0, 1, 300), [0.25, 0.5, 0.75, 1 / 3, 2 / 3, 1e-18]])
    for base in (0, 1):
        off = [base * i if n > base else 0.0 for n, i in zip(nCs, incs)]
        for s in ([1, 1, 1], [1, -1, 1], [1, 1, -1], [-1, 1, 1]):
            p = np.stack([off[d] + incs[d] * (u if s[d] > 0 else 1 - u) for d in range(dim)], 1)
            near += [p, np.nextafter(p, np.inf), np.nextafter(p, -np.inf)]
            if dim == 3:  # x + y = z and the like
                q = p.copy()
                q[:, 2] = off[2] + incs[2] * np.minimum(2 * u, 2 - 2 * u)
                near += [q, np.nextafter(q, np.inf)]
            if dim > 1:
                r = p.copy()
                r[:, 0] = np.nextafter(r[:, 0], np.inf)
                near.append(r)
    rand = rng.uniform(-0.3, 1.3, (20000, dim)) * np.array(nCs) * np.array(incs)
    return np.ascontiguousarray(np.concatenate([grid] + near + [rand]))


CASES = [(1, "II", (50,), (0.019999999999999997,)), (1, "II", (1,), (0.3,)), (1, "II", (5,), (1.0 / 3,)),
         (2, "I", (4, 4), (160.0, 120.0)), (2, "I", (3, 5), (1.0 / 3, 0.2)), (2, "I", (7, 1), (0.1, 1000.1)),
         (2, "I", (100, 3), (1e-3, 7.0)), (2, "II", (3, 5), (85.33333333333333, 51.2)), (2, "II", (1, 9), (1e5 / 3, 1e-4)),
         (3, "I", (2, 2, 2), (48.0, 40.0, 32.0)), (3, "I", (3, 2, 4), (0.1, 0.3, 7.7)), (3, "I", (2, 3, 5), (33.3, 21.1, 5.7)),
         (3, "II", (3, 3, 2), (1.0 / 3, 0.2, 0.7))]


@pytest.mark.parametrize("dim,tess,nCs,incs", CASES)
def test_cells_equal_the_oracle_next_to_every_decision(gpu, orc, dim, tess, nCs, incs):
    torch = gpu
    print("[gpu] lookup edges", dim, tess, nCs, incs, flush=True)
    rng = np.random.default_rng(41)
    pts = points(dim, nCs, incs, rng)
    nC = int(np.prod(nCs)) * (1 if tess == "II" else (4 if dim == 2 else 5))
    want = orc.calc_cell_idx({"dim": dim, "tess": 1 if tess == "I" else 2, "nCs": list(nCs), "incs": list(incs)}, pts)
    cell = torch.full((len(pts),), -7, dtype=torch.int32, device="cuda")
    Calcs(nC, np.float64, dim, dim, tess).calc_cell_idx(None, None, torch.from_numpy(pts).cuda(), cell, dim, dim,
                                                        nCs, incs)
    got = cell.cpu().numpy()
    bad = np.nonzero(got != want)[0]
    assert bad.size == 0, (bad.size, pts[bad[:5]].tolist(), got[bad[:5]].tolist(), want[bad[:5]].tolist())
    assert (got >= 0).all() and (got < nC).all()
