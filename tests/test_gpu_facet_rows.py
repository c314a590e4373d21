"""calc_T_simple and calc_grad_theta from points on and beside multiples of the increments.

Both keep a cell's row until the point leaves the bounds of its cell, so the
bounds have to be those of the cell that the lookup gave.  Where an increment
is not a power of two, a point just below a multiple of it is beside one in
x * (1 / inc) too, and another rounding than the lookup's can put it into the
next box.  The points here start on every multiple of the increment and within
three ulps of it, crossed with the other axes' multiples (walls and vertices)
and with points inside, and arrive on multiples after one substep; the fields
carry them off to either side, each cell's own velocity a little different.
Waves of one point alone (64 copies of it) and mixed waves; end points and
sensitivities must equal the oracle's bit for bit
(cpab/gpu/calc_2Dto2D.cu:202-319, 412-445)."""
import numpy as np
import pytest

from cpabdiffeo_amd.calcs import Calcs

pytestmark = pytest.mark.gpu

CASES = [(1, "II", (9,), (255.0,)), (1, "II", (18,), (640.0,)), (1, "II", (18,), (10.0,)), (1, "II", (7,), (0.7,)),
         (1, "II", (15,), (3.0,)), (1, "II", (10,), (1.0,)), (1, "II", (50,), (1.0,)), (1, "II", (4,), (1.0,)),
         (2, "I", (18, 18), (640.0, 480.0)), (2, "I", (2, 2), (1138.0, 640.0)), (2, "I", (10, 10), (1.0, 1.0)),
         (2, "I", (7, 4), (0.7, 1.0)), (2, "II", (9, 9), (255.0, 255.0)), (2, "II", (10, 15), (1.0, 3.0)),
         (3, "II", (10, 3, 7), (1.0, 3.0, 0.7)), (3, "I", (10, 3, 7), (1.0, 3.0, 0.7))]
NT, NS, DT = 10, 5, 0.01


def beside(n, inc):
    v = []
    for k in range(n + 1):
        lo = hi = k * inc
        v.append(lo)
        for _ in range(3):
            lo, hi = np.nextafter(lo, -np.inf), np.nextafter(hi, np.inf)
            v += [lo, hi]
    return np.array(v)


def start_points(dim, nCs, incs, rng):
    ax = [beside(n, i) for n, i in zip(nCs, incs)]
    ext = np.array(nCs) * np.array(incs)
    pts = []
    for d in range(dim):  # one axis beside a multiple, the others anywhere
        p = rng.uniform(0, 1, (2 * len(ax[d]), dim)) * ext
        p[:, d] = np.tile(ax[d], 2)
        pts.append(p)
    m = 1500 if dim > 1 else 0  # every axis beside one
    pts.append(np.stack([rng.choice(a, m) for a in ax], 1))
    w = np.stack([rng.choice(a, m) for a in ax], 1)  # (on a wall)
    if m:
        w[np.arange(m), rng.integers(0, dim, m)] = 0.0
    pts.append(w)
    return np.ascontiguousarray(np.concatenate(pts))


def arriving(orc, geom, pts, A, u):
    """Points that a substep carries onto pts, within rounding."""
    h = DT / NS
    q = pts - h * u
    for _ in range(4):
        q += pts - orc.calc_T_simple(geom, q, A, h, 1, 1)
    return q


def fields(dim, nCs, incs, nC, rng):
    """(a velocity u, tables whose velocity is near u in every cell, and a little different from cell to cell)."""
    inc, ext = np.array(incs), np.array(incs) * np.array(nCs)
    for signs in range(1 << dim):
        s = np.array([1.0 if signs >> d & 1 else -1.0 for d in range(dim)])
        u = s * rng.uniform(2.0, 6.0, dim) * inc
        A = np.zeros((nC, dim, dim + 1))
        A[:, :, :-1] = rng.normal(size=(nC, dim, dim)) * 0.05 * (inc[:, None] / ext[None, :])
        A[:, :, -1] = u * (1 + 0.02 * rng.normal(size=(nC, dim)))
        yield u, A.reshape(nC, -1)


@pytest.mark.parametrize("dim,tess,nCs,extent", CASES)
def test_points_and_sensitivities_equal_the_oracle(gpu, orc, dim, tess, nCs, extent):
    torch = gpu
    print("[gpu] facet rows", dim, tess, nCs, extent, flush=True)
    rng = np.random.default_rng(61)
    incs = [e / n for e, n in zip(extent, nCs)]
    nC = int(np.prod(nCs)) * (1 if tess == "II" else (4 if dim == 2 else 5))
    geom = {"dim": dim, "tess": 1 if tess == "I" else 2, "nCs": list(nCs), "incs": incs}
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    calcs = Calcs(nC, np.float64, dim, dim, tess)
    wrong = []
    for u, A in fields(dim, nCs, incs, nC, rng):
        pts = start_points(dim, nCs, incs, rng)
        pts = np.concatenate([pts, arriving(orc, geom, pts, A, u)])
        Bs = rng.normal(size=(2, nC, dim, dim + 1))
        want, G = orc.calc_grad_theta(geom, pts, A, Bs, DT, NT, NS)
        assert np.array_equal(orc.calc_T_simple(geom, pts, A, DT, NT, NS), want)
        for copies in (64, 1):  # a point alone in its wave; others beside it
            p = dev(np.repeat(pts, copies, 0))
            out = torch.zeros_like(p)
            calcs.calc_T_simple(None, None, dev(A), p, DT, NT, NS, out, dim, dim, nCs, incs)
            end = torch.zeros_like(p)
            grad = torch.zeros((len(p), dim, 2), dtype=torch.float64, device="cuda")
            calcs.calc_grad_theta(None, None, dev(A), dev(Bs), p, DT, NT, NS, end, grad, dim, dim, nCs, incs)
            for name, got, ref in (("simple", out, want), ("end", end, want), ("grad", grad, G)):
                bad = (got.cpu().numpy() != np.repeat(ref, copies, 0)).reshape(len(p), -1).any(1)
                if bad.any():
                    wrong.append((name, copies, int(bad.sum()) // copies, len(pts), pts[np.nonzero(bad)[0][0] // copies].tolist()))
    assert not wrong, wrong
