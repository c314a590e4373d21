"""calc_T's two phases at the places where their bounds could go wrong.

`advance` takes steps without a lookup while affine functions of a point stay
within bounds of its cell (its triangle, tetrahedron or box, and what the
lookup gives to it beyond the domain's walls and corners).  The points here
start and travel on and across facets, walls and corners, inside and outside
the domain, with fields that are zero across the walls and fields that are
not; end points, fallback counts and trajectories must equal the oracle's bit
for bit, for point counts around a wave (cpab/gpu/calc_2Dto2D.cu:348-408)."""
import numpy as np
import pytest

from cpabdiffeo_amd.calcs import Calcs
from cpabdiffeo_amd.space import CpaSpace

pytestmark = pytest.mark.gpu

#        dim tess  nCs        extent            zero  speed
CASES = [(1, "II", (50,), (1.0,), True, 1.0), (1, "II", (5,), (100.0,), False, 1.0), (1, "II", (1,), (3.0,), False, 1.0),
         (2, "I", (4, 4), (1.0, 1.0), True, 1.0), (2, "I", (4, 4), (640.0, 480.0), False, 1.0),
         (2, "I", (1, 1), (1.0, 1.0), False, 2.0), (2, "I", (3, 5), (90.0, 70.0), False, 2.0),
         (2, "I", (2, 2), (64.0, 64.0), False, 3.0), (2, "II", (3, 4), (30.0, 32.0), False, 2.0),
         (3, "I", (2, 2, 2), (96.0, 80.0, 64.0), True, 1.0), (3, "I", (2, 3, 2), (20.0, 90.0, 40.0), True, 1.5),
         (3, "I", (4, 4, 4), (64.0, 64.0, 64.0), True, 1.0), (3, "I", (1, 2, 3), (8.0, 16.0, 60.0), True, 1.0),
         (3, "II", (2, 2, 3), (8.0, 7.0, 9.0), False, 1.0)]


def start_points(dim, extent, nCs, rng):
    ext, inc = np.array(extent), np.array(extent) / np.array(nCs)
    lattice = np.stack([m.ravel() for m in np.meshgrid(*[np.linspace(0, 1, 13 if dim < 3 else 9)] * dim, indexing="ij")], 1) * ext
    sides = np.repeat(rng.uniform(0, 1, (300, dim)) * ext, 2, 0)
    sides[np.arange(600), rng.integers(0, dim, 600)] = 0.0
    corner = (rng.uniform(-0.3, 0.3, (400, dim)) * inc) + rng.integers(0, 2, (400, dim)) * ext
    tiny = rng.choice([0.0, -0.0, 1e-300, -1e-17, 1e-17, -5e-324], (60, dim)) * ext
    out = rng.uniform(-1.5, 2.5, (600, dim)) * ext
    far = rng.uniform(-40, 40, (60, dim)) * ext
    return np.concatenate([lattice, sides, corner, tiny, out, far, rng.uniform(0, 1, (3000, dim)) * ext])


@pytest.mark.parametrize("dim,tess,nCs,extent,zero,speed", CASES)
def test_points_and_counts_equal_the_oracle(gpu, orc, dim, tess, nCs, extent, zero, speed):
    torch = gpu
    print("[gpu] stretch", dim, tess, nCs, extent, zero, flush=True)
    rng = np.random.default_rng(51)
    sp = CpaSpace([0] * dim, list(extent), list(nCs), zero_v_across_bdry=[zero] * dim, tess=tess,
                  valid_outside=not zero)
    A = (sp.B @ rng.normal(size=sp.d)).reshape(sp.nC, dim, dim + 1)
    A *= speed / max(np.abs(A[:, :, :-1]).max(), np.abs(A[:, :, -1] / np.array(extent)).max())
    g = sp.tessellation.geom()
    pts = start_points(dim, extent, nCs, rng)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    calcs = Calcs(sp.nC, np.float64, dim, dim, tess)
    for sign in (1, -1):
        sA, T = orc.prep(dim, A.reshape(sp.nC, -1), sign, 0.01)
        want, nfb_w, _ = orc.calc_T(g, pts, T, sA, 0.01, 100, 10, probe=True)
        for n in (1, 63, 65, len(pts)):
            p = pts[-n:]
            out = torch.zeros(p.shape, dtype=torch.float64, device="cuda")
            nfb = torch.zeros(n, dtype=torch.int32, device="cuda")
            calcs.calc_T(None, None, dev(T), dev(sA), dev(p), 0.01, 100, 10, out, dim, dim, sp.nCs, sp.incs,
                         n_fallback=nfb)
            bad = np.nonzero((out.cpu().numpy() != want[-n:]).any(1) | (nfb.cpu().numpy() != nfb_w[-n:]))[0]
            assert bad.size == 0, (sign, n, bad.size, p[bad[:4]].tolist())
        traj = calcs.calc_trajectory(None, None, dev(T), dev(sA), dev(pts), 0.01, 100, 10, dim, dim, sp.nCs, sp.incs)
        assert np.array_equal(traj.cpu().numpy(), orc.calc_trajectory(g, pts, T, sA, 0.01, 100, 10)), sign
    assert nfb_w.sum() > 0 or nCs == (1,)
