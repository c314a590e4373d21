"""The adjoint of calc_T's map at the edges of its event log.

The forward sweep logs runs of accepted steps and redone steps as events, and
the last lane of a wave with events left spreads them over the wave.  Here
the time steps stand around a run's length, the point counts around a wave,
and the last point sits in the domain's corner, whose steps a field may all
redo (the field is the draw that redoes most of them).  End points must equal
the oracle's bit for bit, gradients to 1e-9 of the sum of the points'
contributions without their signs (1 100 units of some 30 roundings of
1.1e-16 each, and a factor of 250 for the growth of the products), and a
second run must give the same bits (cpab/gpu/calc_2Dto2D.cu:202-319,
348-408)."""
import numpy as np
import pytest

from cpabdiffeo_amd import adjoint
from cpabdiffeo_amd.space import CpaSpace

pytestmark = pytest.mark.gpu

CASES = [("I", (4, 4), (1.0, 1.0), True), ("I", (3, 5), (90.0, 70.0), True), ("I", (2, 2), (64.0, 64.0), False),
         ("II", (3, 4), (30.0, 32.0), False)]


@pytest.mark.parametrize("nT,nS", [(1, 10), (9, 10), (10, 1), (11, 10), (31, 13), (200, 10)])
@pytest.mark.parametrize("tess,nCs,extent,zero", CASES)
def test_gradients_equal_the_oracle(gpu, orc, tess, nCs, extent, zero, nT, nS):
    torch = gpu
    print("[gpu] adjoint events", tess, nCs, zero, nT, nS, flush=True)
    sp = CpaSpace([0, 0], list(extent), list(nCs), zero_v_across_bdry=[zero] * 2, tess=tess, valid_outside=not zero)
    g, nC, dt = sp.tessellation.geom(), sp.nC, 1.0 / max(nT, 20)
    ext, corner = np.array(extent), np.zeros((1, 2))

    def tables(seed):
        A = (sp.B @ np.random.default_rng(seed).normal(size=sp.d)).reshape(nC, 2, 3)
        return orc.prep(2, (A / max(np.abs(A[:, :, :2]).max(), np.abs(A[:, :, 2] / ext).max())).reshape(nC, 6), 1, dt)

    redone = [orc.calc_T(g, corner, T, sA, dt, nT, nS, probe=True)[1].sum() for sA, T in map(tables, range(12))]
    sA, T = tables(int(np.argmax(redone)))
    print("[gpu] steps redone in the corner", max(redone), "of", nT, flush=True)
    rng = np.random.default_rng(52)
    pts = np.concatenate([rng.uniform(-0.2, 1.2, (300, 2)) * ext, corner])
    lam = rng.standard_normal(pts.shape)
    Bs = np.ascontiguousarray(sp.B.T.reshape(sp.d, nC, 2, 3))
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    pos, G = orc.calc_grad_theta_T(g, pts, T, sA, Bs, orc.trel_sensitivity(2, sA, Bs, dt), dt, nT, nS)
    params = dict(dt=dt, nTimeSteps=nT, nStepsODEsolver=nS)
    for n in (1, 63, 64, 65, len(pts)):
        out = torch.empty((1, n, 2), dtype=torch.float64, device="cuda")
        runs = [adjoint.calc_T_vjp(sp, dev(pts[-n:]), dev(lam[-n:]), dev(sA.reshape(nC, 6)), dev(T.reshape(nC, 6)),
                                   params, pos_out=out).cpu().numpy() for _ in range(2)]
        assert np.array_equal(out.cpu().numpy()[0], pos[-n:])
        assert np.array_equal(*runs)
        want = np.einsum("ni,nij->j", lam[-n:], G[-n:])
        scale = np.einsum("ni,nij->j", np.abs(lam[-n:]), np.abs(G[-n:])).max()
        assert np.abs(runs[0].reshape(-1) @ sp.B - want).max() <= 1e-9 * scale
