"""calc_T_simple and calc_grad_theta where their kernels' forms change.

Both keep a point's row (the sensitivity also its columns' basis rows) until
the point leaves the bounds of its cell, and the sensitivity takes 1, 2, 4 or
8 columns a thread, the last ones shared with the chunk before.  Points start
on and across facets, walls and corners, inside and outside the domain, in
counts around a wave; columns stand around the chunks' widths; end points and
sensitivities must equal the oracle's bit for bit
(cpab/gpu/calc_2Dto2D.cu:202-319, 412-445)."""
import numpy as np
import pytest

from cpabdiffeo_amd.calcs import Calcs
from cpabdiffeo_amd.space import CpaSpace
from test_gpu_stretch import CASES, start_points

pytestmark = pytest.mark.gpu


def setup(dim, tess, nCs, extent, zero, speed):
    sp = CpaSpace([0] * dim, list(extent), list(nCs), zero_v_across_bdry=[zero] * dim, tess=tess,
                  valid_outside=not zero)
    rng = np.random.default_rng(53)
    A = (sp.B @ rng.normal(size=sp.d)).reshape(sp.nC, dim, dim + 1)
    A *= speed / max(np.abs(A[:, :, :-1]).max(), np.abs(A[:, :, -1] / np.array(extent)).max())
    return sp, A.reshape(sp.nC, -1), start_points(dim, extent, nCs, rng), rng


@pytest.mark.parametrize("dim,tess,nCs,extent,zero,speed", CASES)
def test_simple_equals_the_oracle(gpu, orc, dim, tess, nCs, extent, zero, speed):
    torch = gpu
    print("[gpu] simple", dim, tess, nCs, extent, zero, flush=True)
    sp, A, pts, _ = setup(dim, tess, nCs, extent, zero, speed)
    want = orc.calc_T_simple(sp.tessellation.geom(), pts, A, 0.01, 40, 10)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    for n in (1, 63, 65, len(pts)):
        out = torch.zeros((n, dim), dtype=torch.float64, device="cuda")
        Calcs(sp.nC, np.float64, dim, dim, tess).calc_T_simple(None, None, dev(A), dev(pts[-n:]), 0.01, 40, 10, out,
                                                               dim, dim, sp.nCs, sp.incs)
        assert np.array_equal(out.cpu().numpy(), want[-n:], equal_nan=True)


@pytest.mark.parametrize("n,d", [(1, 1), (65, 3), (5000, 1), (5000, 9), (5000, 17), (5000, 37), (5000, 78), (4937, 80)])
@pytest.mark.parametrize("dim,tess,nCs,extent,zero,speed", CASES)
def test_sensitivity_equals_the_oracle(gpu, orc, dim, tess, nCs, extent, zero, speed, n, d):
    torch = gpu
    print("[gpu] sensitivity", dim, tess, nCs, extent, zero, n, d, flush=True)
    sp, A, pts, rng = setup(dim, tess, nCs, extent, zero, speed)
    pts = pts[-n:] if n <= len(pts) else np.concatenate([pts, rng.uniform(0, 1, (n - len(pts), dim)) * extent])
    Bs = rng.normal(size=(d, sp.nC, dim, dim + 1))
    pos, G = orc.calc_grad_theta(sp.tessellation.geom(), pts, A, Bs, 0.01, 10, 5)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    out = torch.zeros((n, dim), dtype=torch.float64, device="cuda")
    grad = torch.full((n, dim, d), np.nan, dtype=torch.float64, device="cuda")
    Calcs(sp.nC, np.float64, dim, dim, tess).calc_grad_theta(None, None, dev(A), dev(Bs), dev(pts), 0.01, 10, 5, out,
                                                             grad, dim, dim, sp.nCs, sp.incs)
    assert np.array_equal(out.cpu().numpy(), pos, equal_nan=True)
    assert np.array_equal(grad.cpu().numpy(), G, equal_nan=True)
