"""Launches whose dynamic LDS reaches the limit of a workgroup.

The integration kernels hold a few bytes of LDS of their own, so tables (and a
batch's order of its points) that fill the 160 KiB of a workgroup exactly do
not fit beside them: 1D tables of 5 120 cells are read from global memory, and
a batch tile whose order ends at the limit is taken without one.  Sizes around
the limit against the oracle, bit for bit."""
import numpy as np
import pytest

from cpabdiffeo_amd import batch
from cpabdiffeo_amd.calcs import Calcs

pytestmark = pytest.mark.gpu

LDS = 160 * 1024


def field(nC, orc, seed):
    rng = np.random.default_rng(seed)
    v = np.concatenate([[0.0], rng.normal(size=nC - 1), [0.0]])
    a = np.diff(v) * nC * 0.01
    A = np.stack([a, 0.01 * v[:-1] - a * np.arange(nC) / nC], 1)
    return orc.prep(1, A, 1, 0.05) + (A,)


@pytest.mark.parametrize("nC", [5118, 5119, 5120, 5121])
def test_tables_around_the_limit(gpu, orc, nC):
    torch = gpu
    assert 5120 * 2 * 2 * 8 == LDS
    print("[gpu] full LDS", nC, flush=True)
    sA, T, A = field(nC, orc, 91)
    pts = np.random.default_rng(92).random((3000, 1))
    g = {"dim": 1, "tess": 2, "nCs": [nC], "incs": [1.0 / nC]}
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    c = Calcs(nC, np.float64, 1, 1, "II")
    out, p = torch.zeros(pts.shape, dtype=torch.float64, device="cuda"), dev(pts)
    want = orc.calc_T(g, pts, T, sA, 0.05, 20, 4)
    c.calc_T(None, None, dev(T), dev(sA), p, 0.05, 20, 4, out, 1, 1, [nC], [1.0 / nC])
    assert np.array_equal(out.cpu().numpy(), want)
    traj = c.calc_trajectory(None, None, dev(T), dev(sA), p, 0.05, 20, 4, 1, 1, [nC], [1.0 / nC])
    assert np.array_equal(traj.cpu().numpy(), orc.calc_trajectory(g, pts, T, sA, 0.05, 20, 4))
    sA2, T2 = dev(np.zeros_like(A)), dev(np.zeros_like(A))
    c.calc_T_prep(dev(A), 1, p, 0.05, 20, 4, out, 1, 1, [nC], [1.0 / nC], sA2, T2)
    assert np.array_equal(out.cpu().numpy(), orc.calc_T(g, pts, T2.cpu().numpy(), sA, 0.05, 20, 4))


@pytest.mark.parametrize("left", [0, 2, 8, 14, 16, 18])
def test_batch_orders_around_the_limit(gpu, orc, left):
    torch = gpu
    nC = 4000
    tile = (LDS - left - nC * 32 - 4096) // 2  # the order ends `left` bytes before the limit
    assert 64 <= tile <= 16384
    print("[gpu] batch order", tile, left, flush=True)
    sA, T, A = field(nC, orc, 93)
    plan = batch.BatchPlan(1, "II", [((nC,), (1.0 / nC,), 20000)])
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    tables = dev(np.concatenate([T, sA]).ravel())
    pts = np.random.default_rng(94).random((20000, 1))
    out = torch.zeros(pts.shape, dtype=torch.float64, device="cuda")
    plan.calc_T(tables, dev(pts), out, 0.05, 20, 4, sched=batch.BatchSched(tile, 1024, 1))
    g = {"dim": 1, "tess": 2, "nCs": [nC], "incs": [1.0 / nC]}
    assert np.array_equal(out.cpu().numpy(), orc.calc_T(g, pts, T, sA, 0.05, 20, 4))
