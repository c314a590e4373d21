"""A batch's grabs of tiles: down to one towards the end, or whole chunks.

Whole where a tile times the steps is below 32 768 and the chunks are 1 024 or
more.  On either side of both limits, counts of tiles that the chunk does not
divide: every point is integrated once.  End points against the oracle, bit for
bit."""
import numpy as np
import pytest

from cpabdiffeo_amd import batch, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("insts,tile,chunk,nT", [(41, 1024, 2, 31), (41, 1024, 2, 32), (35, 1024, 2, 31), (61, 1024, 3, 4),
                                                 (140, 256, 8, 6)])
def test_end_points_equal_the_oracle(gpu, orc, insts, tile, chunk, nT):
    torch = gpu
    print("[gpu] batch grabs", insts, tile, chunk, nT, flush=True)
    sp = configs.unit_space((7,), "II", dim=1)
    rng = np.random.default_rng(31)
    n = 58 * 1024 + 7
    A = np.stack([(sp.B @ rng.normal(size=sp.d)).reshape(sp.nC, 2) for _ in range(insts)])
    A /= np.abs(A).max()
    plan = batch.BatchPlan(1, "II", [(list(sp.nCs), list(sp.incs), n)] * insts)
    tables = plan.prep(torch.from_numpy(A.reshape(-1, 2)).cuda(), 1, 1.0 / nT)
    t = tables.cpu().numpy().reshape(insts, 2, sp.nC, 2)
    pts = rng.random((insts * n, 1))
    out = torch.full(pts.shape, -7.0, dtype=torch.float64, device="cuda")
    plan.calc_T(tables, torch.from_numpy(pts).cuda(), out, 1.0 / nT, nT, 3, sched=batch.BatchSched(tile, 256, chunk))
    got, g = out.cpu().numpy(), sp.tessellation.geom()
    for i in range(insts):
        want = orc.calc_T(g, pts[i * n:(i + 1) * n], t[i, 0], t[i, 1], 1.0 / nT, nT, 3)
        assert np.array_equal(got[i * n:(i + 1) * n], want), i
