"""A batch whose one tile would be nearly 2^31 points.

A block's waves draw a tile's points from a 32-bit cursor, which runs past the
tile's end by up to 64 for each wave, so a tile of the largest size that a
schedule can name has to be cut.  Sampled points (the first, those around 2^30
and 2^31, the last and random ones) against the oracle, bit for bit."""
import numpy as np
import pytest

from cpabdiffeo_amd import batch, configs

pytestmark = pytest.mark.gpu

N = (1 << 31) - 5


def test_largest_tile(gpu, orc):
    torch = gpu
    free, _ = torch.cuda.mem_get_info()
    if free < 16 * N + (4 << 30):
        pytest.skip("needs %.0f GB of free device memory" % (16 * N / 2**30 + 4))
    print("[gpu] batch of one tile of", N, "points", flush=True)
    sp = configs.unit_space((5,), "II", dim=1)
    A = (sp.B @ np.random.default_rng(81).normal(size=sp.d)).reshape(sp.nC, 2)
    A /= np.abs(A).max()
    plan = batch.BatchPlan(1, "II", [((5,), (float(sp.incs[0]),), N)])
    tables = plan.prep(torch.from_numpy(np.ascontiguousarray(A)).cuda(), 1, 0.5)
    t = tables.cpu().numpy().reshape(2, sp.nC, 2)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(82)
    pos0 = torch.rand((N, 1), dtype=torch.float64, device="cuda", generator=gen)
    out = torch.full_like(pos0, -7.0)
    plan.calc_T(tables, pos0, out, 0.5, 2, 3, sched=batch.BatchSched((1 << 31) - 1, 1024, 1))
    torch.cuda.synchronize()
    rng, m = np.random.default_rng(83), 1 << 30
    idx = np.unique(np.concatenate([np.arange(1500), np.arange(m - 1500, m + 1500), np.arange(N - 3000, N),
                                    rng.integers(0, N, 4000)]))
    it = torch.from_numpy(idx).cuda()
    want = orc.calc_T(sp.tessellation.geom(), pos0[it].cpu().numpy(), t[0], t[1], 0.5, 2, 3)
    got = out[it].cpu().numpy()
    bad = np.nonzero((got != want).any(1))[0]
    assert bad.size == 0, (bad.size, idx[bad[:5]])
    assert int((out == -7.0).sum()) == 0  # every point was written
    del pos0, out
    torch.cuda.empty_cache()
