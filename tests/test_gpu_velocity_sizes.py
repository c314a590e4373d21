"""calc_v at point counts around what its resident blocks cover in one walk
over the points (the block and their number follow the table's size), against
the oracle bit for bit (cpab/gpu/calc_2Dto2D.cu:561-602)."""
import numpy as np
import pytest

from cpabdiffeo_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nCs,tess,dim", [((4, 4), "I", 2), ((16, 16), "I", 2), ((50,), "II", 1), ((4, 4, 4), "I", 3)])
def test_any_point_count(gpu, orc, nCs, tess, dim):
    torch = gpu
    sp = configs.unit_space(nCs, tess, dim=dim)
    rng = np.random.default_rng(61)
    sp.update_pat(rng.normal(size=sp.D))
    pts = rng.uniform(-0.1, 1.1, (2 * 256 * 2048 + 3, dim))
    want = orc.calc_v(sp.tessellation.geom(), pts, sp.pat.Avees.reshape(sp.nC, -1))
    for n in (1, 255, 257, 511, 513, 3 * 256 * 512 - 1, 3 * 256 * 512 + 1, 256 * 2048 + 1, len(pts)):
        print("[gpu] calc_v", nCs, n, flush=True)
        v = torch.full((n + 1, dim), 7.0, dtype=torch.float64, device="cuda")
        sp.calc_v(pts=torch.from_numpy(pts[:n]).cuda(), out=v[:n])
        got = v.cpu().numpy()
        assert np.array_equal(got[:n], want[:n]) and (got[n] == 7.0).all(), n
