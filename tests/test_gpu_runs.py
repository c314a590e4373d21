"""Grids and work items in the orders the kernels take them in.

Rows along x are walked in tiles of up to 8 rows, in 2D and in 3D, and
neighbouring work items of one request are integrated as one run; the points
of every grid shape (whole, partial and short bands, rows that no tile fits)
and of every way to cut requests into items must be the oracle's, bit for bit
(cpab/gpu/calc_2Dto2D.cu:348-408)."""
import ctypes

import numpy as np
import pytest

from cpabdiffeo_amd import configs, serving
from cpabdiffeo_amd.calcs import Calcs, context_for

pytestmark = pytest.mark.gpu


def grid(*n):
    ax = [np.arange(k) / k for k in n]
    m = np.meshgrid(*ax[::-1], indexing="ij")
    return np.stack([x.ravel() for x in m[::-1]], 1)


def field(sp, seed):
    A = sp.B @ np.random.default_rng(seed).normal(size=sp.d)
    return (A / np.abs(A).max()).reshape(sp.nC, -1)


@pytest.mark.parametrize("n", [(8, 9), (16, 3), (32, 2), (64, 1), (40, 37), (24, 20), (8, 8, 8), (16, 3, 5), (40, 9, 3),
                               (32, 2, 7), (12, 6, 6), (8, 1, 90)])
def test_calc_T_of_grids(gpu, orc, n):
    torch = gpu
    print("[gpu] grid", n, flush=True)
    sp = configs.unit_space((4, 4) if len(n) == 2 else (2, 3, 2), "I", dim=len(n))
    pts = grid(*n)
    sA, T = orc.prep(len(n), field(sp, 71), 1, 0.01)
    want = orc.calc_T(sp.tessellation.geom(), pts, T, sA, 0.01, 100, 10)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    out = torch.zeros(pts.shape, dtype=torch.float64, device="cuda")
    Calcs(sp.nC, np.float64, len(n), len(n), "I").calc_T(None, None, dev(T), dev(sA), dev(pts), 0.01, 100, 10, out,
                                                         len(n), len(n), sp.nCs, sp.incs)
    assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("dim,tess,nCs", [(1, "II", (50,)), (2, "I", (4, 4)), (2, "II", (3, 5)), (3, "I", (4, 4, 4))])
def test_items_cut_anywhere(gpu, orc, dim, tess, nCs):
    torch = gpu
    print("[gpu] items", dim, tess, flush=True)
    sp = configs.unit_space(nCs, tess, dim=dim)
    g = sp.tessellation.geom()
    rng = np.random.default_rng(72)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    geo = list(nCs) + [0] * (3 - dim) + [float(x) for x in sp.incs] + [1.0] * (3 - dim)
    reqs, keep = [], []
    for k in range(3):
        pts = {1: rng.random((30000, 1)), 2: grid(128, 130), 3: grid(32, 24, 9)}[dim]
        sA, T = orc.prep(dim, field(sp, 73 + k), 1, 0.01)
        d = [dev(T), dev(sA), dev(pts)]
        d.append(torch.full_like(d[2], 9.0))
        keep.append(d)
        reqs.append((pts, orc.calc_T(g, pts, T, sA, 0.01, 100, 10)))
    for cut in ("even", "odd", "interleaved"):
        rows = []
        for k, (pts, _) in enumerate(reqs):
            step = 1024 if cut != "odd" else 333
            b = np.arange(0, len(pts), step)
            rows += [(i if cut == "interleaved" else 0, k, s, min(s + step, len(pts))) for i, s in enumerate(b)]
        rows.sort(key=lambda r: r[0])  # (stable)
        it = np.zeros(len(rows), dtype=serving.ITEM)
        for j, (_, k, b, e) in enumerate(rows):
            it[j] = tuple([keep[k][i].data_ptr() for i in range(4)] + [b, e] + geo)
        for d in keep:
            d[3].fill_(9.0)
        sched = serving.Sched(1024, 1024, 1)
        context_for(keep[0][2]).call("cpab_calc_T_items", dim, 1 if tess == "I" else 2, len(it), it.ctypes.data, 0.01,
                                     100, 10, ctypes.byref(sched))
        for k, (_, want) in enumerate(reqs):
            assert np.array_equal(keep[k][3].cpu().numpy(), want), (cut, k)
