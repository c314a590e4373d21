"""Work items that share one of their tables with the item before.

A block keeps an item's tables in LDS for the next one: for that it has to have
the same Trels, the same signed As and the same number of cells.  Items of one
launch in which each of the three changes alone, in one block and in many,
against the oracle, bit for bit."""
import ctypes

import numpy as np
import pytest

from cpabdiffeo_amd import configs, serving
from cpabdiffeo_amd.calcs import context_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,tess,nCs,fewer", [(1, "II", (20,), (7,)), (2, "I", (4, 4), (2, 2)), (3, "I", (2, 2, 2), (1, 1, 2))])
@pytest.mark.parametrize("chunk", [1, 64])
def test_each_item_has_its_own_tables(gpu, orc, dim, tess, nCs, fewer, chunk):
    torch = gpu
    print("[gpu] item tables", dim, tess, chunk, flush=True)
    rng = np.random.default_rng(33)
    sp = configs.unit_space(nCs, tess, dim=dim)
    A = [(sp.B @ rng.normal(size=sp.d)).reshape(sp.nC, -1) for _ in range(2)]
    tabs = [orc.prep(dim, a / np.abs(a).max(), 1, 0.02) for a in A]  # (signed As, Trels)
    few = configs.unit_space(fewer, tess, dim=dim)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    dT, dS = [dev(t[1]) for t in tabs], [dev(t[0]) for t in tabs]
    pts = rng.random((700, dim))
    p = dev(pts)
    rows, outs, wants = [], [], []
    for k in range(40):
        iT, iS, space = (k // 4) % 2, (k // 2) % 2, few if k % 2 or k % 8 == 2 else sp
        g = space.tessellation.geom()
        o = torch.zeros_like(p)
        outs.append(o)
        wants.append(orc.calc_T(g, pts, tabs[iT][1][:space.nC], tabs[iS][0][:space.nC], 0.02, 50, 10))
        geo = list(g["nCs"]) + [0] * (3 - dim) + [float(x) for x in space.incs] + [1.0] * (3 - dim)
        rows.append(tuple([dT[iT].data_ptr(), dS[iS].data_ptr(), p.data_ptr(), o.data_ptr(), 0, len(pts)] + geo))
    it = np.array(rows, dtype=serving.ITEM)
    sched = serving.Sched(1024, 256, chunk)
    context_for(p).call("cpab_calc_T_items", dim, 1 if tess == "I" else 2, len(it), it.ctypes.data, 0.02, 50, 10,
                        ctypes.byref(sched))
    bad = [k for k, (o, w) in enumerate(zip(outs, wants)) if not np.array_equal(o.cpu().numpy(), w)]
    assert not bad, bad
