"""calc_T's two paths, in lockstep and in phases, around where one gives way to the other.

A wave integrates in lockstep where the whole integration is at most 100
substeps, in 3D below 64 steps; a lane may then wait for new points of its wave
in the middle of a step.  Step counts around both limits (and without substeps
or steps), points on walls, at rest, calm and changing cell at most steps;
single calls, and one wave that takes all the points of a batch's tile or of a
work item.
End points, fallback counts and trajectories against the oracle, bit for bit
(cpab/gpu/calc_2Dto2D.cu:348-408)."""
import ctypes

import numpy as np
import pytest

from cpabdiffeo_amd import batch
from cpabdiffeo_amd.calcs import Calcs, context_for
from cpabdiffeo_amd.serving import ITEM
from test_gpu_simple_walls import CASES, points, tables

pytestmark = pytest.mark.gpu

STEPS = [(0, 5), (1, 5), (3, 33), (10, 10), (100, 1), (101, 1), (10, 11), (7, 0), (150, 0), (2, 60), (40, 4), (63, 4), (64, 4), (120, 10)]


@pytest.mark.parametrize("dim,tess,nCs,extent", CASES)
def test_points_counts_and_trajectories_equal_the_oracle(gpu, orc, dim, tess, nCs, extent):
    torch = gpu
    print("[gpu] lockstep", dim, tess, nCs, extent, flush=True)
    rng = np.random.default_rng(19)
    incs = [e / n for e, n in zip(extent, nCs)]
    nC = int(np.prod(nCs)) * (1 if tess == "II" else (4 if dim == 2 else 5))
    geom = {"dim": dim, "tess": 1 if tess == "I" else 2, "nCs": list(nCs), "incs": incs}
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    calcs = Calcs(nC, np.float64, dim, dim, tess)
    pts = points(dim, extent, rng)
    p, N = dev(pts), len(pts)
    plan = batch.BatchPlan(dim, tess, [(nCs, incs, N)])
    one_wave = batch.BatchSched(4096, 64, 1)
    item = np.zeros(1, dtype=ITEM)
    for speed in (0.0, 0.05, 2.0, 20.0):
        A = tables(dim, nC, incs, extent, speed, rng)
        for nT, nS in STEPS:
            what = (speed, nT, nS)
            dt = 1.0 / max(nT, 1)
            sA, T = orc.prep(dim, A, 1, dt)
            want, nfb_w, _ = orc.calc_T(geom, pts, T, sA, dt, nT, nS, probe=True)
            dT, dA = dev(T), dev(sA)
            for n in (N, 65, 1):
                out = torch.zeros((n, dim), dtype=torch.float64, device="cuda")
                nfb = torch.zeros(n, dtype=torch.int32, device="cuda")
                calcs.calc_T(None, None, dT, dA, p[:n].contiguous(), dt, nT, nS, out, dim, dim, nCs, incs, n_fallback=nfb)
                assert np.array_equal(out.cpu().numpy(), want[:n]), (what, n)
                assert np.array_equal(nfb.cpu().numpy(), nfb_w[:n]), (what, n)
            out = torch.zeros_like(p)
            nfb = torch.zeros(N, dtype=torch.int32, device="cuda")
            plan.calc_T(torch.cat([dT.reshape(-1), dA.reshape(-1)]), p, out, dt, nT, nS, sched=one_wave, n_fallback=nfb)
            assert np.array_equal(out.cpu().numpy(), want), (what, "batch")
            assert np.array_equal(nfb.cpu().numpy(), nfb_w), (what, "batch")
            out = torch.zeros_like(p)
            item["trels"], item["As"], item["pos0"], item["out"] = dT.data_ptr(), dA.data_ptr(), p.data_ptr(), out.data_ptr()
            item["begin"], item["end"] = 0, N
            item["nC0"], item["nC1"], item["nC2"] = (list(nCs) + [0, 0])[:3]
            item["inc_x"], item["inc_y"], item["inc_z"] = (incs + [1.0, 1.0])[:3]
            context_for(p).call("cpab_calc_T_items", dim, geom["tess"], 1, item.ctypes.data, dt, nT, nS, ctypes.byref(one_wave))
            assert np.array_equal(out.cpu().numpy(), want), (what, "item")
            if nT > 0:
                traj = calcs.calc_trajectory(None, None, dT, dA, p, dt, nT, nS, dim, dim, nCs, incs)
                assert np.array_equal(traj.cpu().numpy(), orc.calc_trajectory(geom, pts, T, sA, dt, nT, nS)), what
