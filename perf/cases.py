"""The work whose time on MI355X this framework is judged by: sizes and options of real calls through the public
entry points, the plain 64-bit result of each, and the work no implementation can do without.

A case is a dict of plain values; its "kind" names the call:
  points       CpaSpace.calc_T_fwd / calc_T_inv / calc_T_simple of scattered or gridded points (1D, 2D, 3D)
  warp         TransformWrapper(3D): a new transform, calc_T_inv of the pixel grid and the image's (volume's) remap
  field        CpaSpace.calc_v and calc_cell_idx of a dense grid (showing a velocity field and its cells)
  trajectory   CpaSpace.calc_trajectory
  sensitivity  CpaSpace.calc_grad_theta: end points and dT/dtheta of every point
  batch        BatchPlan: tables and end points of many instances, each with its own tessellation
  pairs        adjoint.warp_ssd, forward and backward: the SSD loss of image pairs and its gradient in theta
  chain        DeviceMetropolis: registration chains, set_theta and a run of steps
  served       Server.run on requests that wait together, their points and volumes returned
Integration is over t = 1 in 100 steps with 10 RK2 substeps, as in the benchmark; fields are draws from the
squared-exponential prior (length 0.1, variance 1).
"""
import copy
import functools
import math

import numpy as np
import torch

from cpabdiffeo_amd import adjoint, batch, configs, registration, serving
from cpabdiffeo_amd.space import PAT, CpaSpace
from cpabdiffeo_amd.tessellation import Tessellation
from cpabdiffeo_amd.transform_wrapper import TransformWrapper, TransformWrapper3D

NT, NS, DT = 100, 10, 0.01
PARAMS = dict(dt=DT, nTimeSteps=NT, nStepsODEsolver=NS)


# ------------------------------------------------------------------ cases
def listed():
    return [
        # a set of landmarks carried by a transform: the smallest call, launches and latency only
        dict(name="landmarks_2d_1000", kind="points", what="T", sign=1, tess="I", nx=4, ny=4, nz=0, grid=False, n=1000),
        # the benchmark's single call: a 512 x 512 grid of the unit square
        dict(name="grid_2d_512x512", kind="points", what="T", sign=1, tess="I", nx=4, ny=4, nz=0, grid=True, n=512 * 512),
        # warping a VGA image through the wrapper: cells of 160 x 120 pixels, fields that may leave the image
        dict(name="image_warp_480x640", kind="warp", tess="I", nx=4, ny=4, nz=0, rows=480, cols=640, slices=0),
        # a long 1D signal (time warping): 50 intervals, a million samples
        dict(name="signal_1d_1e6", kind="points", what="T", sign=1, tess="II", nx=50, ny=0, nz=0, grid=False, n=1000000),
        # warping a volume: tetrahedra, trilinear remap
        dict(name="volume_warp_64x80x96", kind="warp", tess="I", nx=2, ny=2, nz=2, rows=80, cols=96, slices=64),
        # the velocity field and the cell map of a large image on a fine tessellation (1 024 cells)
        dict(name="field_2048x2048", kind="field", tess="I", nx=16, ny=16, nz=0, rows=2048, cols=2048),
        # the paths of many points, every step kept
        dict(name="trajectory_65536", kind="trajectory", tess="I", nx=4, ny=4, nz=0, sign=1, n=65536),
        # dT/dtheta of every pixel of a 128 x 128 grid (62 columns), with calc_T_simple's end points
        dict(name="sensitivity_128x128", kind="sensitivity", tess="I", nx=4, ny=4, nz=0, n=128 * 128),
        # many alignments at once, of mixed sizes and tessellations
        dict(name="batch_256", kind="batch", instances=256, most=1000000),
        # one step of gradient-based registration of 64 pairs of 128 x 128 images
        dict(name="pairs_64x128x128", kind="pairs", simple=False, pairs=64, n=128),
        # the benchmark's registration: one chain on a 256 x 256 image, speculation as the benchmark tunes it
        dict(name="chain_256x256", kind="chain", chains=1, n=256, steps=200, spec=32),
        # the served mix of 1D, 2D and 3D requests, all waiting
        dict(name="served_48", kind="served", requests=48),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["points", "points", "warp", "warp", "field", "trajectory", "sensitivity", "batch", "pairs",
                       "chain", "served"])
    tess = rng.choice(["I", "I", "I", "II"])
    nx, ny = rng.choice([(2, 2), (3, 5), (4, 4), (4, 6), (5, 3), (8, 8), (7, 9), (10, 10)])
    if kind == "points":
        dim = rng.choice([1, 2, 2, 3])
        c = dict(kind=kind, what=rng.choice(["T", "T", "T", "simple"]), sign=rng.choice([1, -1]), tess=tess, nx=nx,
                 ny=ny, nz=0, grid=False, n=_log(rng, 500, 2000000))
        if dim == 1:
            c.update(tess="II", nx=rng.choice([5, 10, 32, 50]), ny=0)
        elif dim == 3:
            nx, ny, nz = rng.choice([(2, 2, 2), (3, 3, 3), (4, 4, 4), (2, 3, 4)])
            c.update(nx=nx, ny=ny, nz=nz, n=_log(rng, 500, 300000))
        elif rng.random() < 0.5:
            c.update(grid=True, n=_log(rng, 30, 1500) ** 2)
        if c["what"] == "simple":
            c["n"] = min(c["n"], 250000)
        return c
    if kind == "warp":
        if rng.random() < 0.6:
            return dict(kind=kind, tess=tess, nx=nx, ny=ny, nz=0, rows=_log(rng, 64, 1200), cols=_log(rng, 64, 1200),
                        slices=0)
        k = rng.choice([2, 2, 3, 4])
        return dict(kind=kind, tess=tess, nx=k, ny=k, nz=k, rows=_log(rng, 24, 110), cols=_log(rng, 24, 110),
                    slices=_log(rng, 24, 110))
    if kind == "field":
        return dict(kind=kind, tess=tess, nx=rng.choice([4, 8, 16]), ny=rng.choice([4, 6, 16]), nz=0,
                    rows=_log(rng, 100, 2000), cols=_log(rng, 100, 2000))
    if kind == "trajectory":
        return dict(kind=kind, tess=tess, nx=nx, ny=ny, nz=0, sign=rng.choice([1, -1]), n=_log(rng, 1000, 60000))
    if kind == "sensitivity":
        nx, ny = rng.choice([(2, 2), (3, 3), (4, 4), (3, 5)])
        return dict(kind=kind, tess="I", nx=nx, ny=ny, nz=0, n=_log(rng, 500, 16000))
    if kind == "batch":
        return dict(kind=kind, instances=_log(rng, 8, 200), most=_log(rng, 10000, 1000000))
    if kind == "pairs":
        return dict(kind=kind, simple=rng.random() < 0.25, pairs=_log(rng, 1, 40), n=rng.choice([33, 64, 96, 100, 128]))
    if kind == "chain":
        return dict(kind=kind, chains=rng.choice([1, 1, 4, 16]), n=rng.choice([64, 100, 128, 192]),
                    steps=_log(rng, 10, 60), spec=rng.choice([0, 1, 8]))
    return dict(kind="served", requests=_log(rng, 4, 48))


# ----------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _space(tess, nCs, valid_outside=False):
    """(space on the unit box, the factor S of its prior: theta = S z)."""
    dim = len(nCs)
    sp = CpaSpace([0] * dim, [1] * dim, list(nCs), zero_v_across_bdry=[not valid_outside] * dim, tess=tess,
                  valid_outside=valid_outside)
    w, U = np.linalg.eigh(sp.se_prior_cov(0.1, 1.0))
    return sp, U * np.sqrt(np.clip(w, 0.0, None))


def _ncs(case):
    return tuple(k for k in (case["nx"], case["ny"], case["nz"]) if k)


def _draw_avees(space, factor, seed):
    rng = np.random.default_rng(seed)
    return space.B @ (factor @ rng.standard_normal(space.d))


def _rescaled(Avees, nC, extent):
    """The unit box's field on the box of that extent: x -> s(x / s)."""
    s = np.asarray(extent, dtype=np.float64)
    A = np.asarray(Avees).reshape(nC, len(s), len(s) + 1).copy()
    A[:, :, :-1] *= s[:, None] / s[None, :]
    A[:, :, -1] *= s
    return A.reshape(-1)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(n, dim, seed):
    return torch.rand((n, dim), dtype=torch.float64, device="cuda", generator=_gen(seed))


def _unit_grid(rows, cols):
    y = torch.arange(rows, dtype=torch.float64, device="cuda") / rows
    x = torch.arange(cols, dtype=torch.float64, device="cuda") / cols
    yy, xx = torch.meshgrid(y, x, indexing="ij")
    return torch.stack([xx.reshape(-1), yy.reshape(-1)], 1).contiguous()


def _blobs(shape, seed, shift=0.0, count=30):
    """A float32 image (volume) of Gaussian blobs in [0, 1]; shift moves each centre a little."""
    rng = np.random.default_rng(seed)
    d = len(shape)
    c, s, a = rng.uniform(0, 1, (count, d)), rng.uniform(0.03, 0.12, count), rng.uniform(0.2, 1.0, count)
    c = c + shift * rng.standard_normal((count, d))
    img = torch.zeros(shape, dtype=torch.float64, device="cuda")
    for k in range(count):
        term = torch.full((), float(a[k]), dtype=torch.float64, device="cuda")
        for i, n in enumerate(shape):
            ax = ((torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) / n - float(c[k, i])) ** 2
            term = term[..., None] * torch.exp(-ax / (2 * float(s[k]) ** 2))
        img += term
    return ((img - img.min()) / (img.max() - img.min())).float().contiguous()


@functools.lru_cache(maxsize=None)
def _wrapper(tess, nCs, extent):
    """One wrapper a tessellation and image size, as a program keeps it."""
    if len(nCs) == 2:
        tw = TransformWrapper(nRows=extent[1], nCols=extent[0], nLevels=1, base=nCs, tess=tess)
    else:
        tw = TransformWrapper3D(nRows=extent[1], nCols=extent[0], nSlices=extent[2], nLevels=1, base=nCs, tess=tess)
    tw.params_flow_int.update(PARAMS)
    return tw


@functools.lru_cache(maxsize=None)
def _server():
    return serving.Server(serving.default_kinds())


@functools.lru_cache(maxsize=None)
def _pixel_space(n):
    return configs.pixel_space(n, (4, 4), "I")


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("points", "trajectory", "sensitivity", "field"):
        sp, factor = _space(case["tess"], _ncs(case))
        pat = PAT(sp, _draw_avees(sp, factor, seed))
        pat.device_table()
        st = dict(case=case, space=sp, pat=pat)
        if kind == "field":
            st["pts"] = _unit_grid(case["rows"], case["cols"])
            st["v"] = torch.empty_like(st["pts"])
            st["cell"] = torch.empty(st["pts"].shape[0], dtype=torch.int32, device="cuda")
            return st
        n = case["n"]
        if kind == "sensitivity" or (kind == "points" and case["grid"]):
            side = int(round(math.sqrt(n)))
            st["pts"] = _unit_grid(side, side) if side * side == n else _uniform(n, 2, seed)
        else:
            st["pts"] = _uniform(n, sp.dim_domain, seed)
        st["out"] = torch.empty_like(st["pts"])
        if kind == "sensitivity":
            st["grad"] = torch.empty((n, sp.dim_domain, sp.d), dtype=torch.float64, device="cuda")
        return st
    if kind == "warp":
        nCs = _ncs(case)
        extent = (case["cols"], case["rows"], case["slices"])[:len(nCs)]
        unit, factor = _space(case["tess"], nCs, valid_outside=len(nCs) == 2)
        Av = _rescaled(_draw_avees(unit, factor, seed), unit.nC, extent)
        img = _blobs(extent[::-1], seed)
        if len(nCs) == 2:
            pts = torch.from_numpy(Tessellation([0, 0], list(extent), [1, 1], "II").dense_grid_img()).cuda()
        else:
            pts = torch.from_numpy(Tessellation([0] * 3, list(extent), [1, 1, 1], "II").dense_grid_img()).cuda()
        return dict(case=case, tw=_wrapper(case["tess"], nCs, extent), Avees=Av, img=img, pts=pts,
                    inv=torch.empty_like(pts), warped=torch.empty_like(img))
    if kind == "batch":
        rng, sizes = np.random.default_rng(seed), np.random.default_rng(case["instances"])
        insts, Avs = [], []
        for _ in range(case["instances"]):
            g, n = int(sizes.choice([4, 8, 16])), math.exp(sizes.uniform(math.log(1e3), math.log(case["most"])))
            sp, factor = _space("I", (g, g))
            insts.append(((g, g), (1.0 / g, 1.0 / g), int(round(n))))
            Avs.append((sp.B @ (factor @ rng.standard_normal(sp.d))).reshape(-1, 6))
        plan = batch.BatchPlan(2, "I", insts)
        pts = _uniform(plan.nPts, 2, seed)
        return dict(case=case, plan=plan, insts=insts, As=torch.from_numpy(np.concatenate(Avs)).cuda(), pts=pts,
                    out=torch.empty_like(pts), tables=torch.empty(plan.tableDoubles, dtype=torch.float64, device="cuda"))
    if kind == "pairs":
        n, m = case["n"], case["pairs"]
        unit, factor = _space("I", (4, 4))
        rng = np.random.default_rng(seed)
        B = torch.from_numpy(np.ascontiguousarray(registration.pixel_basis(unit, n))).cuda()
        src = torch.stack([_blobs((n, n), seed * 1000 + i) for i in range(m)])
        dst = torch.stack([_blobs((n, n), seed * 1000 + i, shift=0.02) for i in range(m)])
        dst = dst + 0.02 * torch.randn(dst.shape, device="cuda", generator=_gen(seed))
        theta = torch.from_numpy(0.3 * (rng.standard_normal((m, unit.d)) @ factor.T)).cuda()
        return dict(case=case, space=_pixel_space(n), B=B, src=src, dst=dst.contiguous(), theta=theta.requires_grad_(True))
    if kind == "chain":
        problem = registration.RegistrationProblem(n=case["n"], seed=seed)
        chains = registration.DeviceMetropolis(problem, nChains=case["chains"], scale=0.01, seed=seed,
                                               trace_len=case["steps"], spec_depth=case["spec"])
        return dict(case=case, chains=chains, zero=np.zeros(chains.d))
    # the mix's sizes by the case, its transforms and points by the seed
    srv, rng = _server(), np.random.default_rng(seed)
    reqs = serving.make_mix(case["requests"], srv.kinds, seed=case["requests"])
    for r in reqs:
        r.theta, r.seed = srv.kinds[r.kind].factor @ rng.standard_normal(srv.kinds[r.kind].d), int(rng.integers(1 << 31))
    return dict(case=case, server=srv, requests=reqs)


# -------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "points":
        sp = state["space"]
        kw = dict(pat=state["pat"], pts=state["pts"], out=state["out"], **PARAMS)
        if case["what"] == "simple":
            return sp.calc_T_simple(mysign=case["sign"], **kw)
        return sp.calc_T_fwd(**kw) if case["sign"] == 1 else sp.calc_T_inv(**kw)
    if kind == "warp":
        tw = state["tw"]
        tw.update_pat_from_Avees(state["Avees"], 0)
        tw.calc_T_inv(state["pts"], state["inv"], 0)
        tw.remap_fwd(state["inv"], state["img"], state["warped"])
        return {"points": state["inv"], "warped": state["warped"]}
    if kind == "field":
        sp = state["space"]
        sp.calc_v(pat=state["pat"], pts=state["pts"], out=state["v"])
        sp.calc_cell_idx(state["pts"], state["cell"])
        return {"v": state["v"], "cell": state["cell"]}
    if kind == "trajectory":
        return state["space"].calc_trajectory(pat=state["pat"], pts=state["pts"], mysign=case["sign"], **PARAMS).gpu
    if kind == "sensitivity":
        state["space"].calc_grad_theta(pat=state["pat"], pts=state["pts"], transformed=state["out"],
                                       grad_per_point=state["grad"], **PARAMS)
        return {"points": state["out"], "grad": state["grad"]}
    if kind == "batch":
        plan = state["plan"]
        plan.prep(state["As"], 1, DT, state["tables"])
        return plan.calc_T(state["tables"], state["pts"], state["out"], DT, NT, NS)
    if kind == "pairs":
        theta = state["theta"]
        theta.grad = None
        loss = adjoint.warp_ssd(theta, state["B"], state["src"], state["dst"], state["space"], PARAMS, sign=-1,
                                simple=case["simple"])
        loss.sum().backward()
        return {"loss": loss.detach(), "grad": theta.grad}
    if kind == "chain":
        mh = state["chains"]
        mh.step_counter.zero_()
        mh.n_accepted.zero_()
        mh.set_theta(state["zero"])
        mh.run(case["steps"])
        return {"theta": mh.theta, "ll": mh.ll, "accepted": mh.n_accepted, "trace": mh.trace}
    reqs = [copy.copy(r) for r in state["requests"]]
    state["server"].run(reqs, keep=True, realtime=False)
    return [r.result for r in reqs]


# ------------------------------------------------------------------- work
# Floating-point operations of one Trel step (two cell lookups and an affine product) and of one RK2 substep (one
# lookup, two affine products, the midpoint and the update) by dimension; redone steps come on top and are not counted.
STEP = {1: 8, 2: 38, 3: 70}
SUBSTEP = {1: 11, 2: 41, 3: 75}
COLUMN = 40           # one substep of one column of the 2D forward sensitivity
ADJOINT_STEP = 16     # one accepted step back, 2D
ADJOINT_SUBSTEP = 71  # one RK2 substep back, 2D


def work(case):
    kind = case["kind"]
    if kind in ("points", "trajectory", "sensitivity"):
        n, dim = case["n"], len(_ncs(case))
        io = 8 * dim * n
        if kind == "points":
            return dict(bytes=2 * io, flops=n * NT * (STEP[dim] if case["what"] == "T" else NS * SUBSTEP[dim]))
        if kind == "trajectory":
            return dict(bytes=io * (NT + 2), flops=n * NT * STEP[dim])
        d = _space(case["tess"], _ncs(case))[0].d
        return dict(bytes=io * (2 + d), flops=n * NT * NS * (SUBSTEP[dim] + COLUMN * d))
    if kind == "warp":
        dim = len(_ncs(case))
        n = case["rows"] * case["cols"] * (case["slices"] or 1)
        return dict(bytes=n * (2 * 8 * dim + 8), flops=n * (NT * STEP[dim] + 16))
    if kind == "field":
        n = case["rows"] * case["cols"]
        return dict(bytes=n * (16 + 16 + 4), flops=n * 24)
    if kind == "batch":
        n = case["instances"] * (case["most"] - 1e3) / math.log(case["most"] / 1e3)  # the mean of the sizes
        return dict(bytes=32 * n, flops=n * NT * STEP[2])
    if kind == "pairs":
        n = case["pairs"] * case["n"] ** 2
        per = NT * NS * (SUBSTEP[2] + ADJOINT_SUBSTEP) if case["simple"] else NT * (STEP[2] + ADJOINT_STEP)
        return dict(bytes=8 * n, flops=n * per)
    if kind == "chain":
        n = case["n"] ** 2
        return dict(bytes=8 * n, flops=case["chains"] * (case["steps"] + 1) * n * (NT * STEP[2] + 16))
    n1, n2, n3 = 0.4 * 990000 / math.log(100), 0.4 * 279347, 0.2 * 64 ** 3  # mean points of a request, by dimension
    return dict(bytes=case["requests"] * (16 * n1 + 32 * n2 + 56 * n3),
                flops=case["requests"] * NT * (n1 * STEP[1] + n2 * STEP[2] + n3 * STEP[3]))


# ------------------------------------------------------------------ exact
class _Geo:
    """The cells of one box, or, with tensors for the counts and increments, of each point's own box."""

    def __init__(self, dim, tess, nCs, incs):
        self.dim, self.tess, self.n, self.inc = dim, tess, nCs, incs

    def at(self, idx):
        pick = [v[idx] if isinstance(v, torch.Tensor) else v for v in list(self.n) + list(self.inc)]
        return _Geo(self.dim, self.tess, pick[:self.dim], pick[self.dim:])


def _geo(sp):
    return _Geo(sp.dim_domain, sp.tess, [int(k) for k in sp.nCs], [float(x) for x in sp.incs])


def _cells(g, p):
    def box(q, n):
        q = torch.clamp(q, min=0.0)
        return torch.minimum(q, torch.as_tensor(n - 1, dtype=torch.float64, device=q.device)).round().long()

    if g.dim == 1 or g.tess == "II":
        c, stride = 0, 1
        for d in range(g.dim):
            x = p[:, d]
            inc = torch.as_tensor(g.inc[d], dtype=torch.float64, device=x.device)
            c = c + box((x - torch.fmod(x, inc)) / inc, g.n[d]) * stride
            stride = stride * g.n[d]
        return c
    fr, ix = [], []
    for d in range(g.dim):
        inc = torch.as_tensor(g.inc[d], dtype=torch.float64, device=p.device)
        top = torch.as_tensor(g.n[d] * g.inc[0 if d == 2 else d] - 1e-10, dtype=torch.float64, device=p.device)
        x = torch.minimum(torch.clamp(p[:, d], min=0.0), top)
        m = torch.fmod(x, inc)
        fr.append(m / inc)
        ix.append(box((x - m) / inc, g.n[d]))
    if g.dim == 2:
        x, y = fr
        tri = torch.where(x < y, torch.where(1 - x < y, 2, 3), torch.where(1 - x < y, 1, 0))
        px, py, ixc, iyc = p[:, 0], p[:, 1], g.inc[0], g.inc[1]
        up, down = py <= 0, py >= g.n[1] * iyc
        left, right = px <= 0, px >= g.n[0] * ixc
        sx, sy = px / ixc, py / iyc
        tl = torch.where(up & (sy < sx), 0, torch.where(down & (sy - g.n[1] > -sx), 2, 3))
        tr = torch.where(up & (-sy > sx - g.n[0]), 0, torch.where(down & (sy - g.n[1] > sx - g.n[0]), 2, 1))
        out = torch.where(left, tl, torch.where(right, tr, torch.where(up, 0, 2)))
        return (ix[0] + ix[1] * g.n[0]) * 4 + torch.where(left | right | up | down, out, tri)
    x, y, z = fr
    flip = (ix[0] + ix[1] + ix[2]) % 2 == 1
    x, y = torch.where(flip, y, x), torch.where(flip, 1 - x, y)
    tet = torch.where(-x + y - z >= 0, 3, torch.where(x - y - z >= 0, 4, 0))
    tet = torch.where(-x - y + z >= 0, 1, torch.where(x + y + z - 2 >= 0, 2, tet))
    return (ix[0] + ix[1] * g.n[0] + ix[2] * g.n[0] * g.n[1]) * 5 + tet


def _affine(tab, c, p):
    A = tab[c]
    return (A[:, :, :-1] * p[:, None, :]).sum(2) + A[:, :, -1]


def _expm(A, dt):
    """The Trels of tables (cells, dim, dim + 1)."""
    sq = torch.zeros((A.shape[0], A.shape[1] + 1, A.shape[1] + 1), dtype=torch.float64)
    sq[:, :-1] = A.cpu() * dt
    return torch.linalg.matrix_exp(sq)[:, :-1].to(A.device)


def _substep(g, A, base, p):
    c = _cells(g, p) + base
    h = DT / NS
    return p + h * _affine(A, c, p + h / 2 * _affine(A, c, p)), c


def _flow(g, A, base, p, simple=False, each=None, tape=None):
    """End points of calc_T (calc_T_simple) from the signed tables; base: each point's first table row.  each is
    called with the points after every step; tape takes every unit (kind, points' indices, start points, rows)."""
    everyone = torch.arange(p.shape[0], device=p.device)
    base = torch.zeros_like(everyone) + base
    T = None if simple else _expm(A, DT)
    for _ in range(NT):
        if simple:
            redo, p2 = everyone, p.clone()
        else:
            c = _cells(g, p) + base
            q = _affine(T, c, p)
            ok = _cells(g, q) + base == c
            redo = (~ok).nonzero()[:, 0]
            if tape is not None:
                k = ok.nonzero()[:, 0]
                tape.append(("T", k, p[k], c[k]))
            p2 = torch.where(ok[:, None], q, p)
        gr, r, b = g.at(redo), p[redo], base[redo]
        for _ in range(NS):
            r0 = r
            r, rc = _substep(gr, A, b, r0)
            if tape is not None:
                tape.append(("A", redo, r0, rc))
        p2[redo] = r
        p = p2
        if each is not None:
            each(p)
    return p


def _table(Avees, sp, sign):
    A = torch.from_numpy(np.ascontiguousarray(Avees, dtype=np.float64)).cuda()
    return sign * A.reshape(sp.nC, sp.dim_domain, sp.dim_domain + 1)


def _corners(p, shape):
    """(flat pixel index or -1, weight) of each corner of the multilinear sample at p (x first)."""
    d = p.shape[1]
    lo = torch.floor(p)
    f, lo = p - lo, lo.clamp(-4, 1 << 30).long()
    for k in range(1 << d):
        w, idx, ok = 1.0, 0, torch.ones(p.shape[0], dtype=torch.bool, device=p.device)
        for i in reversed(range(d)):
            n, up = shape[d - 1 - i], k >> i & 1
            at = lo[:, i] + up
            w = w * (f[:, i] if up else 1 - f[:, i])
            idx, ok = idx * n + at.clamp(0, n - 1), ok & (at >= 0) & (at < n)
        yield torch.where(ok, idx, -1), w


def _sample(img, p):
    flat = img.double().reshape(-1)
    return sum(w * torch.where(idx >= 0, flat[idx.clamp(min=0)], 0.0) for idx, w in _corners(p, img.shape))


def _exact_sensitivity(state, A):
    sp, g, p = state["space"], _geo(state["space"]), state["pts"]
    B = torch.from_numpy(sp.BasMats).cuda().permute(1, 0, 2, 3).contiguous()  # (cells, d, dim, dim + 1)
    q = torch.zeros((p.shape[0], sp.d, 2), dtype=torch.float64, device="cuda")
    h = DT / NS

    def slope(c, p, q):
        Bc, L = B[c], A[c][:, :, :-1]
        return (Bc[..., :-1] * p[:, None, None, :]).sum(3) + Bc[..., -1] + (L[:, None] * q[:, :, None, :]).sum(3)

    for _ in range(NT * NS):
        c = _cells(g, p)
        m = p + h / 2 * _affine(A, c, p)
        q = q + h * slope(c, m, q + h / 2 * slope(c, p, q))
        p = p + h * _affine(A, c, m)
    return {"points": p, "grad": q.transpose(1, 2).contiguous()}


def _exact_pairs(state):
    case, sp, B = state["case"], state["space"], state["B"].cpu()
    m, n = case["pairs"], case["n"]
    theta = state["theta"].detach().cpu()
    A = -(theta @ B.T).reshape(m * sp.nC, 2, 3).cuda()
    grid = torch.from_numpy(Tessellation([0, 0], [n, n], [1, 1], "II").dense_grid_img()).cuda().repeat(m, 1)
    inst = torch.arange(m, device="cuda").repeat_interleave(n * n)
    tape = []
    p = _flow(_geo(sp), A, inst * sp.nC, grid, simple=case["simple"], tape=tape)
    # the sample, its gradient and the loss
    lo = torch.floor(p)
    f, x0, y0 = p - lo, lo[:, 0].clamp(-4, n + 4).long(), lo[:, 1].clamp(-4, n + 4).long()
    src = state["src"].double().reshape(-1)

    def px(y, x):
        ok = (x >= 0) & (x < n) & (y >= 0) & (y < n)
        return torch.where(ok, src[inst * n * n + y.clamp(0, n - 1) * n + x.clamp(0, n - 1)], 0.0)

    v00, v01, v10, v11 = px(y0, x0), px(y0, x0 + 1), px(y0 + 1, x0), px(y0 + 1, x0 + 1)
    fx, fy = f[:, 0], f[:, 1]
    a, b = (1 - fx) * v00 + fx * v01, (1 - fx) * v10 + fx * v11
    r = (1 - fy) * a + fy * b - state["dst"].double().reshape(-1)
    loss = 0.5 * (r * r).reshape(m, -1).sum(1)
    lam = torch.stack([r * ((1 - fy) * (v01 - v00) + fy * (v11 - v10)), r * (b - a)], 1)
    # back through the tape
    GA, GT = torch.zeros_like(A), torch.zeros_like(A)
    T, h = _expm(A, DT), DT / NS
    one = lambda x: torch.cat([x, torch.ones_like(x[:, :1])], 1)  # noqa: E731
    for unit, k, q, c in reversed(tape):
        l = lam[k]
        if unit == "T":
            GT.index_add_(0, c, l[:, :, None] * one(q)[:, None, :])
            lam[k] = (T[c][:, :, :-1] * l[:, :, None]).sum(1)
        else:
            L = A[c][:, :, :-1]
            mid = q + h / 2 * _affine(A, c, q)
            g2 = h * l
            gm = (L * g2[:, :, None]).sum(1)
            g1 = h / 2 * gm
            lam[k] = l + gm + (L * g1[:, :, None]).sum(1)
            GA.index_add_(0, c, g2[:, :, None] * one(mid)[:, None, :] + g1[:, :, None] * one(q)[:, None, :])
    if not case["simple"]:
        Ar = A.cpu().requires_grad_(True)
        sq = torch.cat([Ar * DT, torch.zeros_like(Ar[:, :1])], 1)
        torch.linalg.matrix_exp(sq)[:, :-1].backward(GT.cpu())
        GA = GA + Ar.grad.cuda()
    return {"loss": loss, "grad": -(GA.cpu().reshape(m, -1) @ B)}


def _exact_served(state):
    srv, p = state["server"], PARAMS
    out = [None] * len(state["requests"])
    for name, kind in srv.kinds.items():
        at = [i for i, r in enumerate(state["requests"]) if r.kind == name]
        if not at:
            continue
        sp, reqs = kind.space, [state["requests"][i] for i in at]
        pts, sizes = [], []
        for r in reqs:
            if name == "1d":
                x = _uniform(r.n, 1, r.seed)
            elif name == "3d":
                x = torch.from_numpy(Tessellation([0] * 3, [serving.VOL] * 3, [1] * 3, "II").dense_grid_img()).cuda()
            else:
                x = _unit_grid(r.side, r.side)
            pts.append(x)
            sizes.append(x.shape[0])
        base = torch.repeat_interleave(torch.arange(len(reqs), device="cuda"), torch.tensor(sizes, device="cuda")) * sp.nC
        A = torch.cat([_table(sp.B @ r.theta, sp, kind.sign) for r in reqs])
        end = torch.split(_flow(_geo(sp), A, base, torch.cat(pts)), sizes)
        for i, r, e in zip(at, reqs, end):
            if name == "3d":
                vol = srv.volumes[r.seed % len(srv.volumes)]
                e = _sample(vol, e).reshape(vol.shape)
            out[i] = e
    return out


def exact(case, seed):
    """What run returns, by plain torch in 64 bits; None for a chain (hundreds of evaluations, minutes)."""
    kind = case["kind"]
    if kind == "chain":
        return None
    state = prepare(case, seed)
    if kind == "pairs":
        return _exact_pairs(state)
    if kind == "served":
        return _exact_served(state)
    if kind == "batch":
        n = torch.tensor([k for _, _, k in state["insts"]], device="cuda")
        side = torch.repeat_interleave(torch.tensor([g[0] for g, _, _ in state["insts"]], device="cuda"), n)
        cells = torch.tensor([4 * g[0] * g[1] for g, _, _ in state["insts"]], device="cuda")
        base = torch.repeat_interleave(torch.cumsum(cells, 0) - cells, n)
        g = _Geo(2, "I", [side, side], [1.0 / side.double(), 1.0 / side.double()])
        return _flow(g, state["As"].reshape(-1, 2, 3), base, state["pts"])
    if kind == "warp":
        nCs = _ncs(case)
        sp = state["tw"].L_cpa_space[0]
        inv = _flow(_geo(sp), _table(state["Avees"], sp, -1), 0, state["pts"])
        return {"points": inv, "warped": _sample(state["img"], inv).reshape(state["img"].shape)}
    sp = state["space"]
    A, g = _table(state["pat"].Avees, sp, case.get("sign", 1)), _geo(sp)
    if kind == "field":
        c = _cells(g, state["pts"])
        return {"v": _affine(A, c, state["pts"]), "cell": c.int()}
    if kind == "sensitivity":
        return _exact_sensitivity(state, A)
    if kind == "trajectory":
        rows = [state["pts"]]
        _flow(g, A, 0, state["pts"], each=rows.append)
        return torch.stack(rows)
    return _flow(g, A, 0, state["pts"], simple=case["what"] == "simple")
