"""The adjoint where device memory has no room for its whole workspace.

It then runs its blocks in parts that share a smaller workspace: the same bits
as in one part.  The memory is filled to leave a third of what the call would
take (both maps, one instance and several, a last block that is not full)."""
import numpy as np
import pytest

from cpabdiffeo_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inst,N,trel", [(8, 250000, True), (1, 2000037, True), (1, 2000037, False)])
def test_parts_give_the_same_bits(gpu, inst, N, trel):
    torch = gpu
    nT, nS, dt = 100, 3, 0.01
    need = inst * N * nT * (18 if trel else 16)
    assert need > 2 << 30
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        pytest.skip("needs %.0f GB of free device memory" % (need / 2**30 + 4))
    print("[gpu] adjoint memory", inst, N, trel, flush=True)
    sp = configs.unit_space((4, 4), "I")
    rng = np.random.default_rng(29)
    A = np.stack([(sp.B @ rng.normal(size=sp.d)).reshape(sp.nC, 6) for _ in range(inst)])
    dA = torch.from_numpy(A / np.abs(A).max()).cuda()
    sA, T = torch.empty_like(dA), torch.empty_like(dA)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(30)
    pts = torch.rand((inst, N, 2), dtype=torch.float64, device="cuda", generator=gen)
    lam = torch.rand((inst, N, 2), dtype=torch.float64, device="cuda", generator=gen)

    def run(ctx):
        pos, g = torch.empty_like(pts), torch.empty_like(dA)
        args = [dt, nT, nS, N, 4, 4, 0.25, 0.25, pos.data_ptr(), g.data_ptr()]
        head = [1, sp.nC, inst, pts.data_ptr(), lam.data_ptr()]
        if trel:
            ctx.call("cpab_calc_T_vjp", *head, T.data_ptr(), sA.data_ptr(), *args)
        else:
            ctx.call("cpab_calc_T_simple_vjp", *head, sA.data_ptr(), *args)
        ctx.synchronize()
        return pos, g

    whole, parts = _lib.Context(0), _lib.Context(0)
    filler = None
    try:
        for c in (whole, parts):
            c.bind_stream(torch.cuda.current_stream().cuda_stream)
        whole.call("cpab_prep_trels", 2, inst * sp.nC, dA.data_ptr(), 1, dt, sA.data_ptr(), T.data_ptr())
        want_pos, want_g = run(whole)
        room = torch.empty((2, inst * N, 2), dtype=torch.float64, device="cuda")  # (the second run's results)
        filler = torch.empty(torch.cuda.mem_get_info()[0] - need // 3 - (64 << 20), dtype=torch.uint8, device="cuda")
        del room
        pos, g = run(parts)
        assert torch.equal(pos, want_pos) and torch.equal(g, want_g)
        assert bool(torch.isfinite(g).all()) and bool((g != 0).any())
    finally:
        del filler
        torch.cuda.empty_cache()
        for c in (whole, parts):
            _lib.lib().cpab_destroy(c.handle)
