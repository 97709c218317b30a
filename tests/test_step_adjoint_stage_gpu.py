"""MoL_step_adjoint's stage kernels against the general path on the GPU: rhs_eval_vjp (pass 1 into
slots, pass 2), bc_apply_T and the stage updates in torch. The sizes are those where the kernel can
go wrong: axes whose two edges' extrapolations overlap (3 to 6 points), one point to either side of
a tile, the largest within a tile.

Both sum the same products, with constants multiplied in at other places: a w sums at most 3 x 5
stencil terms and what at most 3 x 2 ghost layers hand back, each with weights below 16/3 /dx^2, so
two results differ by under 64 roundings of the largest term per stage, 256 eps over the four."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bundle", ["scalarwave_cartesian", "maxwell_cartesian"])
@pytest.mark.parametrize("Nxx", [(3, 3, 3), (4, 5, 6), (65, 5, 3), (64, 4, 9), (63, 3, 4)])
def test_stage_kernels_equal_general_path(torch_cuda, bundle, Nxx):
    torch = torch_cuda
    from nrpytutorial_amd.adjoint import RK4Adjoint
    from nrpytutorial_amd.runtime import Bundle, Evolution, Grid, check, ptr
    print("case: %s %s" % (bundle, Nxx), flush=True)
    b = Bundle(bundle)
    g = Grid(b, Nxx)
    ev = Evolution(g)
    adj = RK4Adjoint(ev)
    n = len(b.evol)
    gen = torch.Generator(device="cuda").manual_seed(3)
    L = torch.zeros((n,) + g.shape, dtype=torch.float64, device="cuda")
    g.interior(L).copy_(torch.randn(g.interior(L).shape, generator=gen, dtype=torch.float64, device="cuda"))
    dt = g.find_timestep(0.5)
    f = b.lib.rhs_eval_vjp
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p] * 8
    state = g.empty(n).zero_()

    def w(kbar):
        out = g.empty(n)
        check(f(g.pp(), None, ptr(state), ptr(kbar), ptr(adj.G), ptr(out), None, ev.s()), "rhs_eval_vjp")
        adj.bc_T(out)
        return out
    w3 = w(dt / 6 * L)
    w2 = w(dt / 3 * L + dt * w3)
    w1 = w(dt / 3 * L + dt / 2 * w2)
    w0 = w(dt / 6 * L + dt / 2 * w1)
    want = L + w3 + w2 + w1 + w0
    got = L.clone()
    for a in adj.U + [adj.acc, adj.kbar, adj.w]:
        a.fill_(float("nan"))                # scratch: what is read of it has been written before
    adj.step_back(state, got, dt)
    torch.cuda.synchronize()
    size = max(float(a.abs().max()) for a in (L, w3, w2, w1, w0))
    assert float((got - want).abs().max()) <= 256 * torch.finfo(torch.float64).eps * size
    ghost = torch.ones(g.shape, dtype=torch.bool, device="cuda")
    G = b.NGHOSTS
    ghost[G:-G, G:-G, G:-G] = False
    assert float(got[:, ghost].abs().max()) == 0.0


@pytest.mark.parametrize("bundle", ["scalarwave_cartesian", "maxwell_cartesian"])
def test_unused_arguments_are_not_written(torch_cuda, bundle):
    """A linear right-hand side's adjoint needs no stage states: U1, U2, U3, rt and vjp_G may be any
    arrays, here the state itself, and keep what they hold."""
    torch = torch_cuda
    from nrpytutorial_amd.adjoint import RK4Adjoint
    from nrpytutorial_amd.runtime import Bundle, Evolution, Grid, check, ptr
    print("case: %s unused arguments" % bundle, flush=True)
    g = Grid(Bundle(bundle), (9, 6, 5))
    ev = Evolution(g)
    adj = RK4Adjoint(ev)
    gen = torch.Generator(device="cuda").manual_seed(7)
    state = torch.randn(ev.y_n.shape, generator=gen, dtype=torch.float64, device="cuda")
    lam = torch.zeros_like(state)
    g.interior(lam).copy_(torch.randn(g.interior(lam).shape, generator=gen, dtype=torch.float64, device="cuda"))
    dt = g.find_timestep(0.5)
    want, before = lam.clone(), state.clone()
    adj.step_back(state, want, dt)
    p = ptr(state)
    check(adj.lib.MoL_step_adjoint(g.rfm, g.pp(), g.bc, p, ptr(lam), p, p, p, p, ptr(adj.acc), ptr(adj.kbar), ptr(adj.w), p,
                                   ptr(ev.auxevol), float(dt), ev.s()), "MoL_step_adjoint")
    torch.cuda.synchronize()
    assert bool(torch.equal(state, before)) and bool(torch.equal(lam, want))
