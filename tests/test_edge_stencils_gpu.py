"""The Cartesian scalar-wave and Maxwell RK4 step, whose substeps 1-3 extrapolate the ghost values of
their stencils in registers instead of reading a filled ghost zone, against the same step composed
from the single calls (rhs_eval_rk4_substep, then the composed ghost fill, four times): the state
with its ghosts after each of three steps, on the shortest axes the extrapolation takes, around the
tile width, and with stage arrays that hold NaN before the first step (nothing unfilled is used).
The extrapolations are the same operations in the same order; 1e-14 of the largest value allows
for another contraction of the sums behind them."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
SIZES = [(3, 3, 3), (4, 3, 5), (5, 6, 3), (64, 4, 3), (66, 9, 4), (127, 5, 7)]


@pytest.mark.parametrize("Nxx", SIZES, ids=str)
@pytest.mark.parametrize("name", ["scalarwave_cartesian", "maxwell_cartesian"])
def test_step_equals_filled_substeps(torch_cuda, name, Nxx):
    torch = torch_cuda
    from nrpytutorial_amd.runtime import Bundle, Grid, Evolution, check, ptr
    print("case: %s edge stencils Nxx=%s" % (name, Nxx), flush=True)
    g = Grid(Bundle(name), Nxx)
    ev, ref = Evolution(g), Evolution(g)
    gen = torch.Generator(device="cuda").manual_seed(5)
    ev.y_n.copy_(torch.randn(ev.y_n.shape, dtype=torch.float64, device="cuda", generator=gen))
    ref.y_n.copy_(ev.y_n)                      # the first step starts from these ghosts, filled or not
    for a in (ev.k_odd, ev.k_even, ev.rt):
        a.fill_(float("nan"))
    dt = 0.1 * min(g.params.dxx0, g.params.dxx1, g.params.dxx2)
    f = g.bundle.lib.rhs_eval_rk4_substep
    for step in range(3):
        ev.step(dt, 1, use_graph=step > 0)
        for s, (i, o) in enumerate(((ref.y_n, ref.k_odd), (ref.k_odd, ref.k_even), (ref.k_even, ref.k_odd),
                                    (ref.k_odd, ref.y_n))):
            check(f(s, g.rfm, g.pp(), ptr(ref.auxevol), ptr(i), ptr(ref.y_n), ptr(ref.rt), ptr(o), ctypes.c_double(dt),
                    ref.s()), "rhs_eval_rk4_substep")
            ref.apply_bcs(o, composed=True)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(ev.y_n).all())
        assert float((ev.y_n - ref.y_n).abs().max()) <= 1e-14 * float(ref.y_n.abs().max()), step
    ev.free_graph()
