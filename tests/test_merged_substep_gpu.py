"""rhs_eval_rk4_substep of the spherical BSSN bundle, one launch of its three kernels, against the
kernels launched one by one on the GPU: the same statements per output, so equal bit for bit, for
every substep, on grids of one partial tile, whole tiles, a remainder in each direction and more
tiles than one launch takes, and
with a tile shape set for one kernel only (then they are launched one by one)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [None, (16, 4, 4)])
@pytest.mark.parametrize("Nxx", [(12, 8, 2), (64, 4, 4), (70, 6, 10), (66, 128, 80)])
def test_merged_equals_separate(torch_cuda, Nxx, shape):
    torch = torch_cuda
    from nrpytutorial_amd.runtime import Bundle, Evolution, Grid, check, ptr
    print("case: merged substep %s %s" % (Nxx, shape), flush=True)
    b = Bundle("bssn_spherical_sym2")
    g = Grid(b, Nxx, BH1_mass=0.5, BH2_mass=0.5, BH1_posn_z=0.5, BH2_posn_z=-0.5)
    ev = Evolution(g)
    ev.initial_data()
    ev.apply_bcs(ev.y_n, composed=True)
    check(b.lib.Ricci_eval(g.rfm, g.pp(), ptr(ev.y_n), ptr(ev.auxevol), ev.s()), "Ricci_eval")
    groups = range(len(b.meta["rhs_groups"]))
    kid = b.meta["kernel_ids"]["rhs_eval_rk4_substep_g1"]
    try:
        if shape:
            check(b.lib.nrpy_set_block_shape(kid, *shape), "nrpy_set_block_shape")
        for S in range(4):
            results = []
            for names in (["rhs_eval_rk4_substep"], ["rhs_eval_rk4_substep_g%d" % k for k in groups]):
                rt, out = torch.ones_like(ev.y_n), torch.full_like(ev.y_n, float("nan"))
                for n in names:
                    check(getattr(b.lib, n)(S, g.rfm, g.pp(), ptr(ev.auxevol), ptr(ev.y_n), ptr(ev.y_n), ptr(rt), ptr(out),
                                            ctypes.c_double(0.01), ev.s()), n)
                torch.cuda.synchronize()
                results.append((rt, out))
            assert torch.equal(results[0][0], results[1][0])
            assert torch.equal(g.interior(results[0][1]), g.interior(results[1][1]))
            assert bool(torch.isfinite(g.interior(results[0][1])).all())
    finally:
        b.lib.nrpy_set_block_shape(kid, 0, 0, 0)
