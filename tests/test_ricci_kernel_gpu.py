"""Ricci_eval, one kernel for the six components, against the kernels of its two groups on the GPU:
the same expressions with common subexpressions taken over more outputs, so the two round differently
(each component sums under 1000 products of O(1) values: 1e-12 of its largest value). Sizes: within one tile, one
point past it in each direction, even and odd rows (the two ways tiles reach LDS)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,Nxx", [("bssn_cartesian", (16, 4, 4)), ("bssn_cartesian", (17, 5, 9)),
                                      ("bssn_cartesian", (30, 3, 5)), ("bssn_spherical_sym2", (12, 8, 2)),
                                      ("bssn_spherical_sym2", (65, 6, 2))])
def test_ricci_kernel_equals_group_kernels(torch_cuda, name, Nxx):
    torch = torch_cuda
    from nrpytutorial_amd.runtime import Bundle, Evolution, Grid, check, ptr
    from nrpytutorial_amd.workloads import bssn_gaussian_state_torch
    print("case: %s %s" % (name, Nxx), flush=True)
    b = Bundle(name)
    pars = {} if name == "bssn_cartesian" else dict(BH1_mass=0.5, BH2_mass=0.5, BH1_posn_z=0.5, BH2_posn_z=-0.5)
    g = Grid(b, Nxx, **pars)
    ev = Evolution(g)
    if name == "bssn_cartesian":
        bssn_gaussian_state_torch(ev.y_n, g.xx_dev, b.evol, 2)
    else:
        ev.initial_data()
    ev.apply_bcs(ev.y_n, composed=True)
    one, two = (torch.full((6,) + g.shape, float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
    check(b.lib.Ricci_eval(g.rfm, g.pp(), ptr(ev.y_n), ptr(one), ev.s()), "Ricci_eval")
    for k in range(2):
        check(getattr(b.lib, "Ricci_eval_g%d" % k)(g.rfm, g.pp(), ptr(ev.y_n), ptr(two), ev.s()), "Ricci_eval_g")
    torch.cuda.synchronize()
    for q in range(6):
        a, c = g.interior(one[q]), g.interior(two[q])
        assert float((a - c).abs().max()) <= 1e-12 * float(g.interior(two).abs().max())
    G = b.NGHOSTS
    ghost = torch.ones(g.shape, dtype=torch.bool, device="cuda")
    ghost[G:-G, G:-G, G:-G] = False
    assert bool(torch.isnan(one[:, ghost]).all())
