"""BSSNStepAdjoint.step_back on tensors its kernels cannot take as they are (another stride order,
another type, one tensor as state and cotangent), and on repeated use, on the GPU: the result is that
of contiguous float64 tensors bit for bit, and the state is left as it was."""
import pytest

pytestmark = pytest.mark.gpu


def test_step_back_takes_any_tensor(torch_cuda):
    torch = torch_cuda
    from nrpytutorial_amd.adjoint import BSSNStepAdjoint
    from nrpytutorial_amd.runtime import Bundle, Evolution, Grid
    from nrpytutorial_amd.workloads import bssn_gaussian_state_torch
    print("case: step_back operands", flush=True)
    b = Bundle("bssn_cartesian")
    g = Grid(b, (9, 6, 5))
    ev = Evolution(g)
    bssn_gaussian_state_torch(ev.y_n, g.xx_dev, b.evol, 3)
    ev.apply_bcs(ev.y_n, composed=True)
    ev.post_bcs(ev.y_n)
    y = ev.y_n.clone()
    gen = torch.Generator(device="cuda").manual_seed(4)
    lam = torch.zeros_like(y)
    # values that float32 holds exactly, so the float32 operand is the same cotangent
    g.interior(lam).copy_(torch.randn(g.interior(lam).shape, generator=gen, device="cuda"))
    dt = g.find_timestep(0.5)
    adj = BSSNStepAdjoint(ev)
    want = lam.clone()
    adj.step_back(y, want, dt)
    assert bool(torch.equal(y, ev.y_n)) and bool(torch.isfinite(want).all())

    def strided(a):
        return a.permute(0, 3, 2, 1).contiguous().permute(0, 3, 2, 1)
    got = strided(lam)
    adj.step_back(strided(y), got, dt)
    assert bool(torch.equal(got, want))
    got = lam.float()
    adj.step_back(y, got, dt)
    assert bool(torch.equal(got, want.float()))
    same = y.clone()                                    # state and cotangent in one tensor
    adj.step_back(same, same, dt)
    other = y.clone()
    adj.step_back(y, other, dt)
    assert bool(torch.equal(same, other))
