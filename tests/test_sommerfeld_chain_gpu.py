"""The captured Sommerfeld step of the curvilinear bundles (two launches per substep: the interior
RHS with its update, then every ghost point through its chain of inward neighbours) against the
step in the reference's order (MoL_step_forward_in_time_sommerfeld_unfused), to rounding after
each of three steps, on grids that are not multiples of the tiles and on the shortest axes the
radial stencils and the parity maps take. Two evolutions that share one grid are stepped in
turn, so scratch memory that belonged to the grid would show."""
import ctypes

import numpy as np
import pytest

from test_sommerfeld_gpu import CASES, _setup

pytestmark = pytest.mark.gpu
CURVILINEAR = [c for c in CASES if "cartesian" not in c[0]]


def _launches(b, graph):
    """Nodes of a captured step (MoL_graph begins with its hipGraph_t)."""
    n = ctypes.c_size_t()
    handle = ctypes.cast(graph, ctypes.POINTER(ctypes.c_void_p))[0]
    assert b.lib.hipGraphGetNodes(ctypes.c_void_p(handle), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("Nxx", [(20, 18, 16), (9, 4, 10), (33, 6, 12)], ids=str)
@pytest.mark.parametrize("bundle,pars", CURVILINEAR, ids=[c[0] for c in CURVILINEAR])
def test_captured_step_equals_unfused(torch_cuda, bundle, pars, Nxx):
    torch = torch_cuda
    from nrpytutorial_amd.runtime import Evolution
    print("case: %s captured vs unfused Sommerfeld step, Nxx=%s" % (bundle, Nxx), flush=True)
    b, g, ev, og, y = _setup(torch, bundle, pars, Nxx)
    first = torch.from_numpy(y).cuda()
    other, ref, ref2 = Evolution(g), Evolution(g), Evolution(g)
    for e, f in ((ev, 1.0), (other, 0.5), (ref, 1.0), (ref2, 0.5)):
        e.y_n.copy_(first * f)
    dt = 0.25 * g.find_timestep(0.5)
    for step in range(3):
        for e in (ev, other):
            e.step_sommerfeld(dt, 1)
        for e in (ref, ref2):
            e.step_sommerfeld(dt, 1, unfused=True)
        torch.cuda.synchronize()
        for e in (ev, other):
            assert _launches(b, e.som_graph) == 8       # two a substep: not the unfused step, captured
        for e, r in ((ev, ref), (other, ref2)):
            assert np.isfinite(r.y_n.cpu().numpy()).all()
            for got, want in ((e.y_n, r.y_n), (e.rt, r.rt)):
                # the same operations; the compiler may contract another multiply-add of a point's two
                # evaluations, 1 ulp of X, carried through at most nine chained points and 12 stages
                off = float((got - want).abs().max() / want.abs().max())
                assert off < 1e-13, "step %d: %.2e" % (step, off)
    ev.free_graph()
    other.free_graph()


@pytest.mark.parametrize("bundle,pars", CURVILINEAR, ids=[c[0] for c in CURVILINEAR])
def test_captured_step_reads_xx_at_launch(torch_cuda, bundle, pars):
    """The coordinates that enter a replay are those in xx when the launch's stream comes to it: not
    those of the graph's creation (NaN here), nor of an earlier launch (stretched in between), and
    with the writes still queued on the launch's stream."""
    torch = torch_cuda
    from nrpytutorial_amd.runtime import Evolution
    Nxx = (9, 4, 10)
    print("case: %s captured Sommerfeld step, xx changed between launches" % bundle, flush=True)
    b, g, ev, og, y = _setup(torch, bundle, pars, Nxx)
    first = torch.from_numpy(y).cuda()
    ref = Evolution(g)
    for e in (ev, ref):
        e.y_n.copy_(first)
    dt = 0.25 * g.find_timestep(0.5)
    saved = [x.clone() for x in g.xx_dev]
    for x in g.xx_dev:
        x.fill_(float("nan"))
    ev.step_sommerfeld(dt, 0)                   # creates the graph
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    for scale in (1.0, 1.01):
        with torch.cuda.stream(stream):
            queue = torch.ones(1 << 24, device="cuda")
            for _ in range(20):                 # work in front of the writes
                queue.mul_(1.0001)
            for x, s in zip(g.xx_dev, saved):
                x.copy_(s * scale)
            ev.step_sommerfeld(dt, 2)
            ref.step_sommerfeld(dt, 2, unfused=True)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(ref.y_n).all())
        off = float((ev.y_n - ref.y_n).abs().max() / ref.y_n.abs().max())
        assert off < 1e-13, "scale %g: %.2e" % (scale, off)
    ev.free_graph()
