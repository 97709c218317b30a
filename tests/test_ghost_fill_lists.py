"""The ghost fill's row lists (bcstruct_get_fill) on the CPU: every row, expanded as the fill
kernel expands it, is the composed map's row entry by entry; the list of every ghost covers
each once; and the list of a stage holds exactly the ghosts that some stencil of the bundle's
step kernels reads, found by brute force over all interior points and offsets. The grids
include sides shorter than the extrapolation's three points plus the ghost zones."""
import ctypes
import os
import re

import numpy as np
import pytest

from nrpytutorial_amd.runtime import Bundle, GENDIR, HostBC

CASES = [("scalarwave_cartesian", (9, 7, 5)), ("maxwell_cartesian", (3, 6, 4)), ("bssn_cartesian", (7, 6, 5)),
         ("bssn_spherical_sym2", (10, 8, 2)), ("scalarwave_sinhsphericalv2", (8, 6, 4)),
         ("scalarwave_sinhcylindricalv2", (6, 4, 8)), ("scalarwave_symtp", (8, 6, 4)),
         ("maxwell_sinhcylindrical", (6, 4, 8))]
GENERIC = 1 << 30


def _fill(h, stage):
    f = h.bundle.lib.bcstruct_get_fill
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p, ctypes.c_int] + [ctypes.c_void_p] * 6
    n, m = ctypes.c_int(), ctypes.c_int()
    assert f(h.h, stage, ctypes.byref(n), ctypes.byref(m), None, None, None, None) == 0
    rows = np.zeros((n.value, 4), np.int32)
    coeff, src, neg = np.zeros(m.value), np.zeros(m.value, np.int32), np.zeros(m.value, np.int32)
    assert f(h.h, stage, None, None, rows.ctypes.data, coeff.ctypes.data, src.ctypes.data, neg.ctypes.data) == 0
    return rows, coeff, src, neg


def _expand(row, coeff, src, neg, N0, N01):
    """{(source, negmask): coefficient} of a row."""
    dest, base, code, mask = (int(v) for v in row)
    if code == GENERIC:
        return {(int(src[base + k]), int(neg[base + k])): float(coeff[base + k]) for k in range(mask)}
    terms = {base: 1.0}
    for d, s in enumerate((1, N0, N01)):
        c = (code >> (3 * d)) & 7
        if c == 0:
            continue
        l = c - 3 if c > 3 else c
        s = -s if c > 3 else s
        w = (0.5 * (l + 1) * (l + 2), -float(l * (l + 2)), 0.5 * l * (l + 1))
        terms = {p + a * s: v * w[a] for p, v in terms.items() for a in range(3)}
    return {(p, mask): v for p, v in terms.items()}


def _offsets(bundle):
    text = open(os.path.join(GENDIR, bundle + ".hip")).read()
    body = re.search(r"nrpy_stage_offsets\[\d+\]\[3\] = \{(.*)\};", text).group(1)
    return [tuple(int(v) for v in m) for m in re.findall(r"\{(-?\d+), (-?\d+), (-?\d+)\}", body)]


@pytest.mark.parametrize("name,Nxx", CASES, ids=["%s-%dx%dx%d" % ((n,) + g) for n, g in CASES])
def test_fill_lists_are_the_composed_map(name, Nxx):
    b = Bundle(name)
    h = HostBC(b, Nxx)
    G = b.NGHOSTS
    N = [v + 2 * G for v in Nxx]
    gdest, rowptr, src, coeff, neg = h.composed()
    want = {int(gdest[r]): {(int(src[k]), int(neg[k])): float(coeff[k]) for k in range(rowptr[r], rowptr[r + 1])}
            for r in range(len(gdest))}
    offsets = _offsets(name)
    inside = np.zeros((N[2], N[1], N[0]), bool)
    inside[G:-G, G:-G, G:-G] = True
    read = np.zeros_like(inside)
    for o0, o1, o2 in offsets:
        read[G + o2:N[2] - G + o2, G + o1:N[1] - G + o1, G + o0:N[0] - G + o0] = True
    read &= ~inside
    generic = 0
    for stage, points in ((0, ~inside), (1, read)):
        rows, fc, fs, fn = _fill(h, stage)
        assert sorted(rows[:, 0].tolist()) == np.flatnonzero(points.ravel()).tolist()
        for row in rows:
            assert _expand(row, fc, fs, fn, N[0], N[0] * N[1]) == want[int(row[0])]
        generic += int((rows[:, 2] == GENERIC).sum())
    print("%s: %d ghosts, %d read by stencils, %d generic rows" % (name, (~inside).sum(), read.sum(), generic))


@pytest.mark.parametrize("name", ["scalarwave_cartesian", "bssn_cartesian", "bssn_spherical_sym2", "maxwell_sinhcylindrical"])
def test_stage_offsets_are_what_the_step_kernels_read(name):
    """Every offset at which a substep kernel or Ricci kernel of the bundle reads a gridfunction
    (plain reads, LDS boxes and lane moves) is in the list."""
    text = open(os.path.join(GENDIR, name + ".hip")).read()
    offsets = set(_offsets(name))
    for m in re.finditer(r"\n__global__ void __launch_bounds__\([^)]*\) (rhs_eval_rk4_substep\w*|Ricci_eval_g\d+)__gpu\(", text):
        kernel = text[m.start():text.index("\n}\n", m.start())]
        for o in re.findall(r"in_gfs\[IDX4\(\w+GF, i0([+-]\d+)?,i1([+-]\d+)?,i2([+-]\d+)?\)\]", kernel):
            o = tuple(int(v or 0) for v in o)
            assert o == (0, 0, 0) or o in offsets, (m.group(1), o)
