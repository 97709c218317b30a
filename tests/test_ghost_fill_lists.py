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
    print("%s: %d ghosts, %d read by stencils" % (name, (~inside).sum(), read.sum()))
    assert generic == 0                 # the generic form is for four ghost layers: test_ghost_fill_generic.py


# kernels of the RK4 step: substeps (also as one launch of several, "body", and over a batch) and
# Ricci tensor; the merged kernel itself only calls the bodies
STEP_KERNEL = re.compile(r"\n(?:__global__|static __device__) [^\n]*?\b((?:rhs_eval_rk4_substep\w*?|Ricci_eval(?:_g\d+)?)"
                         r"__(?:gpu_batched|gpu|body))\(")
PLAIN = re.compile(r"double (\w+) = (in_gfs|auxevol_gfs)\[IDX4\((\w+)GF, i0([+-]\d+)?,i1([+-]\d+)?,i2([+-]\d+)?\)\];")
HALO = re.compile(r"in_gfs\[IDX4\(\w+GF, nrpy_xl < (\d+) \? i0 - (\d+) : i0 \+ (\d+),i1,i2\)\];")
BOX = re.compile(r"copy the \((\d+) x (\d+) x (\d+)\)-point box")
LDS = re.compile(r"double (\w+) = nrpy_lds\[\d+\]\[nrpy_li \+ (-?\d+)\];")
MOVE = re.compile(r"double (\w+) = nrpy_xshift<\d+, \d+, (-?\d+)>\(")
NAMED = re.compile(r"_i0(?:([pm])(\d+))?_i1(?:([pm])(\d+))?_i2(?:([pm])(\d+))?$")


def _named(name):
    """The offset in the name that the finite-difference emitter gives a read (none: the centre)."""
    m = NAMED.search(name)
    if not m:
        return (0, 0, 0)
    return tuple((-1 if m.group(2 * d + 1) == "m" else 1) * int(m.group(2 * d + 2) or 0) for d in range(3))


def _kernel_offsets(kernel):
    """(offsets a kernel reads gridfunctions at, number of reads by kind), from the addresses: plain reads,
    reads of an LDS box (split into rows and planes of the box), lane moves and their halo loads."""
    found, kinds = [], {"plain": 0, "lds": 0, "move": 0}
    for name, _, _, *o in PLAIN.findall(kernel):
        found.append((name, tuple(int(v or 0) for v in o)))
        kinds["plain"] += 1
    for a, b, c in HALO.findall(kernel):
        assert a == b == c
        found += [("nrpy_h", (int(a), 0, 0)), ("nrpy_h", (-int(a), 0, 0))]
    box = [tuple(int(v) for v in m) for m in BOX.findall(kernel)]
    assert len(box) <= 1
    for name, k in LDS.findall(kernel):
        bx, by, _ = box[0]
        k, o = int(k), []
        for n in (bx, by):
            r = (k + n // 2) % n - n // 2
            o.append(r)
            k = (k - r) // n
        found.append((name, tuple(o) + (k,)))
        kinds["lds"] += 1
    for name, k in MOVE.findall(kernel):
        found.append((name, (int(k), 0, 0)))
        kinds["move"] += 1
    for name, o in found:
        assert name.startswith("nrpy_") or _named(name) == o, (name, o)
    # nothing that reads a gridfunction went unrecognised
    assert len(re.findall(r"\bin_gfs\[IDX4\(|\bauxevol_gfs\[IDX4\(\w+GF, i0[^\]]*\)\];", kernel)) == \
        kinds["plain"] + len(HALO.findall(kernel))
    assert kernel.count("[nrpy_li + ") == kinds["lds"] and kernel.count("nrpy_xshift<") == kinds["move"]
    return {o for _, o in found} - {(0, 0, 0)}, kinds


SUBSTEP = ["rhs_eval_rk4_substep__gpu"]
GROUPS = ["rhs_eval_rk4_substep_g%d__gpu" % k for k in range(3)]
RICCI = ["Ricci_eval__gpu", "Ricci_eval_g0__gpu", "Ricci_eval_g1__gpu"]
BATCHED = ["Ricci_eval__gpu_batched"] + [k + "_batched" for k in GROUPS]
KERNELS = {"scalarwave_cartesian": SUBSTEP + ["rhs_eval_rk4_substep_edge__gpu", "rhs_eval_rk4_substep_shell__gpu"],
           "maxwell_cartesian": SUBSTEP + ["rhs_eval_rk4_substep_edge__gpu", "rhs_eval_rk4_substep_shell__gpu"],
           "bssn_cartesian": GROUPS + RICCI + BATCHED,
           "bssn_spherical_sym2": GROUPS + RICCI + BATCHED + [k.replace("gpu", "body") for k in GROUPS],
           "maxwell_sinhcylindrical": SUBSTEP + ["rhs_eval_rk4_substep_rim__gpu"],
           "scalarwave_symtp": SUBSTEP + ["rhs_eval_rk4_substep_rim__gpu"],
           "scalarwave_sinhsphericalv2": SUBSTEP + ["rhs_eval_rk4_substep_rim__gpu"]}


@pytest.mark.parametrize("name", sorted(KERNELS))
def test_stage_offsets_are_what_the_step_kernels_read(name):
    """The list holds exactly the offsets at which the bundle's substep and Ricci kernels read gridfunctions
    (plain reads, LDS boxes and lane moves), each kernel named above among them."""
    text = open(os.path.join(GENDIR, name + ".hip")).read()
    offsets, read, kernels, kinds = set(_offsets(name)), set(), [], {"plain": 0, "lds": 0, "move": 0}
    for m in STEP_KERNEL.finditer(text):
        if m.group(1) == "rhs_eval_rk4_substep_merged__gpu":
            continue
        o, n = _kernel_offsets(text[m.start():text.index("\n}\n", m.start())])
        assert o and o <= offsets, (m.group(1), sorted(o - offsets))
        read |= o
        kernels.append(m.group(1))
        for k in kinds:
            kinds[k] += n[k]
    assert sorted(kernels) == sorted(KERNELS[name])
    assert read == offsets
    print("%s: %d offsets, %s" % (name, len(offsets), kinds))
    assert kinds["plain"] > 0 and (kinds["lds"] > 0 and kinds["move"] > 0) == (name == "bssn_cartesian")
