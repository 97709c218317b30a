"""Vector-Jacobian products of finite-difference right-hand sides.

For a right-hand side generated by FD_outputC, the value of output o at an
interior point p is F_o(s_1(p), ..., s_m(p)): a pointwise SymPy expression of
"slots" s_k, each of which is either a gridfunction value at p or a linear
finite-difference stencil D_k of one gridfunction around p (an upwinded
derivative is UpWind*D_up + (1-UpWind)*D_dn with UpWind = (beta^k > 0), which
is piecewise constant in beta). Given a cotangent v_o(p) on the outputs,

    G_k(p)        = sum_o v_o(p) dF_o/ds_k(p)                 (pass 1, pointwise)
    ybar_Y(q)     = G_{Y}(q) + sum_{k on Y} sum_t w_{k,t} G_k(q - t)   (pass 2, transposed stencils)

where the second sum runs over the slots that differentiate gridfunction Y,
t over the stencil offsets of slot k with weights w_{k,t} (including the
1/dx factors), and only interior points q - t contribute. Pass 2 runs over
all points, so ybar holds cotangents at ghost points too; the boundary
transpose (bc_apply_T) folds those back onto the interior points they were
copied or extrapolated from.

Pass 1 is generated by reverse-mode differentiation of the CSE'd forward
expression list: the forward statements are emitted unchanged, then one
adjoint statement per forward temporary in reverse order, adj_t = sum over
consumers c of adj_c * d e_c / d t, then one write per slot. The code is a
small multiple of the forward code, and every derivative is of a small CSE'd
subexpression.
"""
import sympy as sp

from .. import grid as gri
from .. import finite_difference as fin
from .. import loop as lp
from .. import outputC as oc
from .. import reference_metric as rfm
from . import schedule

_PRINT = oc._Printer()


def _ccode(e):
    return _PRINT.doprint(sp.sympify(e))


def _out_name(lhs):
    """'rhs_gfs[IDX4(HDD00GF, i0, i1, i2)]' -> gridfunction name 'hDD00'."""
    tag = lhs.split("IDX4(")[1].split(",")[0].strip()
    for g in gri.glb_gridfcs_list:
        if g.name.upper() + "GF" == tag:
            return g.name
    raise ValueError("cannot identify the output gridfunction of " + lhs)


def _is_slot(sym, deriv_names):
    n = str(sym)
    if n in deriv_names:
        return True
    return gri.variable_type(sym) == "gridfunction"


def vjp_pointwise_body(exprs, upwindcontrolvec="", slot_offset=0, existing=None):
    """C body of pass 1 and the list of its new slots [(slot name, kind, gf, op)].

    kind is "value" (gridfunction value), "deriv" (stencil op on gf), or
    "upwind_up" / "upwind_dn" (the two stencils of an upwinded derivative).
    New slots are written to vjp_G gridfunctions slot_offset, slot_offset + 1, ...;
    a slot named in ``existing`` (slot name -> vjp_G index, from an earlier pass-1
    kernel of the same VJP) is accumulated into instead."""
    existing = existing or {}
    read_block, _, _, derivs = fin.FD_outputC_readblock(exprs, upwindcontrolvec)
    rhs = [sp.sympify(e.rhs) for e in exprs]
    outs = [_out_name(e.lhs) for e in exprs]
    cots = [sp.Symbol("cot_" + n, real=True) for n in outs]
    deriv_names = {str(d) for d in derivs if "_ddnD" not in str(d)}
    repl, red = sp.cse(rhs, sp.numbered_symbols("VJPf_"), order="canonical")
    temps = {t for t, _ in repl}

    adj_terms = {}

    def add(sym, term):
        adj_terms.setdefault(sym, []).append(term)

    # Only temporaries that depend on a slot need adjoints (the rest are constants such
    # as powers of parameters or reference-metric factors).
    active = set()
    for t, e in repl:
        if any((a in active) or _is_slot(a, deriv_names) for a in e.free_symbols):
            active.add(t)

    def tracked(a):
        return a in active or (a not in temps and _is_slot(a, deriv_names))

    for c, e in zip(cots, red):
        for a in e.free_symbols:
            if tracked(a):
                add(a, c * sp.diff(e, a))
    lines = []
    for t, e in repl:
        lines.append("const double %s = %s;" % (t, _ccode(e)))
    for n, c in zip(outs, cots):
        lines.append("const double %s = cot_rhs_gfs[IDX4(%sGF, i0, i1, i2)];" % (c, n.upper()))
    # the reverse sweep, as (index of the forward temporary, line or None)
    sweep = []
    for k in reversed(range(len(repl))):
        t, e = repl[k]
        terms = adj_terms.get(t)
        if not terms:
            sweep.append((k, None))
            continue
        at = sp.Symbol("adj_" + str(t), real=True)
        sweep.append((k, "const double %s = %s;" % (at, _ccode(sp.Add(*terms)))))
        for a in e.free_symbols:
            if tracked(a):
                add(a, at * sp.diff(e, a))
    # A slot's adjoint is complete once the sweep has passed the earliest forward
    # temporary that reads it; its write goes there, so the adjoints it sums need not stay
    # live until the end of the sweep (slot numbering stays by name).
    first_use = {}
    for k, (t, e) in enumerate(repl):
        for a in e.free_symbols:
            if a not in temps and a not in first_use:
                first_use[a] = k
    slot_lines = {}
    slots = []
    slot_syms = sorted((s for s in adj_terms if s not in temps), key=str)
    for s in slot_syms:
        name = str(s)
        g = sp.Add(*adj_terms[s])
        out = slot_lines.setdefault(first_use.get(s, -1), [])
        if name in deriv_names:
            base, op = fin.split_deriv_var(name)
            if "dupD" in op and upwindcontrolvec != "":
                uw = "UpWind" + op[-1]
                out.append("const double adj_%s = %s;" % (name, _ccode(g)))
                for tag, kind, o2, val in (("__up", "upwind_up", op, "%s * adj_%s" % (uw, name)),
                                           ("__dn", "upwind_dn", op.replace("dupD", "ddnD"),
                                            "(1.0 - %s) * adj_%s" % (uw, name))):
                    if name + tag in existing:
                        out.append("vjp_G[IDX4(%d, i0, i1, i2)] += %s;" % (existing[name + tag], val))
                    else:
                        slots.append((name + tag, kind, base, o2))
                        out.append("vjp_G[IDX4(%d, i0, i1, i2)] = %s;" % (slot_offset + len(slots) - 1, val))
                continue
            entry = (name, "deriv", base, op)
        else:
            entry = (name, "value", name, None)
        if name in existing:
            out.append("vjp_G[IDX4(%d, i0, i1, i2)] += %s;" % (existing[name], _ccode(g)))
            continue
        slots.append(entry)
        out.append("vjp_G[IDX4(%d, i0, i1, i2)] = %s;" % (slot_offset + len(slots) - 1, _ccode(g)))
    lines += slot_lines.pop(-1, [])
    for k, line in sweep:
        if line:
            lines.append(line)
        lines += slot_lines.pop(k, [])
    assert not slot_lines
    body = read_block + "/* Reverse sweep: forward temporaries, then their adjoints in reverse order */\n"
    body += "\n".join(lines) + "\n"
    # The adjoint depends on the state unless every emitted adjoint expression is free of
    # forward temporaries, gridfunction values and derivatives (a linear right-hand side).
    used = set()
    for terms in adj_terms.values():
        for t in terms:
            used |= sp.sympify(t).free_symbols
    state_dependent = any(a in active or (a not in temps and _is_slot(a, deriv_names)) or str(a).startswith("UpWind")
                          for a in used)
    return body, slots, state_dependent


def vjp_transpose_bodies(slots, all_points=False):
    """C body of pass 2 (all points): for each gridfunction with a slot, the
    value-slot term plus every derivative slot's transposed stencil. Slots with the
    same operator on the same gridfunction (written by different pass-1 groups) are
    summed before the stencil weights apply. Returns {gf name: C block writing its
    cotangent}."""
    invdx = [sp.Symbol("invdx%d" % d, real=True) for d in range(3)]
    per_gf = {}
    for k, (name, kind, gf, op) in enumerate(slots):
        ops = per_gf.setdefault(gf, {})
        ops.setdefault((kind == "value", op), []).append(k)
    blocks = {}
    for gf, ops in per_gf.items():
        terms = []
        for (is_value, op), ks in ops.items():
            if is_value:
                at = ("vjp_G[IDX4(%d, i0, i1, i2)]" if all_points else "VJP_G_AT(%d, 0, 0, 0)")
                terms.append(" + ".join(at % k for k in ks))
                continue
            if all_points:
                raise ValueError("an all-points VJP cannot contain stencils (slot %s)" % slots[ks[0]][0])
            coeffs, st = fin.compute_fdcoeffs_fdstencl(op)
            fac = invdx[int(op[-2])] * invdx[int(op[-1])] if op.startswith("dDD") else invdx[int(op[-1])]

            def at(s):
                g = ["VJP_G_AT(%d, %d, %d, %d)" % (k, -s[0], -s[1], -s[2]) for k in ks]
                return g[0] if len(g) == 1 else "(" + " + ".join(g) + ")"
            inner = " + ".join("%s*%s" % (_ccode(sp.Rational(c)), at(s)) for c, s in zip(coeffs, st))
            terms.append("%s*(%s)" % (_ccode(fac), inner))
        blocks[gf] = " +\n    ".join(terms)
    return blocks


def vjp_kernels(name, exprs, upwindcontrolvec, pointwise_loopopts, rfm_args, all_points=False, groups=None,
                split_transpose=False, order=None):
    """Generated source of ``<name>_vjp`` (pass 1 + pass 2 + an extern "C" driver).

    all_points: the forward operation is pointwise at every point (AllPoints loop, no
    stencils), so pass 2 reads the slot at the same point without the interior test.
    groups: lists of indices into exprs; pass 1 then runs as one kernel per group (each
    reverse sweep only over its own outputs, as the forward RHS is split to bound register
    pressure), in order on the stream: a group writes the slots it introduces and adds to
    those an earlier group introduced, so vjp_G holds each slot once.
    split_transpose: pass 2 as one kernel per cotangent gridfunction, so each lane sums the
    transposed stencils of one gridfunction instead of all of them.
    order: prefetch distance and region length of pass 1's statement order (schedule.reorder).
    Returns (source, slots, output arrays {gftype: [gf names]}, state_dependent)."""
    groups = groups or [list(range(len(exprs)))]
    slots, state_dependent, p1, uses_auxevol, p1_names = [], False, "", False, []
    bodies = []
    for k, idx in enumerate(groups):
        body1, sl, dep = vjp_pointwise_body([exprs[i] for i in idx], upwindcontrolvec, slot_offset=len(slots),
                                            existing={s[0]: j for j, s in enumerate(slots)})
        slots += sl
        state_dependent = state_dependent or dep
        uses_auxevol = uses_auxevol or "auxevol_gfs[" in body1
        bodies.append(schedule.reorder(body1, *order) if order else body1)
    for k, body1 in enumerate(bodies):
        kname = name + "_vjp_pointwise" + ("_g%d" % k if len(groups) > 1 else "")
        p1_names.append(kname)
        p1 += oc.outCfunction(
            outfile="returnstring", desc="VJP pass 1: pointwise adjoint of %s%s" % (
                name, (", output group %d" % k) if len(groups) > 1 else ""), name=kname,
            params=(rfm_args + "const paramstruct *restrict params,"
                    + ("const REAL *restrict auxevol_gfs," if uses_auxevol else "")
                    + "const REAL *restrict in_gfs,const REAL *restrict cot_rhs_gfs,REAL *restrict vjp_G"),
            body=body1, loopopts=pointwise_loopopts)
    blocks = vjp_transpose_bodies(slots, all_points)
    outputs = {"EVOL": [], "AUXEVOL": []}
    p2, p2_calls = "", []
    body2 = ""
    for gf in sorted(blocks):
        t = gri.find_gftype(gf)
        arr = "cot_in_gfs" if t == "EVOL" else "cot_auxevol_gfs"
        if t not in outputs:
            raise ValueError("VJP input %s has type %s" % (gf, t))
        outputs[t].append(gf)
        stmt = "%s[IDX4(%sGF, i0, i1, i2)] = %s;\n" % (arr, gf.upper(), blocks[gf])
        if split_transpose:
            kname = "%s_vjp_transpose_%s" % (name, gf)
            p2 += oc.outCfunction(
                outfile="returnstring", desc="VJP pass 2: transposed stencils of %s into the cotangent of %s"
                % (name, gf), name=kname,
                params=("const paramstruct *restrict params,const REAL *restrict vjp_G,REAL *restrict " + arr),
                body=stmt, loopopts="AllPoints")
            p2_calls.append("%s(params, vjp_G, %s, stream)" % (kname, arr))
        else:
            body2 += stmt
    has_aux_out = bool(outputs["AUXEVOL"])
    if not split_transpose:
        p2 = oc.outCfunction(
            outfile="returnstring", desc="VJP pass 2: transposed stencils of %s" % name, name=name + "_vjp_transpose",
            params=("const paramstruct *restrict params,const REAL *restrict vjp_G,REAL *restrict cot_in_gfs"
                    + (",REAL *restrict cot_auxevol_gfs" if has_aux_out else "")),
            body=body2, loopopts="AllPoints")
        p2_calls = ["%s_vjp_transpose(params, vjp_G, cot_in_gfs%s, stream)"
                    % (name, ", cot_auxevol_gfs" if has_aux_out else "")]
    rfm_call = "rfmstruct, " if rfm_args else ""
    aux_in = "auxevol_gfs, " if uses_auxevol else ""
    rfm_decl = "const rfm_struct *rfmstruct, " if rfm_args else ""
    calls = "".join("  if ((rc = %s(%sparams, %sin_gfs, cot_rhs_gfs, vjp_G, stream))) return rc;\n"
                    % (n, rfm_call, aux_in) for n in p1_names)
    calls += "".join("  if ((rc = %s)) return rc;\n" % c for c in p2_calls)
    driver = (
        "/* Vector-Jacobian product of %s: given cot_rhs_gfs (cotangent of the RHS at interior\n"
        " * points), writes the cotangent of every input gridfunction at every point into\n"
        " * cot_in_gfs (evolved) and cot_auxevol_gfs (auxiliary evolved; may be NULL when the\n"
        " * system has none). vjp_G is caller-allocated scratch of %d gridfunctions. Gridfunctions\n"
        " * of in_gfs that the RHS does not read get no write: clear cot_in_gfs first. */\n"
        'extern "C" int %s_vjp(%sconst paramstruct *params, const double *auxevol_gfs, const double *in_gfs,\n'
        "    const double *cot_rhs_gfs, double *vjp_G, double *cot_in_gfs, double *cot_auxevol_gfs,\n"
        "    hipStream_t stream) {\n"
        "  int rc;\n"
        "  (void)auxevol_gfs;\n  (void)cot_auxevol_gfs;\n%s"
        "  return NRPY_OK;\n"
        "}\n" % (name, len(slots), name, rfm_decl, calls))
    return p1 + p2 + driver, slots, outputs, state_dependent


def _linear_coefficients(exprs, slots):
    """{slot name: {output gridfunction: d(output)/d(slot)}} of a right-hand side that is linear in
    its slots with coefficients that are the same at every point; None if it is not one."""
    outs = [_out_name(e.lhs) for e in exprs]
    rhs = [sp.expand(sp.sympify(e.rhs)) for e in exprs]
    syms = {str(a): a for r in rhs for a in r.free_symbols}
    names = {s[0] for s in slots}
    coeffs = {}
    for name, kind, _, _ in slots:
        if kind not in ("value", "deriv"):
            return None
        coeffs[name] = {o: c for o, c in ((o, sp.diff(r, syms[name])) for o, r in zip(outs, rhs)) if c != 0}
        for c in coeffs[name].values():
            if any(str(a) in names or gri.variable_type(a) != "Cparameter" for a in c.free_symbols):
                return None
    return coeffs


# The ghost fill of an outer boundary: layers 1 and 2 from the three interior points next to it.
_EXTRAPOLATION = ((3, -3, 1), (6, -8, 3))


def _edge_terms(weights, d, at):
    """C statements that add to s, the transposed stencil of one operator along axis d at a point, what
    the ghost points hand back to it. Ghost layer g holds sum_p W(-g - p) cot(p) over the interior points
    p = 0, 1 next to the boundary, and point m = 0, 1, 2 gets E_g(m) times that, E the extrapolation
    above; the cotangents are among those the point's own stencil reads."""
    lines = []
    for side in (-1, 1):
        W = {1: weights.get(side, 0), 2: weights.get(2 * side, 0)}
        for m in range(3):
            k0 = _EXTRAPOLATION[0][m] * W[1] + _EXTRAPOLATION[1][m] * W[2]
            k1 = _EXTRAPOLATION[0][m] * W[2]
            edge = "NGHOSTS + %d" % m if side < 0 else "Nxx%d + NGHOSTS - %d" % (d, 1 + m)
            lines.append("if (i%d == %s) s += %s*%s + %s*%s;" % (
                d, edge, _ccode(k0), at(side * m), _ccode(k1), at(side * (m - 1))))
    return lines


def linear_stage_kernel(exprs, slots, evol):
    """Source of ``rhs_eval_vjp_rk4_stage``: one stage of the RK4 step adjoint of a right-hand side
    that is linear with coefficients that are the same at every point, on a grid whose ghost points
    are all extrapolated ones (None for any other right-hand side).

    Pass 1 of the vector-Jacobian product is then a multiplication by constants, so the transposed
    stencils read the cotangent itself and the constants join the stencil weights: no vjp_G. The
    transposed ghost fill is a change of the weights at the three points next to a boundary
    (_edge_terms), so no ghost cotangent is stored, and the sum w goes straight into the stage's
    updates, acc_out = acc_in + w and kbar_out = a L + b w. kbar_out is not the array the stencils
    read."""
    coeffs = _linear_coefficients(exprs, slots)
    if coeffs is None:
        return None
    invdx = [sp.Symbol("invdx%d" % d, real=True) for d in range(3)]
    reads, body, sums = {}, [], {}

    def cot(o, off):
        name = "cot_%s" % o + "".join("_i%d%s%d" % (d, "p" if v > 0 else "m", abs(v)) for d, v in enumerate(off) if v)
        reads[name] = "VJP_COT_AT(%sGF, %d, %d, %d)" % ((o.upper(),) + tuple(off))
        return name

    per_gf = {}
    for name, kind, gf, op in slots:
        for o, c in sorted(coeffs[name].items()):
            if kind == "value":
                term, fac = cot(o, (0, 0, 0)), c
            else:
                w, st = fin.compute_fdcoeffs_fdstencl(op)
                d = int(op[-1])
                weights = {s[d]: x for x, s in zip(w, st)}
                if any(s[e] for s in st for e in range(3) if e != d) or max(map(abs, weights)) > 2:
                    return None                      # _edge_terms: along one axis, two points at most
                fac = c * (invdx[d]**2 if op.startswith("dDD") else invdx[d])

                def at(v):
                    return cot(o, tuple(v if e == d else 0 for e in range(3)))
                if (o, op) not in sums:
                    sums[o, op] = "t_%s_%s" % (o, op)
                    body.append("double %s = %s;" % (sums[o, op], " + ".join(
                        "%s*%s" % (_ccode(sp.Rational(x)), at(-v)) for v, x in sorted(weights.items()))))
                    body += [l.replace(" s += ", " %s += " % sums[o, op]) for l in _edge_terms(weights, d, at)]
                term = sums[o, op]
            per_gf.setdefault(gf, []).append(term if fac == 1 else "%s*%s" % (_ccode(fac), term))
    if sorted(per_gf) != sorted(evol):
        return None
    body = ["const double %s = %s;" % kv for kv in reads.items()] + body
    body += ["const double w_%s = %s;" % (gf, " + ".join(per_gf[gf])) for gf in evol]
    # every read of acc_in and L before the first store: the compiler cannot tell the arrays apart
    body += ["const double acc_%s = acc_in[IDX4(%sGF, i0, i1, i2)], L_%s = S > 0 ? L[IDX4(%sGF, i0, i1, i2)] : 0.0;"
             % (gf, gf.upper(), gf, gf.upper()) for gf in evol]
    for gf in evol:
        body += ["{", "  const double w = S == 3 ? scale * w_%s : w_%s;" % (gf, gf),
                 "  acc_out[IDX4(%sGF, i0, i1, i2)] = acc_%s + w;" % (gf.upper(), gf),
                 "  if (S > 0) kbar_out[IDX4(%sGF, i0, i1, i2)] = a * L_%s + b * w;" % (gf.upper(), gf), "}"]
    body = "\n".join(body) + "\n"
    unpack = "".join("  const %s %s = params.%s;\n" % (lp._ctype(t), n, n) for n, t in lp._used_cparams(body)
                     if not n.startswith("Nxx"))
    unpack += "".join("  const int %s%d = params.%s%d;\n" % (n, d, n, d) for n in ("Nxx", "Nxx_plus_2NGHOSTS")
                      for d in range(3))
    args = ("const double *cot, const double *L, const double *acc_in, double *acc_out, double *%skbar_out, "
            "const double scale, const double a, const double b")
    return r"""
// A cotangent array, 0 outside the interior; the load stays in range as VJP_G_AT's does.
#define VJP_COT_AT(gf, o0, o1, o2)                                                                  \
  nrpy_vjp_select((i0) + (o0) >= NGHOSTS && (i0) + (o0) < Nxx0 + NGHOSTS && (i1) + (o1) >= NGHOSTS && \
                      (i1) + (o1) < Nxx1 + NGHOSTS && (i2) + (o2) >= NGHOSTS &&                     \
                      (i2) + (o2) < Nxx2 + NGHOSTS,                                                 \
                  cot[IDX4(gf, (i0) + (o0), (i1) + (o1), (i2) + (o2))])
// One stage of the RK4 step adjoint: w = (transposed ghost fill and stencils of rhs_eval) cot, times
// scale in stage 3 (whose kbar is scale L). Bound by its arrays: five read or written per gridfunction
// (three in stages 3 and 0) besides the stencil's neighbours, which the caches hold. Scalar wave at
// 128^3: 30 us a stage; slots, transposed stencils, ghost transpose, clearing and the update as
// launches of their own took 18 + 35 + 12 + 6 + 26 us. One point a lane and 64 x 4 tiles, as the
// forward substep: neighbours along x in the same cache lines.
template <int S>
__global__ void __launch_bounds__(256) rhs_eval_vjp_rk4_stage__gpu(const paramstruct params, """ + args % "__restrict__ " + r""") {
""" + unpack + _indent(r"""NRPY_BLOCK_COORDS(Nxx0, Nxx1, Nxx2);
const int i0 = NGHOSTS + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
const int i1 = NGHOSTS + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
const int i2 = NGHOSTS + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
if (i0 >= Nxx0 + NGHOSTS || i1 >= Nxx1 + NGHOSTS || i2 >= Nxx2 + NGHOSTS) return;
""" + body) + r"""}
static int rhs_eval_vjp_rk4_stage(const int S, const paramstruct *params, """ + args % "" + r""", hipStream_t stream) {
  const dim3 block(64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  switch (S) {
""" + "".join("    case %d: hipLaunchKernelGGL(rhs_eval_vjp_rk4_stage__gpu<%d>, grid, block, 0, stream, *params, cot, L, "
              "acc_in, acc_out, kbar_out, scale, a, b); break;\n" % (s, s) for s in range(4)) + r"""  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}
"""


def _indent(text):
    return "".join("  " + l + "\n" for l in text.splitlines())
