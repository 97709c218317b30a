"""Boundary-condition setup for the generated bundles.

``Set_up_CurviBoundaryConditions`` keeps the reference's entry point
(CurviBoundaryConditions/CurviBoundaryConditions.py:18-254). The map builder,
the sequential and composed ghost fills and their transpose are compiled into
every bundle from csrc/nrpy_runtime.h; this function writes the per-system
part (gridfunction #defines and parity types) and checks the choice of
boundary condition.

``sommerfeld_boundary_condition_class`` keeps the reference's class
(CurviBoundaryConditions.py:259-658): per-EVOL-gridfunction dictionaries of
value at infinity, radial falloff power and wave speed, keyed ``<NAME>GF``.
``hip_source()`` emits the radiation condition as HIP:

* a device function giving r and d f/d r = sum_i (d_i f)(d x^i / d r) at a
  point, with d_i f from one-sided stencils along directions in which the
  point lies on a boundary face or within NGHOSTS of the array edge and from
  centred stencils otherwise (fd_order 2, 4 or 6; the reference's stencils and
  coefficients), and d x^i / d r the first column of the inverse of the
  Jacobian d(r, theta, phi)/d(xx0, xx1, xx2), evaluated per point from the
  Jacobian's nine entries by cofactors (symbolic inversion of the sinh-mapped
  Jacobians swells beyond use);
* ``apply_bcs_sommerfeld``: for every outer ghost point, innermost layer
  first, rhs = -v [d f/d r + (f - f_inf)/r]; with falloff power n > 0 the
  difference between the evolved RHS and the pure-advection RHS one point
  inward (dest + FACE) is added, scaled by (r_inward/r)^n; then the inner
  (parity) ghost points copy the RHS of their source points. Points of one
  layer depend on points of the same layer reached through FACE (an i1-face
  point's inward neighbour may be an i0-face point of the layer), so each
  layer runs as three launches (i0-, i1-, i2-faces) followed by the parity
  copy, which reproduces the reference's sequential order.
"""
import os

import sympy as sp

from .. import NRPy_param_funcs as par
from .. import grid as gri
from .. import indexedexp as ixp
from .. import reference_metric as rfm

BOUNDARY_CONDITIONS = ("QuadraticExtrapolation", "Sommerfeld")


def Set_up_CurviBoundaryConditions(Ccodesdir, verbose=True, Cparamspath=os.path.join("../"),
                                   enable_copy_of_static_Ccodes=True, BoundaryCondition="QuadraticExtrapolation"):
    """Write ``gridfunction_defines.h`` (EVOL/AUX/AUXEVOL #defines and parity types, as
    the reference's gridfunction_defines.h) into ``Ccodesdir``. ``Cparamspath`` and
    ``enable_copy_of_static_Ccodes`` are accepted for compatibility: the static BC code is
    part of every compiled bundle."""
    if BoundaryCondition not in BOUNDARY_CONDITIONS:
        raise ValueError("BoundaryCondition must be one of %s, not %s" % (BOUNDARY_CONDITIONS, BoundaryCondition))
    from ..codegen import bundle as bd
    os.makedirs(Ccodesdir, exist_ok=True)
    defines, lists = bd.gf_defines_and_meta()
    out = "/* Generated by CurviBoundaryConditions.Set_up_CurviBoundaryConditions (%s). */\n" % BoundaryCondition
    out += defines + "\n"
    for kind in ("evol", "aux", "auxevol"):
        names = lists[kind]
        if names:
            out += "static const int8_t %s_gf_parity[%d] = {%s};\n" % (
                kind, len(names), ", ".join(str(bd.parity_type(n)) for n in names))
    with open(os.path.join(Ccodesdir, "gridfunction_defines.h"), "w") as f:
        f.write(out)
    if verbose:
        print("Evolved parity: ( " + ", ".join("%s:%d" % (n, bd.parity_type(n)) for n in lists["evol"]) + " )")
    return os.path.join(Ccodesdir, "gridfunction_defines.h")


class sommerfeld_boundary_condition_class():
    """Per-gridfunction Sommerfeld parameters and the HIP code that applies them."""

    def __init__(self, fd_order=2, vars_at_inf_default=0., vars_radial_falloff_power_default=3.,
                 vars_speed_default=1.):
        evolved, _, _ = gri.gridfunction_lists()
        if fd_order not in (2, 4, 6):
            raise ValueError("Sommerfeld fd_order must be 2, 4 or 6")
        NRPy_FD_order = par.parval_from_str("finite_difference::FD_CENTDERIVS_ORDER")
        if NRPy_FD_order < fd_order:
            raise ValueError("The global central finite differencing order within NRPy+ must be greater than or "
                             "equal to the Sommerfeld boundary condition's finite differencing order")
        self.fd_order = fd_order
        self.vars_at_infinity = {}
        self.vars_speed = {}
        self.vars_radial_falloff_power = {}
        for gf in evolved:
            self.vars_at_infinity[gf.upper() + "GF"] = vars_at_inf_default
            self.vars_radial_falloff_power[gf.upper() + "GF"] = vars_radial_falloff_power_default
            self.vars_speed[gf.upper() + "GF"] = vars_speed_default

    def sommerfeld_params(self):
        """The three per-gridfunction arrays, in EVOL gridfunction order, as device constants."""
        def arr(d):
            return "{" + ", ".join(repr(float(v)) for v in d.values()) + "}"
        return ("// Sommerfeld EVOL grid function parameters\n"
                "static __constant__ double evolgf_at_inf[NUM_EVOL_GFS] = %s;\n"
                "static __constant__ double evolgf_radial_falloff_power[NUM_EVOL_GFS] = %s;\n"
                "static __constant__ double evolgf_speed[NUM_EVOL_GFS] = %s;\n"
                % (arr(self.vars_at_infinity), arr(self.vars_radial_falloff_power), arr(self.vars_speed)))

    @staticmethod
    def jacobian():
        """r and the Jacobian J[i][j] = d xxSph^i / d xx^j of the current reference metric."""
        rfm.reference_metric()
        J = [[sp.diff(rfm.xxSph[i], rfm.xx[j]) for j in range(3)] for i in range(3)]
        return rfm.xxSph[0], J

    @staticmethod
    def contraction_from_jacobian(J, fdD):
        """sum_i fdD_i dx^i/dr, dx^i/dr = (J^-1)[i][0] = cofactor(0, i) / det J (the column of
        the inverse Jacobian that the generated code evaluates numerically at each point)."""
        c0 = J[1][1] * J[2][2] - J[1][2] * J[2][1]
        c1 = -(J[1][0] * J[2][2] - J[1][2] * J[2][0])
        c2 = J[1][0] * J[2][1] - J[1][1] * J[2][0]
        det = J[0][0] * c0 + J[0][1] * c1 + J[0][2] * c2
        return (fdD[0] * c0 + fdD[1] * c1 + fdD[2] * c2) / det

    @staticmethod
    def _simplified():
        """Whether the contraction is simplified symbolically: for every coordinate system
        without "Sinh" in its name, as the reference does (CurviBoundaryConditions.py:337-364;
        there simplification takes too long on the Sinh systems). The simplified form is also
        regular where the spherical Jacobian is singular, e.g. on the z axis of a Cartesian
        grid with an odd number of points along x and y: (fdD . x)/r instead of 0/0."""
        return "Sinh" not in par.parval_from_str("reference_metric::CoordSystem")

    @classmethod
    def radial_contraction(cls):
        """(r, sum_i fdD_i dx^i/dr) as SymPy expressions in the current reference metric:
        dx^i/dr = (J^-1)[i][0], each simplified and then their contraction simplified where
        _simplified() says so, else the cofactor ratio the generated code evaluates."""
        r, J = cls.jacobian()
        fdD = ixp.declarerank1("fdD")
        if not cls._simplified():
            return r, cls.contraction_from_jacobian(J, fdD)
        c = [J[1][1] * J[2][2] - J[1][2] * J[2][1], -(J[1][0] * J[2][2] - J[1][2] * J[2][0]),
             J[1][0] * J[2][1] - J[1][1] * J[2][0]]
        det = J[0][0] * c[0] + J[0][1] * c[1] + J[0][2] * c[2]
        dxdr = [sp.simplify(c[i] / det) for i in range(3)]
        return r, sp.simplify(sum(fdD[i] * dxdr[i] for i in range(3)))

    @staticmethod
    def _direction_code(d, fd_order):
        """C statements setting fdD<d> at (i0,i1,i2) from f (one gridfunction, 3D index).
        Both stencils are evaluated and the reference's test (one-sided on a boundary face or
        within NGHOSTS of the array's edge, else centred) selects one: under a branch each
        stencil's loads would be waited for in turn. Away from the faces S = 0, so the
        one-sided stencil reads the point itself; the centred stencil reads around an index
        held inside the array, which changes nothing where it is selected."""
        ix = ["i0", "i1", "i2"]
        R = fd_order // 2

        def at(shift, centre=False):
            idx = list(ix)
            base = "nrpy_ic%d" % d if centre else ix[d]
            idx[d] = "%s+%s" % (base, shift) if shift else base
            return "fa(%s,%s,%s)" % tuple(idx)
        one = {2: [("-1.5", 0), ("2.", 1), ("-0.5", 2)],
               4: [("u0", 0), ("u1", 1), ("u2", 2), ("u3", 3), ("u4", 4)],
               6: [("u0", 0), ("u1", 1), ("u2", 2), ("u3", 3), ("u4", 4), ("u5", 5), ("u6", 6)]}[fd_order]
        oneside = " + ".join("%s*%s" % (c, at("%d*S" % k if k else "")) for c, k in one)
        if fd_order == 2:
            cen = "(%s - %s)*0.5" % (at("1", True), at("-1", True))
        elif fd_order == 4:
            cen = "(-c2*%s + c1*%s - c1*%s + c2*%s)" % (at("2", True), at("1", True), at("-1", True), at("-2", True))
        else:
            cen = ("(c3*%s - c2*%s + c1*%s - c1*%s + c2*%s - c3*%s)"
                   % (at("3", True), at("2", True), at("1", True), at("-1", True), at("-2", True), at("-3", True)))
        return ("  {\n"
                "    const bool one_sided = abs(F%d) == 1 || %s + NGHOSTS >= Nxx_plus_2NGHOSTS%d || %s - NGHOSTS <= 0;\n"
                "    int S = F%d;\n"
                "    if (%s + NGHOSTS >= Nxx_plus_2NGHOSTS%d) S = -1;\n"
                "    if (%s - NGHOSTS <= 0) S = +1;\n"
                "    const int nrpy_ic%d = min(max(%s, %d), Nxx_plus_2NGHOSTS%d - 1 - %d);\n"
                "    const double one = S*(%s)*invdx%d;\n"
                "    const double cen = %s*invdx%d;\n"
                "    fdD%d = one_sided ? one : cen;\n"
                "  }\n" % (d, ix[d], d, ix[d], d, ix[d], d, ix[d], d, ix[d], R, d, R, oneside, d, cen, d, d))

    def dfdr_function(self, fd_order=None):
        """Device function nrpy_sommerfeld_r_dfdr (CurviBoundaryConditions.py:329-516)."""
        from .. import outputC as oc
        from ..codegen import bundle as bd
        fd_order = fd_order or self.fd_order
        if self._simplified():
            r, contraction = self.radial_contraction()
            body = oc.outputC([r, contraction], ["*r_out", "*dfdr_out"], "returnstring",
                              params="includebraces=False,outCverbose=False")
        else:
            r, J = self.jacobian()
            body = oc.outputC([r] + [J[i][j] for i in range(3) for j in range(3)],
                              ["*r_out"] + ["J%d%d" % (i, j) for i in range(3) for j in range(3)], "returnstring",
                              params="includebraces=False,outCverbose=False")
            body = "double J00, J01, J02, J10, J11, J12, J20, J21, J22;\n" + body
            body += ("const double cof0 = J11*J22 - J12*J21, cof1 = -(J10*J22 - J12*J20), cof2 = J10*J21 - J11*J20;\n"
                     "*dfdr_out = (fdD0*cof0 + fdD1*cof1 + fdD2*cof2)/(J00*cof0 + J01*cof1 + J02*cof2);\n")
        coef = self._stencil_constants(fd_order)
        dirs = "".join(self._direction_code(d, fd_order) for d in range(3))
        text = coef + dirs + "".join("  " + line + "\n" for line in body.splitlines())
        unpack = bd._unpack_for(text).replace("params->", "params.")
        for n in ("Nxx_plus_2NGHOSTS0", "Nxx_plus_2NGHOSTS1", "Nxx_plus_2NGHOSTS2", "invdx0", "invdx1", "invdx2"):
            if "const int %s =" % n not in unpack and "const double %s =" % n not in unpack:
                unpack += "  const %s %s = params.%s;\n" % ("int" if n.startswith("Nxx") else "double", n, n)
        return ("// r and d f/d r at (i0,i1,i2) of one gridfunction f, read as fa(i0,i1,i2); F = the point's\n"
                "// FACE (CurviBoundaryConditions.py:329-516).\n"
                "template <typename FA>\n"
                "static __device__ void nrpy_sommerfeld_r_dfdr(const paramstruct &params, const double *__restrict__ "
                "xx0_arr, const double *__restrict__ xx1_arr, const double *__restrict__ xx2_arr, "
                "FA fa, const int F0, const int F1, const int F2, const int i0, const int i1, "
                "const int i2, double *r_out, double *dfdr_out) {\n" + unpack +
                "  const double xx0 = xx0_arr[i0], xx1 = xx1_arr[i1], xx2 = xx2_arr[i2];\n"
                "  (void)xx0; (void)xx1; (void)xx2; (void)F0; (void)F1; (void)F2;\n"
                "  double fdD0 = 1e100, fdD1 = 1e100, fdD2 = 1e100;\n"
                "  (void)fdD0; (void)fdD1; (void)fdD2;\n" + text + "}\n")

    def geometry_functions(self):
        """dfdr_function in two parts, for the kernels that keep the geometry in a table:
        nrpy_sommerfeld_geometry gives r and what the derivative needs of the Jacobian at a point
        (the three cofactors and the determinant, or the simplified contraction's three
        coefficients over 1), nrpy_sommerfeld_dfdr_from contracts the stencils with them. The
        other kernels keep dfdr_function: in two parts it issues the stencils' loads after the
        geometry and divides once more per coefficient (eager steps 6 to 25% slower)."""
        from .. import outputC as oc
        from ..codegen import bundle as bd
        if self._simplified():
            r, contraction = self.radial_contraction()
            fdD = ixp.declarerank1("fdD")
            unit = [contraction.subs({fdD[j]: 1 if i == j else 0 for j in range(3)}) for i in range(3)]
            body = oc.outputC([r] + unit + [sp.Integer(1)], ["geo[%d]" % k for k in range(5)], "returnstring",
                              params="includebraces=False,outCverbose=False")
        else:
            r, J = self.jacobian()
            body = "double J00, J01, J02, J10, J11, J12, J20, J21, J22;\n" + oc.outputC(
                [r] + [J[i][j] for i in range(3) for j in range(3)],
                ["geo[0]"] + ["J%d%d" % (i, j) for i in range(3) for j in range(3)], "returnstring",
                params="includebraces=False,outCverbose=False")
            body += ("const double cof0 = J11*J22 - J12*J21, cof1 = -(J10*J22 - J12*J20), cof2 = J10*J21 - J11*J20;\n"
                     "geo[1] = cof0; geo[2] = cof1; geo[3] = cof2;\n"
                     "geo[4] = J00*cof0 + J01*cof1 + J02*cof2;\n")
        unpack = bd._unpack_for(body).replace("params->", "params.")
        dirs = "".join(self._direction_code(d, self.fd_order) for d in range(3))
        coef = self._stencil_constants(self.fd_order)
        dunpack = bd._unpack_for(coef + dirs).replace("params->", "params.")
        for n in ("Nxx_plus_2NGHOSTS0", "Nxx_plus_2NGHOSTS1", "Nxx_plus_2NGHOSTS2", "invdx0", "invdx1", "invdx2"):
            if "const int %s =" % n not in dunpack and "const double %s =" % n not in dunpack:
                dunpack += "  const %s %s = params.%s;\n" % ("int" if n.startswith("Nxx") else "double", n, n)
        return ("// r and the radial derivative's geometry at a point: geo = r, then a_i and b of\n"
                "// d f/d r = sum_i fdD_i a_i / b.\n"
                "static __device__ void nrpy_sommerfeld_geometry(const paramstruct &params, const double xx0, "
                "const double xx1, const double xx2, double *geo) {\n" + unpack +
                "  (void)xx0; (void)xx1; (void)xx2;\n" + "".join("  " + line + "\n" for line in body.splitlines()) + "}\n"
                "template <typename FA>\n"
                "static __device__ double nrpy_sommerfeld_dfdr_from(const paramstruct &params, const double *geo, FA fa, "
                "const int F0, const int F1, const int F2, const int i0, const int i1, const int i2) {\n" + dunpack +
                "  double fdD0 = 1e100, fdD1 = 1e100, fdD2 = 1e100;\n" + coef + dirs +
                "  const double cof0 = geo[1], cof1 = geo[2], cof2 = geo[3];\n"
                "  return (fdD0*cof0 + fdD1*cof1 + fdD2*cof2)/geo[4];\n}\n")

    @staticmethod
    def _stencil_constants(fd_order):
        if fd_order == 4:
            return ("  const double u0 = -25./12., u1 = 4., u2 = -3., u3 = 4./3., u4 = -1./4.;\n"
                    "  const double c1 = 2./3., c2 = 1./12.;\n")
        if fd_order == 6:
            return ("  const double u0 = -49./20., u1 = 6., u2 = -15./2., u3 = 20./3., u4 = -15./4., u5 = 6./5., "
                    "u6 = -1./6.;\n  const double c1 = 3./4., c2 = 3./20., c3 = 1./60;\n")
        return ""

    def hip_source(self, chain=False):
        """Parameters, r/dfdr device function, kernels and the apply_bcs_sommerfeld launcher; with
        ``chain`` also the one-launch form for grids with inner boundary points."""
        # the one-sided stencils reach fd_order points inward from a point within NGHOSTS of an edge
        minn = ("#define NRPY_SOMMERFELD_MIN_N (NGHOSTS + %d + 1)\n#define NRPY_SOMMERFELD_FD %d\n"
                % (self.fd_order, self.fd_order))
        return (self.sommerfeld_params() + minn + self.dfdr_function() + _SOMMERFELD_KERNELS +
                (self.geometry_functions() + _SOMMERFELD_CHAIN if chain else ""))

    def write_sommerfeld_main_Ccode(self, Ccodesdir):
        os.makedirs(os.path.join(Ccodesdir, "boundary_conditions"), exist_ok=True)
        path = os.path.join(Ccodesdir, "boundary_conditions", "apply_bcs_sommerfeld.h")
        with open(path, "w") as f:
            f.write(self.hip_source())
        return path

    def write_sommerfeld_file(self, Ccodesdir):
        path = self.write_sommerfeld_main_Ccode(Ccodesdir)
        print("\nSuccessfully generated Sommerfeld boundary condition C code")
        return path


_SOMMERFELD_KERNELS = r'''
// The radiation condition's right-hand side at outer point (i0,i1,i2) of gridfunction gf
// (apply_bcs_sommerfeld in CurviBoundaryConditions.py:538-620). fa(i,j,k): that gridfunction
// of the state the RHS is evaluated from; rn(o): the same gridfunction's RHS at the point's
// inward neighbour (i0,i1,i2) + FACE, flat index o.
// (r_offset / r)^n: the falloff powers in use are small integers (2 or 3), for which products
// replace the general FP64 pow, the largest part of a lane's arithmetic in the face kernels
// (within 2 ulp of the rounded power); any other power takes pow.
__device__ __forceinline__ double nrpy_som_falloff(const double q, const double n) {
  return n == 3.0 ? q * q * q : n == 2.0 ? q * q : n == 1.0 ? q : pow(q, n);
}
template <typename FA, typename RN>
__device__ __forceinline__ double nrpy_sommerfeld_rhs(const paramstruct &params, const double *__restrict__ xx0,
                                                      const double *__restrict__ xx1, const double *__restrict__ xx2,
                                                      const int gf, const int i0, const int i1, const int i2,
                                                      const int F0, const int F1, const int F2, FA fa, RN rn) {
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1;
  const double char_speed = evolgf_speed[gf];
  const double var_at_infinity = evolgf_at_inf[gf];
  const double radial_falloff_power = evolgf_radial_falloff_power[gf];
  double r = 1e100, partial_i_f = 1e100;
  nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, F1, F2, i0, i1, i2, &r, &partial_i_f);
  const double invr = 1. / r;
  const double source_rhs = -char_speed * (partial_i_f + invr * (fa(i0, i1, i2) - var_at_infinity));
  double out = source_rhs;
  if (radial_falloff_power > 0) {
    const int j0 = i0 + F0, j1 = i1 + F1, j2 = i2 + F2;
    double r_offset = 1e100, partial_i_f_offset = 1e100;
    nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, F1, F2, j0, j1, j2, &r_offset, &partial_i_f_offset);
    const double invr_offset = 1. / r_offset;
    const size_t o = (size_t)j0 + (size_t)N0 * ((size_t)j1 + (size_t)N1 * (size_t)j2);
    const double extrap_rhs = char_speed * (partial_i_f_offset + invr_offset * (fa(j0, j1, j2) - var_at_infinity));
    const double diff_between_advection_and_f_rhs = rn(o) + extrap_rhs;
    out = source_rhs + diff_between_advection_and_f_rhs * nrpy_som_falloff(r_offset * invr, radial_falloff_power);
  }
  return out;
}
// The same along an i0-face row, layer after layer (FACE (F0, 0, 0)): the inward neighbour of
// layer gz + 1's point is layer gz's point, with the same FACE, so its r and
// X = d f/d r + (f - f_inf)/r are the ones that point computed. have_in: r_in and X_in hold
// them (from the call for the layer before); else they are evaluated at (i0 + F0, i1, i2).
// On return r_in and X_in hold this point's. rn: the neighbour's RHS.
template <typename FA>
__device__ __forceinline__ double nrpy_sommerfeld_rhs_row(const paramstruct &params, const double *__restrict__ xx0,
                                                          const double *__restrict__ xx1,
                                                          const double *__restrict__ xx2, const int gf, const int i0,
                                                          const int i1, const int i2, const int F0, FA fa,
                                                          const double rn, const bool have_in, double &r_in,
                                                          double &X_in) {
  const double char_speed = evolgf_speed[gf];
  const double var_at_infinity = evolgf_at_inf[gf];
  const double radial_falloff_power = evolgf_radial_falloff_power[gf];
  double r = 1e100, partial_i_f = 1e100;
  nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, 0, 0, i0, i1, i2, &r, &partial_i_f);
  const double invr = 1. / r;
  const double X = partial_i_f + invr * (fa(i0, i1, i2) - var_at_infinity);
  const double source_rhs = -char_speed * X;
  double out = source_rhs;
  if (radial_falloff_power > 0) {
    double r_offset = r_in, X_offset = X_in;
    if (!have_in) {
      const int j0 = i0 + F0;
      double partial_i_f_offset = 1e100;
      r_offset = 1e100;
      nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, 0, 0, j0, i1, i2, &r_offset, &partial_i_f_offset);
      const double invr_offset = 1. / r_offset;
      X_offset = partial_i_f_offset + invr_offset * (fa(j0, i1, i2) - var_at_infinity);
    }
    const double extrap_rhs = char_speed * X_offset;
    const double diff_between_advection_and_f_rhs = rn + extrap_rhs;
    out = source_rhs + diff_between_advection_and_f_rhs * nrpy_som_falloff(r_offset * invr, radial_falloff_power);
  }
  r_in = r;
  X_in = X;
  return out;
}
// The same at outer point d, f read from global memory.
__device__ __forceinline__ double nrpy_sommerfeld_point(const paramstruct &params, const double *__restrict__ xx0,
                                                        const double *__restrict__ xx1,
                                                        const double *__restrict__ xx2, const int gf, const int d,
                                                        const int F0, const int F1, const int F2,
                                                        const double *__restrict__ f, const double *rhs) {
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1;
  const int i0 = d % N0, i1 = (d / N0) % N1, i2 = d / (N0 * N1);
  return nrpy_sommerfeld_rhs(params, xx0, xx1, xx2, gf, i0, i1, i2, F0, F1, F2,
                             [f, N0, N1](const int a, const int b, const int c) { return f[a + N0 * (b + N1 * c)]; },
                             [rhs](const size_t o) { return rhs[o]; });
}

// The i0-faces on grids whose ghost points are all outer points: there the group of layer
// gz is every (i0, i1, i2) with i0 = NGHOSTS - 1 - gz (FACE +1) or N0 - NGHOSTS + gz (FACE -1)
// and (i1, i2) in the box the earlier layers grew, [NGHOSTS - gz, N - NGHOSTS + gz). In a row
// whose (i1, i2) is interior, each of these points needs only the RHS of its inward
// neighbour in the same row (the interior point, or the layer before), and no other face
// group feeds it, while those that read it come later in the reference's order: so one
// launch before the layers takes every layer of the interior rows, each lane its row's
// points layer after layer (the edge rows stay in their layers' i0 slots).
// On an i0-face consecutive points lie in different rows, so a load of one value per lane
// touches as many cache lines as lanes. A block of 256 lanes takes a 32 x 8 tile of interior
// rows (i1, i2) and first copies what the stencils reach into LDS, rows of NRPY_SOM_XW
// points, x fastest: along i0 the one-sided and centred stencils of the points and of their
// inward neighbours stay in [0, NGHOSTS + FD] (mirrored on the high side); along i1 and i2
// a row's centred stencil stays within FD / 2 of it, and the one-sided one (the row next
// to the ghost zone, i = NGHOSTS) reaches FD points inward, inside the tile's own rows or
// its upper halo (the box ends at the grid's edge).
#define NRPY_SOM_TY 32
#define NRPY_SOM_TZ 8
#define NRPY_SOM_HALO (NRPY_SOMMERFELD_FD / 2)
#define NRPY_SOM_XW (NGHOSTS + NRPY_SOMMERFELD_FD + 1)
#define NRPY_SOM_BOXN (NRPY_SOM_XW * (NRPY_SOM_TY + 2 * NRPY_SOM_HALO) * (NRPY_SOM_TZ + 2 * NRPY_SOM_HALO))
static_assert(NRPY_SOM_HALO <= NGHOSTS, "the x-face box starts inside the grid");
struct nrpy_som_xtile {
  int F0, y0, z0, hi1, hi2, bx0, by0, by1, bz0, bz1;
};
__host__ __device__ static inline int nrpy_som_xface_ntiles(const int N1, const int N2) {
  const int n1 = N1 - 2 * NGHOSTS, n2 = N2 - 2 * NGHOSTS;
  return 2 * ((n1 + NRPY_SOM_TY - 1) / NRPY_SOM_TY) * ((n2 + NRPY_SOM_TZ - 1) / NRPY_SOM_TZ);
}
// tile t of nrpy_som_xface_ntiles(N1, N2): its rows [y0, min(y0 + TY, hi1)) x [z0, min(z0 +
// TZ, hi2)), its side (F0 +1: the low i0-faces) and the box [bx0, bx0 + XW) x [by0, by1) x
// [bz0, bz1) copied to LDS
__host__ __device__ static inline nrpy_som_xtile nrpy_som_xface_tile(const int N0, const int N1, const int N2,
                                                                     int t) {
  nrpy_som_xtile T;
  T.hi1 = N1 - NGHOSTS;
  T.hi2 = N2 - NGHOSTS;
  const int nty = (T.hi1 - NGHOSTS + NRPY_SOM_TY - 1) / NRPY_SOM_TY;
  const int side = t % 2;
  t /= 2;
  T.y0 = NGHOSTS + (t % nty) * NRPY_SOM_TY;
  T.z0 = NGHOSTS + (t / nty) * NRPY_SOM_TZ;
  T.F0 = side == 0 ? 1 : -1;
  T.bx0 = side == 0 ? 0 : N0 - NRPY_SOM_XW;
  T.by0 = T.y0 - NRPY_SOM_HALO;
  T.by1 = T.y0 + NRPY_SOM_TY + NRPY_SOM_HALO < N1 ? T.y0 + NRPY_SOM_TY + NRPY_SOM_HALO : N1;
  T.bz0 = T.z0 - NRPY_SOM_HALO;
  T.bz1 = T.z0 + NRPY_SOM_TZ + NRPY_SOM_HALO < N2 ? T.z0 + NRPY_SOM_TZ + NRPY_SOM_HALO : N2;
  return T;
}
// Block (tile blockIdx.x of the interior rows, i.e. of layer 0's group; gridfunction
// blockIdx.y) of 256 lanes: copies the box, then lane l takes row (y0 + l % 32, z0 + l / 32)
// if it is interior and computes its i0-face points from the innermost layer out, the
// inward neighbour's RHS the interior point's (read from rhs), then the one this lane
// computed last. FUSED: the RK4 update of substep S as nrpy_sommerfeld_outer_rk4_kernel does,
// with R as the RHS array; else the RHS goes to rhs. Every global load is issued before the
// box copy, so a lane waits for memory once.
template <int FUSED, int S>
__global__ void __launch_bounds__(NRPY_SOM_TY * NRPY_SOM_TZ) nrpy_sommerfeld_xface_kernel(const paramstruct params,
                                                                   const double *__restrict__ xx0,
                                                                   const double *__restrict__ xx1,
                                                                   const double *__restrict__ xx2,
                                                                   const double *__restrict__ gfs, double *rhs_gfs,
                                                                   double *y_n, double *rt, double *out,
                                                                   const double dt) {
  __shared__ double box[NRPY_SOM_BOXN];
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1, N2 = params.Nxx_plus_2NGHOSTS2;
  const size_t Ntot = (size_t)N0 * N1 * N2;
  const nrpy_som_xtile T = nrpy_som_xface_tile(N0, N1, N2, (int)blockIdx.x);
  const int gf = (int)blockIdx.y;
  const double *f = gfs + (size_t)gf * Ntot;
  const int BY = T.by1 - T.by0, BZ = T.bz1 - T.bz0, nbox = NRPY_SOM_XW * BY * BZ;
  const int i1 = T.y0 + (int)threadIdx.x % NRPY_SOM_TY, i2 = T.z0 + (int)threadIdx.x / NRPY_SOM_TY;
  const bool live = i1 < T.hi1 && i2 < T.hi2;
  // a lane past the grid's edge loads at the tile's first row (inside the grid) and stores nothing
  const size_t row = (size_t)N0 * ((size_t)(live ? i1 : T.y0) + (size_t)N1 * (size_t)(live ? i2 : T.z0));
  double *rhs = rhs_gfs + (size_t)gf * Ntot;
  size_t dl[NGHOSTS];
  double yv[NGHOSTS], rv[NGHOSTS];
#pragma unroll
  for (int gz = 0; gz < NGHOSTS; gz++) {
    dl[gz] = row + (size_t)(T.F0 > 0 ? NGHOSTS - 1 - gz : N0 - NGHOSTS + gz);
    yv[gz] = FUSED && S < 3 ? y_n[(size_t)gf * Ntot + dl[gz]] : 0.0;
    rv[gz] = FUSED && S > 0 ? (S < 3 ? rt[(size_t)gf * Ntot + dl[gz]]
                                     : y_n[(size_t)gf * Ntot + dl[gz]] + rt[(size_t)gf * Ntot + dl[gz]])
                            : 0.0;
  }
  // the interior RHS next to the face: FUSED, from the compact array the shell kernel fills after
  // the NUM_EVOL_GFS grids of R ([gf][i2][i1][side]); else from the RHS grid
  const size_t xrow = (size_t)(live ? i1 : T.y0) + (size_t)N1 * (size_t)(live ? i2 : T.z0);
  double prev = FUSED ? rhs_gfs[(size_t)NUM_EVOL_GFS * Ntot + 2 * ((size_t)gf * N1 * N2 + xrow) + (T.F0 > 0 ? 0 : 1)]
                      : rhs[row + (size_t)(T.F0 > 0 ? NGHOSTS : N0 - 1 - NGHOSTS)];
  for (int e = (int)threadIdx.x; e < nbox; e += (int)blockDim.x) {
    const int x = e % NRPY_SOM_XW, y = (e / NRPY_SOM_XW) % BY, z = e / (NRPY_SOM_XW * BY);
    box[e] = f[(T.bx0 + x) + N0 * ((T.by0 + y) + N1 * (T.bz0 + z))];
  }
  __syncthreads();
  if (!live) return;
  const auto fa = [&](const int a, const int b, const int c) {
    return box[(a - T.bx0) + NRPY_SOM_XW * ((b - T.by0) + BY * (c - T.bz0))];
  };
  // r and d f/d r + (f - f_inf)/r of the point this lane computed last (its next inward neighbour)
  double r_in = 0.0, X_in = 0.0;
#pragma unroll
  for (int gz = 0; gz < NGHOSTS; gz++) {
    const int i0 = T.F0 > 0 ? NGHOSTS - 1 - gz : N0 - NGHOSTS + gz;
    const double ki = nrpy_sommerfeld_rhs_row(params, xx0, xx1, xx2, gf, i0, i1, i2, T.F0, fa, prev, gz > 0, r_in, X_in);
    prev = ki;
    rhs[dl[gz]] = ki;
    if (FUSED) {
      const size_t i = (size_t)gf * Ntot + dl[gz];
      if (S == 0) {
        rt[i] = ki * dt * (1.0 / 6.0);
        out[i] = yv[gz] + ki * dt * (1.0 / 2.0);
      } else if (S == 1) {
        rt[i] = rv[gz] + ki * dt * (1.0 / 3.0);
        out[i] = yv[gz] + ki * dt * (1.0 / 2.0);
      } else if (S == 2) {
        rt[i] = rv[gz] + ki * dt * (1.0 / 3.0);
        out[i] = yv[gz] + ki * dt;
      } else {
        out[i] = rv[gz] + ki * dt * (1.0 / 6.0);
      }
    }
  }
}
static void nrpy_sommerfeld_xface_launch(const int fused, const int S, const paramstruct *params, double *xx[3],
                                         const int num_gfs, double *gfs, double *rhs, double *y_n, double *rt,
                                         double *out, const double dt, hipStream_t stream) {
  const dim3 grid((unsigned)nrpy_som_xface_ntiles(params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2),
                  (unsigned)num_gfs);
  const dim3 block(NRPY_SOM_TY * NRPY_SOM_TZ);
  if (!fused)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<0, 0>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else if (S == 0)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 0>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else if (S == 1)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 1>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else if (S == 2)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 2>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 3>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
}

// One face group of one ghost layer: lane p of block row blockIdx.y handles outer point p of
// gridfunction blockIdx.y (no integer division per lane).
__global__ void nrpy_sommerfeld_outer_kernel(const paramstruct params, const double *__restrict__ xx0,
                                             const double *__restrict__ xx1, const double *__restrict__ xx2, int n,
                                             const int *__restrict__ dest, const int8_t *__restrict__ face, int num_gfs,
                                             const double *__restrict__ gfs, double *__restrict__ rhs_gfs) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), gf = (int)blockIdx.y;
  if (p >= n || gf >= num_gfs) return;
  const size_t Ntot = (size_t)params.Nxx_plus_2NGHOSTS0 * params.Nxx_plus_2NGHOSTS1 * params.Nxx_plus_2NGHOSTS2;
  const int d = dest[p];
  double *rhs = rhs_gfs + (size_t)gf * Ntot;
  rhs[d] = nrpy_sommerfeld_point(params, xx0, xx1, xx2, gf, d, face[3 * p], face[3 * p + 1], face[3 * p + 2],
                                 gfs + (size_t)gf * Ntot, rhs);
}

// The same, fused with the RK4 update at the outer point (the arithmetic of
// nrpy_rk4_update_all): the RHS at outer points goes to the scratch array R (where the
// interior kernel left it at the points next to the boundary), and the stage value of
// substep S to out (and the running total to rt).
template <int S>
__global__ void nrpy_sommerfeld_outer_rk4_kernel(const paramstruct params, const double *__restrict__ xx0,
                                                 const double *__restrict__ xx1, const double *__restrict__ xx2,
                                                 int n, const int *__restrict__ dest, const int8_t *__restrict__ face,
                                                 int num_gfs, const double *__restrict__ gfs, double *__restrict__ R,
                                                 double *y_n, double *rt, double *out, const double dt) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), gf = (int)blockIdx.y;
  if (p >= n || gf >= num_gfs) return;
  const size_t Ntot = (size_t)params.Nxx_plus_2NGHOSTS0 * params.Nxx_plus_2NGHOSTS1 * params.Nxx_plus_2NGHOSTS2;
  const int d = dest[p];
  double *rhs = R + (size_t)gf * Ntot;
  const size_t i = (size_t)gf * Ntot + d;
  // the update's operands are loaded before the condition's arithmetic, not after its store
  const double yv = S < 3 ? y_n[i] : 0.0;
  const double rv = S == 0 ? 0.0 : S < 3 ? rt[i] : y_n[i] + rt[i];
  const double ki = nrpy_sommerfeld_point(params, xx0, xx1, xx2, gf, d, face[3 * p], face[3 * p + 1],
                                          face[3 * p + 2], gfs + (size_t)gf * Ntot, rhs);
  rhs[d] = ki;
  if (S == 0) {
    rt[i] = ki * dt * (1.0 / 6.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 1) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 2) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt;
  } else {
    out[i] = rv + ki * dt * (1.0 / 6.0);
  }
}

// Substep S of the fused Sommerfeld RK4 step at the outer points, layer by layer and face
// group by face group in the reference's order. gfs: the substep's input state; R: the
// RHS scratch, holding the interior RHS at the points next to the boundary. For grids
// without inner boundary points only (NRPY_ERR_PARAM otherwise).
extern "C" int apply_bcs_sommerfeld_rk4(const int S, const paramstruct *params, double *xx[3], const bc_struct *bc,
                                        const int NUM_GFS, double *gfs, double *R, double *y_n, double *rt,
                                        double *out, const double dt, hipStream_t stream) {
  if (!params || !bc || !xx || !xx[0] || !xx[1] || !xx[2] || !gfs || !R || !y_n || !rt || !out)
    return NRPY_ERR_NULL;
  if (S < 0 || S > 3 || NUM_GFS < 1 || NUM_GFS > NUM_EVOL_GFS) return NRPY_ERR_PARAM;
  if (bc->N[0] != params->Nxx_plus_2NGHOSTS0 || bc->N[1] != params->Nxx_plus_2NGHOSTS1 ||
      bc->N[2] != params->Nxx_plus_2NGHOSTS2)
    return NRPY_ERR_SHAPE;
  if (bc->N[0] < NRPY_SOMMERFELD_MIN_N || bc->N[1] < NRPY_SOMMERFELD_MIN_N || bc->N[2] < NRPY_SOMMERFELD_MIN_N)
    return NRPY_ERR_SHAPE;
  for (int gz = 0; gz < NGHOSTS; gz++)
    if (bc->num_ib_gz_pts[gz] > 0) return NRPY_ERR_PARAM;
  const int B = 256;
  nrpy_sommerfeld_xface_launch(1, S, params, xx, NUM_GFS, gfs, R, y_n, rt, out, dt, stream);
  for (int gz = 0; gz < NGHOSTS; gz++) {
    int start = 0;
    for (int dir = 0; dir < 3; dir++) {
      const int end = bc->ob_dir_end[gz][dir];
      // the i0-face group: its edge rows only (the interior rows were launched above)
      const int n = dir == 0 ? bc->ob_xedge_off[gz + 1] - bc->ob_xedge_off[gz] : end - start;
      if (n > 0) {
        const dim3 grid((unsigned)((n + B - 1) / B), (unsigned)NUM_GFS);
        const int *dst = dir == 0 ? bc->d_ob_xedge_dest + bc->ob_xedge_off[gz] : bc->d_ob_dest + bc->ob_off[gz] + start;
        const int8_t *fc = dir == 0 ? bc->d_ob_xedge_face + 3 * (size_t)bc->ob_xedge_off[gz]
                                    : bc->d_ob_face + 3 * (size_t)(bc->ob_off[gz] + start);
        switch (S) {
          case 0: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<0>, grid, dim3(B), 0, stream, *params, xx[0],
                                     xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
          case 1: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<1>, grid, dim3(B), 0, stream, *params, xx[0],
                                     xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
          case 2: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<2>, grid, dim3(B), 0, stream, *params, xx[0],
                                     xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
          default: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<3>, grid, dim3(B), 0, stream, *params, xx[0],
                                      xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
        }
      }
      start = end;
    }
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}

// Sommerfeld radiation condition on the RHS at every ghost point: outer points
// from the radiation condition, inner points by parity from their sources.
// xx: the three device coordinate arrays; gfs_parity: host array of NUM_GFS
// parity types; gfs: the state the RHS was evaluated from; rhs_gfs: its RHS,
// valid at interior points. NUM_GFS <= NUM_EVOL_GFS (per-gridfunction
// parameters are those of the EVOL gridfunctions).
extern "C" int apply_bcs_sommerfeld(const paramstruct *params, double *xx[3], const bc_struct *bc, const int NUM_GFS,
                                    const int8_t *gfs_parity, double *gfs, double *rhs_gfs, hipStream_t stream) {
  if (!xx || !xx[0] || !xx[1] || !xx[2] || !rhs_gfs) return NRPY_ERR_NULL;
  if (NUM_GFS > NUM_EVOL_GFS) return NRPY_ERR_PARAM;
  nrpy_gf_parity_args gfp;
  memset(&gfp, 0, sizeof(gfp));
  int rc = nrpy_bc_check(params, bc, NUM_GFS, gfs_parity, gfs, &gfp);
  if (rc) return rc;
  if (bc->N[0] < NRPY_SOMMERFELD_MIN_N || bc->N[1] < NRPY_SOMMERFELD_MIN_N || bc->N[2] < NRPY_SOMMERFELD_MIN_N)
    return NRPY_ERR_SHAPE;
  const size_t Ntot = (size_t)bc->N[0] * bc->N[1] * bc->N[2];
  const int B = 256;
  bool all_outer = true;   // every ghost point an outer point: the interior rows' i0-faces take the tiled kernel
  for (int gz = 0; gz < NGHOSTS; gz++) all_outer = all_outer && bc->num_ib_gz_pts[gz] == 0;
  if (all_outer)
    nrpy_sommerfeld_xface_launch(0, 0, params, xx, NUM_GFS, gfs, rhs_gfs, nullptr, nullptr, nullptr, 0.0, stream);
  for (int gz = 0; gz < NGHOSTS; gz++) {
    int start = 0;
    for (int dir = 0; dir < 3; dir++) {
      const int end = bc->ob_dir_end[gz][dir];
      const bool edge = dir == 0 && all_outer;   // the i0-face group's edge rows only
      const int n = edge ? bc->ob_xedge_off[gz + 1] - bc->ob_xedge_off[gz] : end - start;
      if (n > 0) {
        hipLaunchKernelGGL(nrpy_sommerfeld_outer_kernel, dim3((unsigned)((n + B - 1) / B), (unsigned)NUM_GFS), dim3(B),
                           0, stream,
                           *params, xx[0], xx[1], xx[2], n,
                           edge ? bc->d_ob_xedge_dest + bc->ob_xedge_off[gz] : bc->d_ob_dest + bc->ob_off[gz] + start,
                           edge ? bc->d_ob_xedge_face + 3 * (size_t)bc->ob_xedge_off[gz]
                                : bc->d_ob_face + 3 * (size_t)(bc->ob_off[gz] + start),
                           NUM_GFS, gfs, rhs_gfs);
      }
      start = end;
    }
    const int ni = bc->num_ib_gz_pts[gz];
    if (ni > 0) {
      const size_t work = (size_t)ni * NUM_GFS;
      hipLaunchKernelGGL(nrpy_bc_inner_kernel, dim3((unsigned)((work + B - 1) / B)), dim3(B), 0, stream, ni,
                         bc->d_ib_dest + bc->ib_off[gz], bc->d_ib_src + bc->ib_off[gz],
                         bc->d_ib_parity + 10 * (size_t)bc->ib_off[gz], NUM_GFS, gfp, Ntot, rhs_gfs);
    }
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}
'''

_SOMMERFELD_CHAIN = r'''
// The whole condition in two launches per substep, for grids with inner boundary points. The
// reference's order (layer by layer, face group by face group, then the parity copies) makes a
// chain of each outer point: its RHS is
//   rhs_p = A_p + (rhs_q + B_p) (r_q / r_p)^n,   q its inward neighbour (an interior point, or an
// outer point one step further in), A_p = -v X_p, B_p = v X_q, X = d f/d r + (f - f_inf)/r with
// the stencils of p's FACE. A and B need only the state the substep starts from, so they are
// evaluated for every outer point at once, in extra blocks of the interior RHS launch
// (nrpy_sommerfeld_eval); the second launch (nrpy_sommerfeld_chain_kernel) walks each ghost
// point's chain from the interior out, at most 3 NGHOSTS multiply-adds, an inner point that of
// the point it copies, and does the RK4 update there. Every point's FACE follows from its
// indices: the axis with the largest distance outside the interior, the last of equals
// (nrpy_sommerfeld_chainable: known from building the lists). The operations are those of
// nrpy_sommerfeld_rhs; the results agree to rounding.
// Both launches are bound by latency. On the Maxwell 50x4x100 grid (MI355X) the condition's 9
// launches of 4-7 us with gaps of 2.4 us took 70 us a substep; one launch that evaluated the
// chains point after point 48 us, 25 us with r, the cofactors and the determinant from a table
// (geo, 5 values per point) instead of the Jacobian. MoL_graph_launch fills the table before its
// replays, on their stream, so that the coordinates are read when and where the step reads its
// other arrays (one launch of about 5 us per call, not per step).
// Scratch of a captured step: R, NUM_EVOL_GFS gridfunctions: the RHS at the interior points a
// chain or copy ends at (rhs_eval_rk4_substep_rim), A at the outer points; then B, as many; then geo.
#define NRPY_SOM_NSCRATCH (2 * NUM_EVOL_GFS + 5)

// Step k of n (k = 0 the innermost) of the chain with layers l: its axis.
__device__ __forceinline__ int nrpy_som_chain_axis(const int l0, const int l1, const int l2, const int k) {
  int m0 = l0, m1 = l1, m2 = l2, a = 0;
  for (int j = l0 + l1 + l2 - 1; j >= k; j--) {
    const int far = max(m0, max(m1, m2));
    a = m2 == far ? 2 : m1 == far ? 1 : 0;
    m0 -= a == 0;
    m1 -= a == 1;
    m2 -= a == 2;
  }
  return a;
}

// A and B at outer point number t % n of the lists (all layers) of gridfunction t / n.
__device__ __forceinline__ void nrpy_sommerfeld_eval(const paramstruct &params, const size_t t, const int n,
                                                     const int *__restrict__ dest, const int8_t *__restrict__ face,
                                                     const double *__restrict__ gfs, double *__restrict__ R) {
  if (t >= (size_t)n * NUM_EVOL_GFS) return;
  const int gf = (int)(t / n), p = (int)(t % n);
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1;
  const size_t Ntot = (size_t)N0 * N1 * params.Nxx_plus_2NGHOSTS2;
  const double *__restrict__ geo = R + (size_t)(2 * NUM_EVOL_GFS) * Ntot;
  const double *__restrict__ f = gfs + (size_t)gf * Ntot;
  const int d = dest[p], F0 = face[3 * p], F1 = face[3 * p + 1], F2 = face[3 * p + 2];
  const int i0 = d % N0, i1 = (d / N0) % N1, i2 = d / (N0 * N1);
  const auto fa = [f, N0, N1](const int a, const int b, const int c) { return f[a + N0 * (b + N1 * c)]; };
  const double char_speed = evolgf_speed[gf], var_at_infinity = evolgf_at_inf[gf];
  double X[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int j0 = i0 + q * F0, j1 = i1 + q * F1, j2 = i2 + q * F2;
    const size_t at = (size_t)j0 + N0 * ((size_t)j1 + N1 * (size_t)j2);
    const double g[5] = {geo[at], geo[Ntot + at], geo[2 * Ntot + at], geo[3 * Ntot + at], geo[4 * Ntot + at]};
    const double invr = 1. / g[0];
    X[q] = nrpy_sommerfeld_dfdr_from(params, g, fa, F0, F1, F2, j0, j1, j2) + invr * (fa(j0, j1, j2) - var_at_infinity);
  }
  R[(size_t)gf * Ntot + d] = -char_speed * X[0];
  R[(size_t)(NUM_EVOL_GFS + gf) * Ntot + d] = char_speed * X[1];
}

// The chain of at most MAX steps: every operand is loaded before the first multiply-add.
template <int MAX>
__device__ __forceinline__ double nrpy_som_walk(const nrpy_fill_row row, const int *l, const int *F, const int n,
                                                const int N0, const int N1, const size_t Ntot, const int gf,
                                                const double *__restrict__ R) {
  const double *__restrict__ A = R + (size_t)gf * Ntot;
  const double *__restrict__ B = A + (size_t)NUM_EVOL_GFS * Ntot;
  const double *__restrict__ r = R + (size_t)(2 * NUM_EVOL_GFS) * Ntot;
  const double power = evolgf_radial_falloff_power[gf];
  double a[MAX], b[MAX], rp[MAX + 1];
  double ki = A[row.base];
  rp[0] = r[row.base];
  int at = row.base;
#pragma unroll
  for (int k = 0; k < MAX; k++) {
    if (k < n) {
      const int ax = nrpy_som_chain_axis(l[0], l[1], l[2], k);
      at -= ax == 0 ? F[0] : ax == 1 ? F[1] * N0 : F[2] * N0 * N1;
    }
    a[k] = A[at];
    b[k] = B[at];
    rp[k + 1] = r[at];
  }
#pragma unroll
  for (int k = 0; k < MAX; k++) {
    const double invr = 1. / rp[k + 1];
    const double next = power > 0 ? a[k] + (ki + b[k]) * nrpy_som_falloff(rp[k] * invr, power) : a[k];
    ki = k < n ? next : ki;
  }
  return ki;
}

template <int S>
__global__ void __launch_bounds__(256)
nrpy_sommerfeld_chain_kernel(const paramstruct params, const int nrows, const nrpy_fill_row *__restrict__ rows,
                             const nrpy_gf_parity_args gfp, const double *__restrict__ R, double *y_n, double *rt,
                             double *out, const double dt) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), gf = (int)blockIdx.y;
  if (p >= nrows) return;
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1, N2 = params.Nxx_plus_2NGHOSTS2;
  const size_t Ntot = (size_t)N0 * N1 * N2;
  const nrpy_fill_row row = rows[p];
  const size_t i = (size_t)gf * Ntot + row.dest;
  const double yv = S < 3 ? y_n[i] : 0.0;
  const double rv = S == 0 ? 0.0 : S < 3 ? rt[i] : y_n[i] + rt[i];
  int l[3], F[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int c = (row.code >> (3 * d)) & 7;
    l[d] = c > 3 ? c - 3 : c;
    F[d] = c > 3 ? -1 : 1;
  }
  const int n = l[0] + l[1] + l[2];
  double ki;
  if (n == 0)
    ki = R[(size_t)gf * Ntot + row.base];
  else if (n <= NGHOSTS)
    ki = nrpy_som_walk<NGHOSTS>(row, l, F, n, N0, N1, Ntot, gf, R);
  else
    ki = nrpy_som_walk<3 * NGHOSTS>(row, l, F, n, N0, N1, Ntot, gf, R);
  if (row.negmask & (1 << gfp.p[gf])) ki = -ki;
  if (S == 0) {
    rt[i] = ki * dt * (1.0 / 6.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 1) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 2) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt;
  } else {
    out[i] = rv + ki * dt * (1.0 / 6.0);
  }
}

// The geometry table, at the ghost points and the interior points next to them.
__global__ void __launch_bounds__(256)
nrpy_sommerfeld_geometry_kernel(const paramstruct params, const double *__restrict__ xx0,
                                const double *__restrict__ xx1, const double *__restrict__ xx2,
                                double *__restrict__ geo) {
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1, N2 = params.Nxx_plus_2NGHOSTS2;
  const size_t Ntot = (size_t)N0 * N1 * N2, at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= Ntot) return;
  const int i0 = (int)(at % N0), i1 = (int)((at / N0) % N1), i2 = (int)(at / ((size_t)N0 * N1));
  if (i0 > NGHOSTS && i0 < N0 - 1 - NGHOSTS && i1 > NGHOSTS && i1 < N1 - 1 - NGHOSTS && i2 > NGHOSTS &&
      i2 < N2 - 1 - NGHOSTS)
    return;
  double g[5];
  nrpy_sommerfeld_geometry(params, xx0[i0], xx1[i1], xx2[i2], g);
#pragma unroll
  for (int k = 0; k < 5; k++) geo[k * Ntot + at] = g[k];
}

// Whether the two launches cover the grid's ghost points: each is an outer point or a copy of
// an outer or interior point (no generic row), each outer point's FACE is the one its indices
// give, and every interior point a chain or copy ends at lies within NGHOSTS of an edge. All of it
// is known from building the maps: going over the rows here took 2 ms of each graph creation
// at 200x16x400.
static bool nrpy_sommerfeld_chainable(const bc_struct *bc) {
  return bc->fill_all.n > 0 && bc->fill_all.near_edges && bc->face_by_distance;
}

// The geometry table in the scratch of a captured step.
static int nrpy_sommerfeld_geometry_fill(const paramstruct *params, const double *const xx[3], double *scratch,
                                         hipStream_t stream) {
  const size_t Ntot =
      (size_t)params->Nxx_plus_2NGHOSTS0 * params->Nxx_plus_2NGHOSTS1 * params->Nxx_plus_2NGHOSTS2;
  hipLaunchKernelGGL(nrpy_sommerfeld_geometry_kernel, dim3((unsigned)((Ntot + 255) / 256)), dim3(256), 0, stream, *params,
                     xx[0], xx[1], xx[2], scratch + 2 * NUM_EVOL_GFS * Ntot);
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}

// Device memory of a captured step on the grid, nothing in it yet. nullptr where the two launches do
// not cover the grid, or without memory: the caller takes the unfused step.
static double *nrpy_sommerfeld_chain_scratch(const paramstruct *params, double *xx[3], const bc_struct *bc) {
  if (!params || !bc || !xx || !xx[0] || !xx[1] || !xx[2] || nrpy_check_params(params)) return nullptr;
  if (bc->N[0] != params->Nxx_plus_2NGHOSTS0 || bc->N[1] != params->Nxx_plus_2NGHOSTS1 ||
      bc->N[2] != params->Nxx_plus_2NGHOSTS2 || bc->N[0] < NRPY_SOMMERFELD_MIN_N || bc->N[1] < NRPY_SOMMERFELD_MIN_N ||
      bc->N[2] < NRPY_SOMMERFELD_MIN_N || !nrpy_sommerfeld_chainable(bc))
    return nullptr;
  const size_t Ntot = (size_t)bc->N[0] * bc->N[1] * bc->N[2];
  double *p = nullptr;
  if (hipMalloc((void **)&p, sizeof(double) * NRPY_SOM_NSCRATCH * Ntot) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

static int nrpy_sommerfeld_chain(const int S, const paramstruct *params, const bc_struct *bc, const int8_t *gfs_parity,
                                 double *R, double *y_n, double *rt, double *out, const double dt, hipStream_t stream) {
  nrpy_gf_parity_args gfp;
  memset(&gfp, 0, sizeof(gfp));
  const int rc = nrpy_bc_check(params, bc, NUM_EVOL_GFS, gfs_parity, R, &gfp);
  if (rc) return rc;
  const nrpy_fill_list &L = bc->fill_all;
  const int B = 64;
  const dim3 grid((unsigned)((L.n + B - 1) / B), NUM_EVOL_GFS);
  switch (S) {
    case 0: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<0>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp, R,
                               y_n, rt, out, dt); break;
    case 1: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<1>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp, R,
                               y_n, rt, out, dt); break;
    case 2: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<2>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp, R,
                               y_n, rt, out, dt); break;
    default: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<3>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp,
                                R, y_n, rt, out, dt); break;
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}
'''
