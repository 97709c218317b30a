"""Statement order of large kernel bodies (codegen/schedule.py): the reordered body computes the
plain body's values. Bodies are run statement by statement in Python on random stencil values,
reads before they are first used; every write must agree to the rounding of sums of up to a few
hundred terms added in another order (1e-13 of the sum of the terms' magnitudes, bounded here by
running both bodies on values of one sign and size)."""
import math
import random
import re

import pytest

from nrpytutorial_amd.codegen import schedule

SYNTHETIC = """{
  /* Step 1 of 3: reads */
  const double a = in_gfs[IDX4(AGF, i0,i1,i2)];
  const double a_i0p1_i1_i2 = in_gfs[IDX4(AGF, i0+1,i1,i2)];
  const double a_i0m1_i1_i2 = in_gfs[IDX4(AGF, i0-1,i1,i2)];
  const double b = in_gfs[IDX4(BGF, i0,i1,i2)];
  const double unused = in_gfs[IDX4(CGF, i0,i1,i2)];
  const double a_dDD00_p1 = (a_i0p1_i1_i2 - a) + (a_i0m1_i1_i2 - a);
  const double third = 1.0/3.0;
  const double Up0 = (b > 0.0) ? 1.0 : 0.0;
  const double d = invdx0*(third*a_i0p1_i1_i2 - third*a_i0m1_i1_i2);
  const double dead = a*b + d;
  const double t0 = -a*b - third*(a + 2*b)*(a + 2*b) + ((b)*(b));
  const double t1 = Up0*(d - t0) + t0;
  /* Step 3 of 3: writes */
  out_gfs[IDX4(OGF, i0, i1, i2)] = t1 + sqrt(a*a + b*b)/(a + 3*b) - (-d);
  out_gfs[IDX4(PGF, i0, i1, i2)] += 2*(a + 2*b)*a_dDD00_p1 - t0;
  out_gfs[IDX4(QGF, i0, i1, i2)] = b;
  out_gfs[IDX4(RGF, i0, i1, i2)] = third;
}
"""


def _run(body, seed):
    """{write target: value} of a body on seeded values of its reads."""
    env, out, reads = {"sqrt": math.sqrt, "cbrt": lambda x: math.copysign(abs(x) ** (1 / 3), x), "pow": pow}, {}, {}
    for k in range(3):
        env["invdx%d" % k] = 1.5 + k

    def value(text):
        m = re.match(r"\((.*)\) \? (.*) : (.*)$", text)
        if m:
            return value(m.group(2)) if eval(m.group(1), env) else value(m.group(3))
        return eval(text, env)
    for name in re.findall(r"\b(?:f\d+_of_\w+|eta)\b", body):
        env[name] = 1.0 + 0.1 * (hash_of(name) % 7)
    seen = set()
    for l in body.splitlines():
        l = l.strip()
        if not l or l in "{}" or l.startswith(("/*", "//", "__builtin_amdgcn_")):
            continue
        m = re.match(r"(?:const )?double (\w+) = (.*);$", l)
        if m:
            assert m.group(1) not in seen, "declared twice: " + m.group(1)
            seen.add(m.group(1))
            if "[" in m.group(2):
                reads.setdefault(m.group(2), random.Random("%d %s" % (seed, m.group(2))).uniform(0.5, 1.5))
                env[m.group(1)] = reads[m.group(2)]
            else:
                env[m.group(1)] = value(m.group(2))
            continue
        m = re.match(r"(\w+\[.*\]) (\+?=) (.*);$", l)
        if m:
            assert m.group(1) not in out
            out[m.group(1)] = value(m.group(3))
            continue
        m = re.match(r"(\w+) ([+-])= (.*);$", l)
        assert m, l
        env[m.group(1)] += value(m.group(3)) if m.group(2) == "+" else -value(m.group(3))
    return out


def hash_of(name):
    return sum(ord(c) * (k + 1) for k, c in enumerate(name))


@pytest.mark.parametrize("prefetch,region,sync", [(0, 0, False), (7, 3, False), (40, 16, True), (1000, 1, False)])
def test_reordered_body_computes_the_same(prefetch, region, sync):
    for body in (SYNTHETIC, _maxwell()):
        new = schedule.reorder(body, prefetch, region, sync)
        assert new == schedule.reorder(body, prefetch, region, sync)
        assert ("__builtin_amdgcn_s_barrier" in new) == sync
        for seed in (1, 2):
            want, got = _run(body, seed), _run(new, seed)
            assert sorted(want) == sorted(got)
            for k in want:
                assert abs(got[k] - want[k]) <= 1e-13 * max(1.0, abs(want[k])), (k, want[k], got[k])


def test_differences_stay_whole():
    new = schedule.reorder(SYNTHETIC, 4, 0)
    assert "const double a_dDD00_p1 = (a_i0p1_i1_i2 - a) + (a_i0m1_i1_i2 - a);" in new


def test_dead_statements_and_unknown_ones():
    assert "unused" not in schedule.reorder(SYNTHETIC, 4, 0)
    with pytest.raises(ValueError):
        schedule.reorder(SYNTHETIC.replace("  /* Step 3", "  for (int k = 0; k < 3; k++) f(k);\n  /* Step 3"), 4, 0)
    with pytest.raises(ValueError):
        schedule.reorder(SYNTHETIC.replace("in_gfs[IDX4(BGF, i0,i1,i2)];", "in_gfs[IDX4(BGF, i0,i1,i2)] + 1.0;"), 4, 0)


_CACHE = {}


def _maxwell():
    """The right-hand side of the generated curvilinear Maxwell bundle: reads, stencils, upwind-free
    expressions with reference-metric tables, eight writes."""
    if "m" not in _CACHE:
        import os
        from nrpytutorial_amd.runtime import GENDIR
        t = open(os.path.join(GENDIR, "maxwell_sinhcylindrical.hip")).read()
        i = t.index(" rhs_eval__gpu(")
        k = t[i:t.index("\n}\n", i)]
        _CACHE["m"] = k[k.index("  {\n"):]
    return _CACHE["m"]
