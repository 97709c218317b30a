"""The ghost fill's generic rows on the CPU: rows that are not products of one-dimensional
extrapolations, which no bundle's maps have (three ghost layers; test_ghost_fill_lists.py), but a
system generated with four does: layer 4 of an extrapolation is one.

The library's own text is compiled with g++ (nrpy_build_fill, nrpy_fill_point and the batch's
concatenated list from nrpy_runtime.h and nrpy_batch.h) over hand-made composed maps of a grid with
four ghost layers: extrapolated points of all layers along one, two and three axes on either side,
parity copies, sums of sources with different parity masks, a product with one coefficient changed, an
empty row. Every ghost value, for 1, 2 and 8 gridfunctions per thread and a number of gridfunctions
that is no multiple of them, equals the plain sum over the map's entries; the data are small whole
numbers, so both are exact. The same for two grids' lists appended to one. Control: a generic row
whose base is not moved when its terms are appended reads the other grid's terms."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "nrpytutorial_amd", "csrc")


def _piece(src, start, end="\n}\n"):
    i = src.index(start)
    return src[i:src.index(end, i) + len(end)]


def _pieces(rebase):
    run = open(os.path.join(CSRC, "nrpy_runtime.h")).read()
    batch = open(os.path.join(CSRC, "nrpy_batch.h")).read()
    append = _piece(batch, "struct nrpy_batch_fill_list {", "\n};\n")
    append = append[:append.index("  bool upload()")] + "};\n"
    move = "R.base += (int)h_terms.size();"
    assert move in append
    if not rebase:
        append = append.replace(move, ";")
    point = run.index("template <int K>\n__device__ __forceinline__ void nrpy_fill_point(")
    return dict(structs=(_piece(run, "struct nrpy_fill_row {", "\n};\n") + _piece(run, "struct nrpy_fill_term {", "\n};\n") +
                         re.search(r"^#define NRPY_FILL_GENERIC .*\n", run, re.M).group(0) +
                         _piece(run, "struct nrpy_fill_list {", "\n};\n") +
                         _piece(run, "struct nrpy_gf_parity_args {", "\n};\n")),
                code=(_piece(run, "__host__ __device__ static inline double nrpy_extrap_weight(") +
                      _piece(run, "static void nrpy_build_fill(") + _piece(run[point:], "template <int K>") + append))


PROG = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stddef.h>
#include <algorithm>
#include <vector>
using std::min;
using std::max;
#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__
#define NGHOSTS 4
struct paramstruct { int Nxx_plus_2NGHOSTS0, Nxx_plus_2NGHOSTS1, Nxx_plus_2NGHOSTS2; };
%(structs)s
struct bc_struct { int nghost = 0; std::vector<int> h_gdest, h_rowptr, h_src, h_negmask; std::vector<double> h_coeff; };
%(code)s
struct Grid {
  paramstruct p;
  bc_struct bc;
  std::vector<int> anchor;
  std::vector<char> take;
  nrpy_fill_list L;
  size_t Ntot;
  void row(int dest, int anch, const std::vector<int> &src, const std::vector<double> &c, const std::vector<int> &m) {
    bc.h_gdest.push_back(dest);
    anchor.push_back(anch);
    take.push_back(1);
    bc.h_src.insert(bc.h_src.end(), src.begin(), src.end());
    bc.h_coeff.insert(bc.h_coeff.end(), c.begin(), c.end());
    bc.h_negmask.insert(bc.h_negmask.end(), m.begin(), m.end());
    bc.h_rowptr.push_back((int)bc.h_src.size());
    bc.nghost++;
  }
};
static Grid make(int n0, int n1, int n2) {
  Grid g;
  const int N[3] = {n0 + 2 * NGHOSTS, n1 + 2 * NGHOSTS, n2 + 2 * NGHOSTS};
  g.p = {N[0], N[1], N[2]};
  g.Ntot = (size_t)N[0] * N[1] * N[2];
  g.bc.h_rowptr.push_back(0);
  const int stride[3] = {1, N[0], N[0] * N[1]};
  int count = 0;
  for (int idx = 0; idx < (int)g.Ntot; idx++) {
    const int i[3] = {idx %% N[0], (idx / N[0]) %% N[1], idx / (N[0] * N[1])};
    std::vector<int> src(1, 0);
    std::vector<double> c(1, 1.0);
    int out = 0;
    for (int d = 0; d < 3; d++) {
      const int l = i[d] < NGHOSTS ? NGHOSTS - i[d] : i[d] >= N[d] - NGHOSTS ? i[d] - (N[d] - NGHOSTS - 1) : 0;
      const int at = i[d] < NGHOSTS ? NGHOSTS : i[d] >= N[d] - NGHOSTS ? N[d] - NGHOSTS - 1 : i[d];
      const int s = i[d] < NGHOSTS ? stride[d] : -stride[d];
      out += l > 0;
      std::vector<int> src2;
      std::vector<double> c2;
      for (size_t k = 0; k < src.size(); k++)
        for (int a = 0; a < (l ? 3 : 1); a++) {
          /* Lagrange's quadratic through 0, 1, 2 at -l, as whole numbers */
          const double w[3] = {(l + 1) * (l + 2) / 2.0, -(double)l * (l + 2), l * (l + 1) / 2.0};
          src2.push_back(src[k] + at * stride[d] + a * s);
          c2.push_back(c[k] * (l ? w[a] : 1.0));
        }
      src = src2;
      c = c2;
    }
    if (!out) continue;
    std::vector<int> m(src.size(), 0);
    switch (count++ %% 7) {
      case 1: std::fill(m.begin(), m.end(), 5); break;                     /* a parity copy of an extrapolated point */
      case 2: m[0] = 3; break;                                             /* sources of different parity */
      case 3: c[0] += 1.0; break;                                          /* not the extrapolation's weights */
      case 4: src.clear(); c.clear(); m.clear(); break;                    /* an empty row */
      default: break;
    }
    g.row(idx, idx, src, c, m);
  }
  nrpy_build_fill(&g.p, &g.bc, g.anchor, g.take, &g.L);
  return g;
}
static double value(int gf, size_t i) { return (double)((int)((i * 7 + gf * 13) %% 41) - 20); }
static std::vector<double> want(const Grid &g, int num, const nrpy_gf_parity_args &gfp) {
  std::vector<double> f(g.Ntot * num);
  for (int gf = 0; gf < num; gf++)
    for (size_t i = 0; i < g.Ntot; i++) f[gf * g.Ntot + i] = value(gf, i);
  std::vector<double> out = f;
  for (int gf = 0; gf < num; gf++)
    for (int r = 0; r < g.bc.nghost; r++) {
      double s = 0.0;
      for (int k = g.bc.h_rowptr[r]; k < g.bc.h_rowptr[r + 1]; k++)
        s += ((g.bc.h_negmask[k] >> gfp.p[gf]) & 1 ? -1.0 : 1.0) * g.bc.h_coeff[k] * f[gf * g.Ntot + g.bc.h_src[k]];
      out[gf * g.Ntot + g.bc.h_gdest[r]] = s;
    }
  return out;
}
template <int K>
static long differ(const Grid &g, const nrpy_fill_row *rows, int n, const nrpy_fill_term *terms, int num,
                   const nrpy_gf_parity_args &gfp) {
  std::vector<double> f(g.Ntot * num);
  for (int gf = 0; gf < num; gf++)
    for (size_t i = 0; i < g.Ntot; i++) f[gf * g.Ntot + i] = value(gf, i);
  for (int r = 0; r < n; r++)
    for (int gf0 = 0; gf0 < num; gf0 += K)
      nrpy_fill_point<K>(rows[r], terms, g.p.Nxx_plus_2NGHOSTS0, g.p.Nxx_plus_2NGHOSTS0 * g.p.Nxx_plus_2NGHOSTS1, g.Ntot,
                         gf0, num, gfp, f.data());
  const std::vector<double> w = want(g, num, gfp);
  long bad = 0;
  for (size_t q = 0; q < w.size(); q++) bad += !(f[q] == w[q]);
  return bad;
}
int main() {
  const int num = 5;
  nrpy_gf_parity_args gfp = {};
  for (int gf = 0; gf < num; gf++) gfp.p[gf] = (int8_t)(gf %% 3);
  const Grid A = make(5, 3, 4), B = make(3, 6, 3);
  long bad = 0, generic = 0, product[4] = {0, 0, 0, 0}, appended = 0;
  for (const Grid *g : {&A, &B}) {
    for (const nrpy_fill_row &R : g->L.h_rows) {
      generic += R.code == NRPY_FILL_GENERIC;
      if (R.code != NRPY_FILL_GENERIC) product[!!(R.code & 7) + !!(R.code & 56) + !!(R.code & 448)]++;
    }
    if (g->L.near_edges || g->L.n != g->bc.nghost) bad++;
    bad += differ<1>(*g, g->L.h_rows.data(), g->L.n, g->L.h_terms.data(), num, gfp);
    bad += differ<2>(*g, g->L.h_rows.data(), g->L.n, g->L.h_terms.data(), num, gfp);
    bad += differ<8>(*g, g->L.h_rows.data(), g->L.n, g->L.h_terms.data(), num, gfp);
  }
  nrpy_batch_fill_list both;
  both.append(A.L, 0);
  both.append(B.L, 1);
  if (both.n != A.L.n + B.L.n || both.h_inst.front() != 0 || both.h_inst.back() != 1) appended++;
  appended += differ<8>(A, both.h_rows.data(), A.L.n, both.h_terms.data(), num, gfp);
  appended += differ<8>(B, both.h_rows.data() + A.L.n, B.L.n, both.h_terms.data(), num, gfp);
  printf("%%ld %%ld %%ld %%ld %%ld %%ld\n", bad, appended, generic, product[1], product[2], product[3]);
  return 0;
}
"""


def _run(tmp_path, rebase=True):
    src, exe = str(tmp_path / "fill.cpp"), str(tmp_path / "fill")
    with open(src, "w") as f:
        f.write(PROG % _pieces(rebase))
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=address,undefined", "-o", exe, src], check=True)
    r = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=100)
    return [int(v) for v in r.stdout.split()]


def test_generic_rows_are_the_map(tmp_path):
    bad, appended, generic, one, two, three = _run(tmp_path)
    print("%d generic rows, %d + %d + %d products" % (generic, one, two, three))
    assert bad == 0 and appended == 0
    assert min(generic, one, two, three) > 50


def test_control_terms_not_moved(tmp_path):
    bad, appended = _run(tmp_path, rebase=False)[:2]
    assert bad == 0 and appended > 0
