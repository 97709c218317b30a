"""The order of a launch's tiles (NRPY_BLOCK_COORDS_AS in nrpy_runtime_pre.h) on the CPU: the macro's own text,
compiled with g++, gives every tile of the index box to exactly one block, through whole planes and
in slabs, for box sides from one point to several slabs, tile shapes the kernels use. With whole planes tile t of an XCD's
range is the box's tile number t; in slabs i2 runs inside a slab of 8 tiles along i1."""
import os
import re
import subprocess

PRE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nrpytutorial_amd", "csrc",
                   "nrpy_runtime_pre.h")

PROG = r"""
#include <stdio.h>
#include <vector>
#include <algorithm>
using std::min;
static struct { int x, y, z; } blockDim, blockIdx;
%(macros)s
static long tile(int nb, bool whole, int n0, int n1, int n2, int nbx, int nby) {
  NRPY_BLOCK_COORDS_AS(nb, whole, n0, n1, n2)
  return nrpy_bx < 0 || nrpy_by < 0 || nrpy_bz < 0 || nrpy_bx >= nbx || nrpy_by >= nby ? -1
                                                                                       : nrpy_bx + (long)nbx * (nrpy_by + (long)nby * nrpy_bz);
}
int main() {
  const int shapes[5][3] = {{64, 4, 1}, {64, 1, 4}, {16, 4, 4}, {16, 16, 1}, {1, 1, 1}};
  const int sides[11] = {1, 3, 7, 8, 9, 16, 17, 31, 33, 64, 67};
  long bad = 0, boxes = 0, order = 0;
  for (const auto &s : shapes)
    for (int n0 : {1, 17, 70})
      for (int n1 : sides)
        for (int n2 : sides)
          for (int whole = 0; whole < 2; whole++) {
            blockDim.x = s[0]; blockDim.y = s[1]; blockDim.z = s[2];
            const int nbx = (n0 + s[0] - 1) / s[0], nby = (n1 + s[1] - 1) / s[1], nbz = (n2 + s[2] - 1) / s[2];
            const int nb = nbx * nby * nbz;
            std::vector<int> seen(nb, 0);
            std::vector<long> of(nb);
            for (int b = 0; b < nb; b++) {
              blockIdx.x = b;
              const long t = tile(nb, whole, n0, n1, n2, nbx, nby);
              if (t < 0 || t >= nb) { bad++; continue; }
              seen[t]++;
              of[b] = t;
            }
            for (int v : seen) bad += v != 1;
            boxes++;
            /* blocks x, x + 8, ... of an XCD are consecutive in the order */
            std::vector<long> rank(nb);
            long r = 0;
            for (int z = 0; whole && z < nb; z++) rank[z] = z;
            for (int y0 = 0; !whole && y0 < nby; y0 += NRPY_SLAB)
              for (int z = 0; z < nbz; z++)
                for (int y = y0; y < min(y0 + NRPY_SLAB, nby); y++)
                  for (int x = 0; x < nbx; x++) rank[x + (long)nbx * (y + (long)nby * z)] = r++;
            for (int b = 0; !bad && b + NRPY_NUM_XCD < nb; b++) order += rank[of[b + NRPY_NUM_XCD]] != rank[of[b]] + 1;
          }
  printf("%%ld %%ld %%ld\n", bad, order, boxes);
}
"""


def test_every_tile_once(tmp_path):
    src = open(PRE).read()
    macros = "".join(re.search(r"^#define %s\b.*?(?<!\\)\n" % n, src, re.M | re.S).group(0)
                     for n in ("NRPY_NUM_XCD", "NRPY_SLAB", "NRPY_BLOCK_COORDS_AS"))
    c, exe = str(tmp_path / "tiles.cpp"), str(tmp_path / "tiles")
    with open(c, "w") as f:
        f.write(PROG % {"macros": macros})
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, c], check=True)
    bad, order, boxes = (int(v) for v in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split())
    assert boxes == 5 * 3 * 11 * 11 * 2 and bad == 0 and order == 0


def test_kernels_take_the_form_their_reads_call_for():
    """Kernels without a neighbour's read go through whole planes, others by the size of a plane."""
    gen = os.path.join(os.path.dirname(PRE), "generated", "bssn_cartesian.hip")
    text = open(gen).read()
    for name, form in (("enforce_detgammabar_constraint", "_POINTWISE"), ("Ricci_eval", ""), ("rhs_eval_rk4_substep_g1", ""),
                       ("Ricci_eval_vjp_transpose_hDD00", ""), ("enforce_detgammabar_constraint_vjp_pointwise", "_POINTWISE"),
                       ("initial_data", "_POINTWISE")):
        m = re.search(r"__global__ [^\n]*\b%s__gpu\(" % name, text)
        assert m, name
        assert "  NRPY_BLOCK_COORDS%s(" % form in text[m.start():text.index("\n}\n", m.start())], name
    assert "#define NRPY_SLAB_MIN_PLANE 2604\n" in text
    assert "#define NRPY_SLAB_MIN_PLANE 0x7fffffff\n" in open(gen.replace("cartesian", "spherical_sym2")).read()
