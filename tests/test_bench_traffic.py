"""The HBM traffic that bench.py prints for the slowest BSSN kernel is that of the committed counters, and
those were collected for the kernel as it is: its text and tile order hash to what the counters'
summary names. With another text, or another output group, nothing is printed."""
import json
import os
import shutil

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNEL = "rhs_eval_rk4_substep_g2"


def test_traffic_is_of_the_present_kernel(tmp_path):
    with open(os.path.join(ROOT, "profiles", KERNEL + "_bssn192_traffic.json")) as f:
        d = json.load(f)
    assert bench.measured_traffic(KERNEL, 192, d["outputs"]) == d["hbm_bytes_per_launch"]
    assert bench.measured_traffic(KERNEL, 192, d["outputs"][:-1]) is None
    csrc = os.path.join(ROOT, "nrpytutorial_amd", "csrc")
    os.makedirs(str(tmp_path / "generated"))
    for name in ("nrpy_runtime_pre.h", os.path.join("generated", "bssn_cartesian.hip")):
        shutil.copy(os.path.join(csrc, name), str(tmp_path / name))
    assert bench.kernel_text_hash(KERNEL, str(tmp_path)) == d["kernel_text_sha1"]
    p = str(tmp_path / "nrpy_runtime_pre.h")
    text = open(p).read()
    with open(p, "w") as f:
        f.write(text.replace("#define NRPY_SLAB 8", "#define NRPY_SLAB 16"))
    assert bench.kernel_text_hash(KERNEL, str(tmp_path)) != d["kernel_text_sha1"]
