"""bench.py's host logic on the CPU: the mixed-vs-FP64 comparison of two states, the HBM-traffic
table of two counter files, and the single-GPU refusal of --gpus above 1 (before anything
touches a GPU)."""

import csv
import json
import os
import re
import subprocess
import sys

import numpy as np

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_compare_forms_relative_errors_and_separation():
    rng = np.random.default_rng(3)
    ref = {k: rng.standard_normal((5, 4, 8)) for k in ("uf", "vf", "wf", "pf")}
    scale = {"uf": 1e-6, "vf": 2e-7, "wf": 0.0, "pf": 3e-5}
    mixed = {}
    for k, a in ref.items():
        d = rng.standard_normal(a.shape)
        mixed[k] = a + scale[k] * np.linalg.norm(a) / np.linalg.norm(d) * d
    x = np.linspace(0.0, 1.0, 16)
    cf0 = np.cos(2 * np.pi * x)                      # + to -, then - to +
    cf1 = cf0 * (1 + 1e-6)
    wall = {0: (cf0, 0.25, 0.75), 1: (cf1, 0.25 + 3e-9, np.nan)}
    errs, sep, finite = bench.compare_forms({0: ref, 1: mixed}, wall)
    for k in ("uf", "vf", "wf", "pf"):
        assert abs(errs[k] - scale[k]) <= 1e-3 * scale[k] + 1e-18, (k, errs[k])
    assert abs(errs["wall_shear"] - 1e-6) < 1e-9
    assert sep["x_sep_fp64"] == 0.25 and abs(sep["x_sep_abs_diff"] - 3e-9) < 1e-15
    assert sep["x_reatt_abs_diff"] is None           # no reattachment in one form: JSON null
    assert finite
    mixed["pf"] = mixed["pf"].copy()
    mixed["pf"][0, 0, 0] = np.nan
    assert not bench.compare_forms({0: ref, 1: mixed}, wall)[2]


def test_several_gpus_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120, cwd=ROOT)
    assert r.returncode == 2
    assert "one GPU" in r.stderr


def test_traffic_table_of_counter_files(tmp_path):
    """Two steps of each form as the counter runs list them: a calibrating copy, and each step
    ended by the norm, by the name that its kernel has in the sources."""
    with open(os.path.join(ROOT, "lsbflow_amd", "csrc", "spectral.hip")) as fh:
        norm = re.search(r"__global__ void (k_norm\w*)\(", fh.read()).group(1)
    step = {"fp64": "void lsb::k_yfwd_rhs<double, double, 16, 16, 16>(int)",
            "mixed": "void lsb::k_yfwd_rhs<float, float, 16, 16, 16>(int)"}
    names = ["__amd_rocclr_copyBuffer"]
    for form in ("fp64", "mixed"):
        names += 2 * [step[form], f"lsb::{norm}(lsb::FieldList<double>, int)"]
    kib = bench.COPY_BYTES / 1024.0
    files = []
    for counter, copied in (("FETCH_SIZE", kib / 2), ("WRITE_SIZE", kib)):
        files.append(str(tmp_path / f"{counter}.csv"))
        with open(files[-1], "w", newline="") as fh:
            w = csv.writer(fh)
            w.writerow(["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
            for i, n in enumerate(names):
                v = copied if i == 0 else 100.0 if "double, double" in n else 50.0 if "float" in n else 1.0
                w.writerow([i, n, counter, v])
    out = str(tmp_path / "traffic.json")
    assert bench.pmc_summarize(*files, out_path=out) == 0
    with open(out) as fh:
        t = json.load(fh)
    assert t["classes"]["fp64"]["rhs"]["bytes_per_step"] == 100 * 1024 * 3
    assert t["classes"]["mixed"]["rhs"]["bytes_per_step"] == 50 * 1024 * 3
