"""The kernels that bench.py names for a timing class are those its launches run."""
import re
from pathlib import Path

import bench

CSRC = Path(bench.__file__).resolve().parent / "pyinla_amd" / "csrc"


def _names(label):
    return set(re.findall(r"k_\w+", label))


def test_grouped_class_names_every_kernel_of_a_plan():
    text = (CSRC / "bta_gemm.hip").read_text()
    at = text.index("void DevPlan::launch")
    body = text[at:text.index("\n}\n", at)]
    default = body[body.index("switch (e.kernel)"):]
    assert _names(bench.class_kernel(2, 2000, 400, 400)) == set(re.findall(r"run\((k_\w+)", default))


def test_update_class_names_both_forms():
    text = (CSRC / "bta_potrf.hip").read_text()
    assert "k_gemm_nt_sub" in text
    assert _names(bench.class_kernel(1, 4500, 200, 200)) == {"k_gemm_nt_sub", "k_gemm_grouped"}


def test_panel_variants_by_their_launches():
    n = 2 * 200
    assert bench.class_kernel(0, 2000, n, n) == "k_panel_flow"
    assert bench.class_kernel(0, 2000, 32 * n, n) == "k_panel_step"
    assert bench.class_kernel(0, 40, 2, n) == "k_chain64"
    assert bench.class_kernel(0, 40, n, n) == "k_panel_step"  # arrows above 32 rows
    assert bench.class_kernel(3, 40, n, n) == "k_sweep_solo" and bench.class_kernel(3, 65, n, n) == "k_sweep"
