"""The estimate that a batched factorization's waves are cut by (bta_batch_rule.h)
against steps measured on an MI355X: us per block step, launch included, of equal
problems of nT tile columns side by side in one launch."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "pyinla_amd" / "csrc"
CUS, CAP = 256, 512

# nT: us of 1, 2, ... 20 problems
MEASURED = {
    2: [40, 41, 41, 41, 41, 41, 41, 41, 41, 41, 42, 42, 42, 42, 42, 42, 42, 42, 42, 42],
    4: [68, 69, 70, 70, 69, 69, 70, 70, 70, 73, 70, 72, 74, 73, 76, 74, 72, 76, 79, 88],
    8: [123, 123, 124, 129, 128, 132, 134, 151, 145, 153, 158, 182, 177, 188, 193, 218, 210, 217, 246, 272],
    13: [189, 196, 213, 220, 254, 284, 292, 332, 360, 401, 418, 472, 505, 549, 589, 634, 683, 714, 812, 830],
    19: [276, 303, 392, 464, 547, 642, 773, 893, 1026, 1198, 1356, 1514, 1659, 1779, 2075, 2203, 2283, 2467, 2711, 2836],
    25: [362, 538, 698, 990, 1192, 1543, 1863, 2313, 2612, 3004, 3318, 3713, 4008, 4412, 4850, 5217, 5664, 5893, 6457, 6668],
    32: [547, 953, 1459, 2243, 2828, 3681, 4433, 5222, 6168, 6759, 7550, 8372, 9068, 9550, 10806, 11262, 12299, 12766, 13713, 14500],
    40: [889, 1784, 3225, 4679, 6057, 7310, 9024, 10281, 12069, 13428, 15472, 16580, 18811, 19301, 22349, 22301, 25205, 25403, 27684, 28397],
}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    gxx = shutil.which("g++")
    assert gxx, "g++ is needed for the host model"
    exe = tmp_path_factory.mktemp("rule") / "batch_rule_model"
    subprocess.run([gxx, "-O1", "-std=c++17", "-Wall", "-Werror", "-I", str(CSRC),
                    str(HERE / "native" / "batch_rule_model.cpp"), "-o", str(exe)], check=True)

    def run(lines):
        out = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
        return [float(x) for x in out.stdout.split()]
    return run


def test_estimate_is_near_the_measured_steps(rule):
    keys = [(t, k) for t, row in MEASURED.items() for k in range(1, len(row) + 1)]
    est = rule([f"t {CUS} {CAP} " + " ".join([str(t)] * k) for t, k in keys])
    for (t, k), e in zip(keys, est):
        assert 0.75 <= e / MEASURED[t][k - 1] <= 1.25, (t, k, e)


@pytest.mark.parametrize("np_", [2, 3, 4, 6, 7, 9, 12, 16, 18, 20, 24, 40])
def test_waves_are_near_the_fastest_measured(rule, np_):
    for t, row in MEASURED.items():
        nl = int(rule([f"l 20 {CUS} {CAP} " + " ".join([f"10:{t}"] * np_)])[0])

        def waves(k):
            full, rest = divmod(np_, k)
            return full * row[k - 1] + (row[rest - 1] if rest else 0)
        best = min(waves(k) for k in range(1, min(np_, 20) + 1))
        assert waves(nl) <= 1.1 * best, (t, nl, waves(nl), best)


def test_uneven_problems_and_limits(rule):
    assert rule([f"l 20 {CUS} {CAP} 40:4 30:8 8:32"])[0] >= 1
    assert rule([f"l 2 {CUS} {CAP} " + " ".join(["5:2"] * 9)])[0] == 2
    assert rule([f"l 20 {CUS} 8 " + " ".join(["5:2"] * 9)])[0] <= 4  # no more than have a helper each
