"""The triangular sweeps' workgroups with some of them kept out until the others end
(host model over the kernel's own walk, bta_sweep_walk.h): whichever subset it is,
the others take over their seats and every stage completes.

The model also has the rule that looked for late seats among the outputs of stage
0 that an item of stage 1 waits for: a backward sweep with an arrow then stops for
good when the workgroups of the first rows are away, because the triangular
product of stage 1 reads the rows from its own on."""
import itertools
import random
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "pyinla_amd" / "csrc"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    gxx = shutil.which("g++")
    assert gxx, "g++ is needed for the host model"
    exe = tmp_path_factory.mktemp("walk") / "sweep_walk_model"
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-I", str(CSRC),
                    str(HERE / "native" / "sweep_walk_model.cpp"), "-o", str(exe)], check=True)

    def run(cases):
        text = "".join(f"{t} {n} {b} {a} {cap} {watch} {','.join(map(str, late)) or '-'}\n"
                       for t, n, b, a, cap, watch, late in cases)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout
        rows = [tuple(map(int, line.split())) for line in out.splitlines()]
        assert len(rows) == len(cases)
        return rows
    return run


def _seats(t, b, cap):
    return min(2 * ((b + 15) // 16) if t else (b + 7) // 8, cap, 512)


def test_every_subset_of_a_few_seats(model):
    cases = []
    for t, a in ((0, 0), (0, 3), (1, 0), (1, 3)):
        for b, cap, n in ((70, 256, 3), (70, 7, 3), (100, 4, 2), (130, 5, 1), (70, 1, 4)):
            s = _seats(t, b, cap)
            for late in itertools.chain.from_iterable(itertools.combinations(range(s), k) for k in range(s)):
                cases.append((t, n, b, a, cap, 1, late))
    assert all(ok for ok, _ in model(cases))


@pytest.mark.parametrize("b,cap", [(92, 256), (400, 256), (800, 256), (1600, 256), (2000, 256), (4500, 512)])
def test_one_seat_or_one_die_of_eight_or_random_seats(model, b, cap):
    rng = random.Random(b)
    cases = []
    for t, a in ((0, 0), (0, 6), (1, 0), (1, 6)):
        s = _seats(t, b, cap)
        lates = [[q] for q in (0, 1, 2, s // 2, s - 1)]
        lates += [list(range(1, s)), list(range(0, s - 1)), list(range(s // 2)), list(range(s // 2, s))]
        lates += [list(range(x, s, 8)) for x in range(8)] + [list(range(0, s, 2)), list(range(1, s, 2))]
        lates += [rng.sample(range(s), rng.randrange(1, s)) for _ in range(8)]
        cases += [(t, 2, b, a, cap, 1, late) for late in lates]
    bad = [c for c, (ok, _) in zip(cases, model(cases)) if not ok]
    assert not bad, bad[0]


@pytest.mark.parametrize("b", [92, 400, 1600])
def test_outputs_of_the_first_seats_have_no_reader(model, b):
    """Looking at outputs instead of claims: stage 1 completes without seat 0 of a
    backward sweep with an arrow, and nobody ever runs its items."""
    forms = [(0, 0), (0, 6), (1, 0), (1, 6)]
    got = model([(t, 3, b, a, 256, 0, [0]) for t, a in forms])
    assert [ok for ok, _ in got] == [1, 1, 1, 0]
