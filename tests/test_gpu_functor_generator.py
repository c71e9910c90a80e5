"""The region generator of user functors (tests/cpp/generator.hip): parallel rounds unless
the functor states its evaluation's work, then by that; the bins are the same."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "generator")


@pytest.fixture(scope="module")
def ways():
    assert os.path.exists(EXE), "build tests/cpp/generator (python tests/cpp/build.py)"
    out = subprocess.run([EXE], capture_output=True, text=True, timeout=120, check=True).stdout
    return {k: (int(a), int(b)) for k, a, b in (line.split() for line in out.strip().split("\n"))}


@pytest.mark.parametrize("case,workgroup", [("unstated_300", False), ("unstated_4000", False), ("cheap_300", True),
                                            ("cheap_4000", True), ("dear_300", False), ("dear_4000", False),
                                            ("nonsense_300", False), ("nonsense_4000", False)])
def test_generator(ways, case, workgroup):
    steps, rounds = ways[case]
    assert (steps > 0, rounds > 0) == (workgroup, not workgroup)


def test_same_bins(ways):
    assert ways["same"][0] == 1
