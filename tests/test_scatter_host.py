"""CPU check of the gradient scatter's addressing (mbx_amd/csrc/scatter.hpp), built for the host."""
import os
import subprocess

import pytest

from conftest import ROOT

CPP = os.path.join(ROOT, "tests", "cpp")
# the first atoms around which 96 * atom, 32 * 3 * atom and 3 * atom leave 31 and 32 bits, and the last
FIRST = [0, 3, 22369621, 22369622, 44739242, 44739243, 715827882, 715827883, 1431655765, 1431655766, 2 ** 31 - 3]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("scatter") / "scatter_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-I" + os.path.join(CPP, "host"), "-o", out,
                    os.path.join(CPP, "scatter_host.cpp")], check=True)
    return out


@pytest.mark.parametrize("taken", [0, 5, 127, 128])
def test_values_reach_their_atoms(program, taken):
    """Every value once at 3 * first atom + its index, through the table and past a full one."""
    text = subprocess.run([program, str(taken)] + [str(f) for f in FIRST], check=True, capture_output=True,
                          text=True).stdout
    got = sorted(tuple(int(v) for v in line.split()) for line in text.splitlines())
    assert got == sorted((f, c, 3 * f + c) for f in FIRST for c in range(9))
