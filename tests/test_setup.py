"""The shortcuts of csrc/setup.h, run on the CPU from the header the kernels are
built from, against the general code beside them: tests/setup_check.cpp."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("setup") / "setup_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-w",
                    "-I", os.path.join(HERE, "host", "device"), "-I/opt/rocm/include",
                    os.path.join(HERE, "setup_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what,count,least", [("rows", 1000000, 300000), ("facing", 4000000, 400000),
                                              ("empty", 2000000, 100000)])
@pytest.mark.parametrize("seed", ["1", "2"])
def test_shortcuts_equal_the_general_code(program, what, count, least, seed):
    r = subprocess.run([program, what, str(count), seed], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and " mismatches 0" in r.stdout, r.stdout
    assert int(r.stdout.split()[1]) > least, r.stdout
