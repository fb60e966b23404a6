"""The arrays that the stepper's block form, the brick and the adjoint
allocate at first use (tgh_scratch.hpp ensure_arrays), compiled for the CPU
with g++: after a call that found no memory for one of them, the next call
does not take the missing one for made. Every place that allocates several
goes through it."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "treegeneralizedharmonic.jl_amd", "csrc")


def test_a_failed_allocation_is_not_taken_for_made(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not installed")
    exe = str(tmp_path / "scratch_arrays")
    subprocess.run([gxx, "-std=c++17", "-O1", "-o", exe, os.path.join(HERE, "native", "scratch_arrays.cpp")], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, (res.returncode, res.stdout, res.stderr)
    assert res.stdout.startswith("ok")


@pytest.mark.parametrize("name", ["ensure_block_stage", "ensure_brick", "adj_prepare"])
def test_the_arrays_of_a_form_are_each_looked_at(name):
    src = open(os.path.join(CSRC, "tgh_api.hip")).read()
    body = re.search(r"int %s\(tgh_problem\* p\) \{\n(.*?)\n\}" % name, src, re.S).group(1)
    assert "ensure_device(p, {" in body
    assert "hipMalloc(" not in body
