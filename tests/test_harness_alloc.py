"""The fold harness after an allocation that failed (native/harness_alloc_check.cpp): the next call on
the thread must not write past row arrays that the failed call left short."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("harness") / "harness_alloc_check")
    src = os.path.join(ROOT, "taco_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "include"), "-I", src, "-o", out,
                    os.path.join(HERE, "native", "harness_alloc_check.cpp"), os.path.join(src, "taco", "harness.cpp"),
                    os.path.join(src, "taco", "tokenizer.cpp")], check=True)
    return out


@pytest.mark.parametrize("allocated", [0, 1, 2])  # of the inputs, the queries and the answers
def test_call_after_a_failed_allocation(exe, allocated):
    r = subprocess.run([exe, str(allocated)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout + r.stderr)
