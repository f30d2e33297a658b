"""The instrumented build of the library's host code
(tests/cpp/_build/lifetime_check_asan, run on a GPU by
tests/test_gpu_lifetime_asan.py) as far as it can be checked without a GPU."""
import glob
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJ = os.path.join(ROOT, "tests", "cpp", "_build", "asan_obj")
KERNELS = sorted(os.path.basename(p)[:-4] for p in glob.glob(
    os.path.join(ROOT, "pofd_affine_amd", "csrc", "*.hip"))
    if not p.endswith("calib_copy.hip"))


@pytest.mark.parametrize("name", KERNELS)
def test_kernels_are_launched_by_name(name):
    """A launch through a kernel held as a value (a conditional expression, a
    lambda's parameter) makes clang check the function type in front of what
    is only the kernel's handle in host code, and the check fails or not by
    what lies there.  A launch by name has none."""
    obj = os.path.join(OBJ, name + ".o")
    if not os.path.exists(obj):
        pytest.skip("the instrumented objects are not built here")
    und = subprocess.run(["nm", "-u", obj], capture_output=True, text=True,
                         check=True).stdout
    assert "__asan_" in und  # instrumented
    assert "function_type_mismatch" not in und
