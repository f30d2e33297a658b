"""The instrumented build of the library's host code
(tests/cpp/_build/lifetime_check_asan, run on a GPU by
tests/test_gpu_lifetime_asan.py) as far as it can be checked without a GPU."""
import glob
import hashlib
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")
CSRC = os.path.join(ROOT, "pofd_affine_amd", "csrc")
EXE = os.path.join(CPP, "_build", "lifetime_check_asan")
OBJ = os.path.join(CPP, "_build", "asan_obj")
KERNELS = sorted(os.path.basename(p)[:-4] for p in glob.glob(
    os.path.join(CSRC, "*.hip"))
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


def stale_sources():
    """The sources that are not as the executable was made from."""
    out, seen = [], set()
    with open(EXE + ".sources") as f:
        for line in f:
            digest, name = line.split(None, 1)
            path = os.path.normpath(os.path.join(CPP, name.strip()))
            seen.add(path)
            with open(path, "rb") as g:
                if hashlib.sha256(g.read()).hexdigest() != digest:
                    out.append(path)
    return out + [p for p in glob.glob(os.path.join(CSRC, "*.h"))
                  if p not in seen]


def test_executable_is_of_these_sources():
    if not os.path.exists(EXE):
        pytest.skip("the instrumented executable is not built here")
    assert stale_sources() == []


@pytest.mark.parametrize("header", sorted(
    os.path.basename(p) for p in glob.glob(os.path.join(CSRC, "*.h"))))
def test_objects_follow_the_headers(header):
    """make's own plan after a change of one header takes every object whose
    source includes it, itself or through another header."""
    def uses(path, seen=()):
        with open(path) as f:
            inc = re.findall(r'^#include "(\w+\.h)"', f.read(), re.M)
        return header in inc or any(
            uses(os.path.join(CSRC, i), seen + (i,)) for i in inc
            if i not in seen and os.path.exists(os.path.join(CSRC, i)))
    plan = subprocess.run(
        ["make", "-n", "-C", CPP, "-W",
         os.path.join("../../pofd_affine_amd/csrc", header), "asan"],
        capture_output=True, text=True, check=True).stdout
    for src in glob.glob(os.path.join(CSRC, "*.hip")) + \
            glob.glob(os.path.join(CSRC, "*.cpp")):
        stem = os.path.basename(src).rsplit(".", 1)[0]
        if stem != "calib_copy" and uses(src):
            assert "-o _build/asan_obj/%s.o" % stem in plan, (header, stem)
