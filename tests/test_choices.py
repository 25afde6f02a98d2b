"""Host-only tests of the engine's choices of kernels (tests/cpp/choices.cpp).

The driver is linked with the engine's own objects and fills in plans by hand; no GPU is
used and nothing is launched.
"""
import os
import subprocess

import pytest

from conftest import ROOT
from kissfft_amd import build as B

OBJ = os.path.join(B.LIBDIR, "obj")
OBJECTS = [os.path.join(OBJ, os.path.splitext(s)[0] + ".o") for s in B.ENGINE_SOURCES + ["kfa_rtc_headers.cpp"]]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not all(os.path.exists(o) for o in OBJECTS):
        B.build(["float"], verbose=False)
    exe = str(tmp_path_factory.mktemp("choices") / "choices")
    src = os.path.join(ROOT, "tests", "cpp", "choices.cpp")
    r = subprocess.run([B.HIPCC, *B.HIP_FLAGS, "-I", B.CSRC, "-I", B.INCLUDE, "-x", "hip", src, "-x", "none", *OBJECTS,
                        "-lpthread", "-ldl", "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def check(driver, case):
    r = subprocess.run([driver, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr


@pytest.mark.parametrize("case", ["open_choice_is_not_the_plans", "short_real_rows_do_not_depend_on_the_past",
                                  "shortest_compiled_row_as_set", "short_complex_lines_are_decided", "fixed_split_needs_no_allocation",
                                  "bluestein_only_where_exact", "split_tables_are_bounded",
                                  "compiled_planes_where_they_pay"])
def test_choice(driver, case):
    check(driver, case)
