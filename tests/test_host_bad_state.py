"""The host code's answers to device states that are no results (tests/hostcheck/bad_state.cpp),
on the CPU: the call fails, and nothing is indexed with them."""
import os
import subprocess

import pytest

from test_host_asan import CLANG, HERE, HIPCC, ROOT, run

pytestmark = pytest.mark.skipif(not (os.path.exists(HIPCC) and os.path.exists(CLANG)),
                                reason="no ROCm clang")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("bad_state"))
    src = os.path.join(ROOT, "qrdm_amd", "csrc", "driver.hip")
    run([HIPCC, "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-O1", "-fPIC", "-c", src, "-o", "driver.o"], d)
    run([HIPCC, "--cuda-host-only", "-x", "hip", "-O1", "-c",
         os.path.join(HERE, "hostcheck", "bad_state.cpp"), "-o", "bad_state.o"], d)
    run([CLANG, "driver.o", "bad_state.o", "-o", "bad_state"], d)
    return os.path.join(d, "bad_state")


def result(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.returncode
    return int(r.stdout)


def test_panel_given_up_with_every_column_fixed(program):
    assert result(program, "panel") <= -1000


def test_wide_candidate_past_the_columns(program):
    assert result(program, "index") <= -1000
