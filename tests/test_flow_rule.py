"""CPU tests of the rule that lets a step's sweeps be ordered by data
(csrc/b2g_flow_rule.h, compiled here by itself)."""
import ctypes
import os
import subprocess

import pytest

from util import REPO

WRAPPER = r"""
#include "b2g_flow_rule.h"
extern "C" int stride() { return b2g::kFlowStride; }
extern "C" int reaches(long long bodies) { return b2g::flow_reaches(bodies); }
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "w.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                           os.path.join(REPO, "box2d-optimized_amd", "csrc"), str(d / "w.cpp"), "-o",
                           str(d / "w.so")])
    return ctypes.CDLL(str(d / "w.so"))


def test_states_of_every_body_are_within_32_bit_offsets(rule):
    """A launch's descriptor covers stride * bodies bytes, and its loads' offsets end at the last body's state:
    whatever the rule lets through fits a signed 32-bit word."""
    last = (2 ** 31 - 1) // rule.stride()
    for bodies in (1, 2, 1 << 20, last - 1, last, last + 1, 1 << 24, (1 << 25) - 1, 1 << 25, (1 << 25) + 1, 1 << 26,
                   2 ** 31 - 1):
        reaches = bool(rule.reaches(ctypes.c_longlong(bodies)))
        assert reaches == (rule.stride() * bodies < 2 ** 31), bodies
    assert rule.reaches(ctypes.c_longlong(1_200_000))  # the largest batch of the benchmark, several times over
