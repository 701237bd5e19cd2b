"""CPU tests of the rule that lets a step's sweeps be ordered by data
(csrc/b2g_flow_rule.h, compiled here by itself)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from util import REPO

WRAPPER = r"""
#include "b2g_flow_rule.h"
extern "C" int stride() { return b2g::kFlowStride; }
extern "C" int plan(long long contacts, long long joints, int* per, int* joint_blocks) {
  const b2g::FlowPlan p = b2g::flow_plan(contacts, joints);
  *per = p.per;
  *joint_blocks = p.joint_blocks;
  return p.blocks;
}
extern "C" int rest_steps() { return b2g::kFlowRestSteps; }
extern "C" int resident(int compute_units) { return b2g::flow_resident_blocks(compute_units); }
extern "C" void rest(int steps, const int* withdrawn, int* take) {
  b2g::FlowRest r;
  for (int k = 0; k < steps; ++k) take[k] = r.take(withdrawn[k]);
}
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


def test_a_launch_has_a_lane_for_every_constraint(rule):
    per, jb = ctypes.c_int(), ctypes.c_int()
    for contacts, joints in ((0, 0), (1, 0), (0, 1), (63, 1), (1023, 1), (1024, 1), (34600, 0), (12000, 15000),
                             (65536, 0), (65537, 0), (131072, 0), (131072, 1), (2_000_000_000, 3)):
        blocks = rule.plan(ctypes.c_longlong(contacts), ctypes.c_longlong(joints), ctypes.byref(per),
                           ctypes.byref(jb))
        assert 1 <= per.value <= 64 and jb.value * 4 * per.value >= joints
        assert (blocks - jb.value) * 4 * per.value >= contacts
        assert contacts + joints > 0 or blocks == 0
    # two workgroups of 256 lanes on each of 256 compute units: 131,072 constraints, none more
    assert rule.resident(256) * 256 == 131072
    assert rule.plan(ctypes.c_longlong(131072), ctypes.c_longlong(0), ctypes.byref(per), ctypes.byref(jb)) == 512


def test_steps_rest_from_the_launches_after_a_withdrawal(rule):
    n, rest = 3000, rule.rest_steps()
    withdrawn = np.zeros(n, np.int32)
    withdrawn[10:] = 1  # one launch in step 9, then both of one later
    withdrawn[1000:] = 3
    take = np.zeros(n, np.int32)
    rule.rest(n, withdrawn.ctypes.data_as(ctypes.c_void_p), take.ctypes.data_as(ctypes.c_void_p))
    want = np.ones(n, np.int32)
    want[10:10 + rest] = want[1000:1000 + rest] = 0
    assert np.array_equal(take, want)
