"""CPU tests of the per-world solves' launch rules (csrc/b2g_world_rule.h,
compiled here by itself)."""
import ctypes
import os
import subprocess

import pytest

from util import REPO

WRAPPER = r"""
#include "b2g_world_rule.h"
extern "C" int lanes(int worlds, int cus) { return b2g::captured_world_lanes(worlds, cus); }
extern "C" int joins(int worlds, int past, int cus) { return b2g::pair_class_joins(worlds, past, cus); }
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "w.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I",
                           os.path.join(REPO, "box2d-optimized_amd", "csrc"), str(d / "w.cpp"), "-o",
                           str(d / "w.so")])
    return ctypes.CDLL(str(d / "w.so"))


def test_the_last_classes_share_a_launch_while_each_world_has_a_compute_unit(rule):
    for worlds, past, want in ((0, 0, 0), (5, 0, 0), (1, 1, 1), (50, 3, 1), (256, 1, 1), (257, 1, 0), (257, 257, 0)):
        assert rule.joins(worlds, past, 256) == want, (worlds, past)


def test_captured_workgroups_narrow_as_worlds_grow_in_number(rule):
    lanes = rule.lanes
    for worlds, want in ((1, 1024), (2, 1024), (256, 1024), (257, 512), (640, 512), (641, 256), (1000, 256),
                         (2560, 256), (2561, 128), (4096, 128), (1 << 20, 128)):
        assert lanes(worlds, 256) == want, worlds
    for cus in (32, 64, 128, 256):  # resident: 20 wavefronts of 64 lanes to a compute unit
        for worlds in range(1, 3 * cus):
            if lanes(worlds, cus) >= 512:
                assert worlds <= cus * (1280 // lanes(worlds, cus)) + cus // 2
