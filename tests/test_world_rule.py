"""CPU test of the captured per-world solve's workgroup size
(csrc/b2g_world_rule.h, compiled here by itself)."""
import ctypes
import os
import subprocess

from util import REPO


def test_captured_workgroups_narrow_as_worlds_grow_in_number(tmp_path):
    (tmp_path / "w.cpp").write_text('#include "b2g_world_rule.h"\nextern "C" int lanes(int worlds, int cus) '
                                    "{ return b2g::captured_world_lanes(worlds, cus); }\n")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I",
                           os.path.join(REPO, "box2d-optimized_amd", "csrc"), str(tmp_path / "w.cpp"), "-o",
                           str(tmp_path / "w.so")])
    lanes = ctypes.CDLL(str(tmp_path / "w.so")).lanes
    for worlds, want in ((1, 1024), (2, 1024), (256, 1024), (257, 512), (640, 512), (641, 256), (1000, 256),
                         (2560, 256), (2561, 128), (4096, 128), (1 << 20, 128)):
        assert lanes(worlds, 256) == want, worlds
    for cus in (32, 64, 128, 256):  # resident: 20 wavefronts of 64 lanes to a compute unit
        for worlds in range(1, 3 * cus):
            if lanes(worlds, cus) >= 512:
                assert worlds <= cus * (1280 // lanes(worlds, cus)) + cus // 2
