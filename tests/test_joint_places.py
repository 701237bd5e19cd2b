"""CPU tests of the joints' places in their bodies' update sequences
(csrc/b2g_joints.h, compiled here by itself): the ordered sweeps (b2g_flow.h)
let a wavefront's lanes go in the order of these colours, so a colour or rank
that does not fit its word makes constraints wait for each other."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from util import REPO

WRAPPER = r"""
#include "b2g_joints.h"
struct Ends { int body_a, body_b; };
extern "C" int places(int nj, int nb, const Ends* ends, const int* dynamic, int* order, int* x, int* y, int* degree) {
  b2g::JointTables t;
  if (!b2g::joint_tables(nj, nb, [&](int q) -> const Ends& { return ends[q]; },
                         [&](int b) { return dynamic[b] != 0; }, &t)) return -1;
  for (int k = 0; k < nj; ++k) {
    order[k] = t.order[k];
    x[k] = b2g::pack_joint_ranks(t.places[k]);
    y[k] = t.places[k].colour;
  }
  for (int b = 0; b < nb; ++b) degree[b] = t.degree[b];
  return (int)t.offsets.size() - 1;
}
"""


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    d = tmp_path_factory.mktemp("joints")
    (d / "w.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                           os.path.join(REPO, "box2d-optimized_amd", "csrc"), str(d / "w.cpp"), "-o",
                           str(d / "w.so")])
    lib = ctypes.CDLL(str(d / "w.so"))

    def run(ends, dynamic):
        ends, dynamic = np.ascontiguousarray(ends, np.int32), np.ascontiguousarray(dynamic, np.int32)
        nj, nb = len(ends), len(dynamic)
        order, x, y = (np.zeros(nj, np.int32) for _ in range(3))
        degree = np.zeros(nb, np.int32)
        colours = lib.places(nj, nb, *(a.ctypes.data_as(ctypes.c_void_p) for a in
                                       (ends, dynamic, order, x, y, degree)))
        # as the device unpacks the words
        return colours, order, np.stack([x & 0xff, x >> 8], 1), y, degree
    return run


def _anchored(single, double, flip=False):
    """Pendulums on the static body 0, the last `double` of them with a second link; anchors first."""
    first = [(0, 1 + i) for i in range(single + double)]
    second = [(1 + single + i, 1 + single + double + i) for i in range(double)]
    ends = np.array(first + second, np.int32)
    return ends[:, ::-1] if flip else ends, np.array([0] + [1] * (single + 2 * double), np.int32)


def _random(seed, nj, nb, statics):
    rng = np.random.default_rng(seed)
    ends = np.stack([rng.integers(0, nb, nj), rng.integers(0, nb - 1, nj)], 1)
    ends[:, 1] += ends[:, 1] >= ends[:, 0]
    return ends, (np.arange(nb) >= statics).astype(np.int32)


GRAPHS = {
    "none": (np.zeros((0, 2), np.int32), [1, 1]),
    "one": ([[0, 1]], [0, 1]),
    "255_on_one_static": _anchored(255, 0),
    "256_on_one_static": _anchored(256, 1),
    "300_of_them_10_double": _anchored(290, 10),
    "1202_of_them_1_double": _anchored(1200, 1),
    "1202_the_other_way_round": _anchored(1200, 1, True),
    "5000_of_them_777_double": _anchored(4223, 777),
    "random": _random(1, 3000, 900, 3),
    "random_one_static": _random(2, 700, 40, 1),
}


@pytest.mark.parametrize("name", list(GRAPHS))
def test_places_hold_colour_and_ranks(tables, name):
    ends, dynamic = GRAPHS[name]
    ends, dynamic = np.asarray(ends, np.int32).reshape(-1, 2), np.asarray(dynamic)
    colours, order, rank, colour, degree = tables(ends, dynamic)
    assert sorted(order) == list(range(len(ends))) and (np.diff(colour) >= 0).all()
    assert colours == (colour.max() + 1 if len(ends) else 0) and (rank < 64).all()
    seen = {}
    for k, q in enumerate(order):
        for side in (0, 1):
            b = ends[q, side]
            if not dynamic[b]:
                assert rank[k, side] == 0
                continue
            assert rank[k, side] == len(seen.get(b, []))
            assert colour[k] not in seen.get(b, [])  # a dynamic body's joints differ in colour
        for b in set(ends[q]):
            if dynamic[b]:
                seen.setdefault(b, []).append(colour[k])
    assert all(degree[b] == len(seen.get(b, [])) for b in range(len(dynamic)))


@pytest.mark.parametrize("name", [n for n in GRAPHS if n != "none"])
@pytest.mark.parametrize("per", [1, 2, 3, 64])
def test_ordered_sweeps_come_to_an_end(tables, name, per):
    """The ordered sweeps' rule, wavefront by wavefront: the lanes of a wave's least (iteration, colour) go once
    each dynamic body of theirs has had the updates that precede them. Every joint gets through."""
    ends, dynamic = (np.asarray(v) for v in GRAPHS[name])
    _, order, rank, colour, degree = tables(ends, dynamic)
    body, dyn = ends[order], dynamic[ends[order]] != 0
    count, iterations = np.zeros(len(dynamic), int), 3
    turn = np.zeros(len(order), int)
    while True:
        went = False
        for lo in range(0, len(order), per):
            lanes = np.arange(lo, min(lo + per, len(order)))
            lanes = lanes[turn[lanes] < iterations]
            if len(lanes) == 0:
                continue
            key = turn[lanes] * 64 + colour[lanes]
            lanes = lanes[key == key.min()]
            want = turn[lanes, None] * degree[body[lanes]] + rank[lanes]
            if (dyn[lanes] & (count[body[lanes]] != want)).any():
                continue
            for k in lanes:
                count[np.unique(body[k][dyn[k]])] += 1
            turn[lanes] += 1
            went = True
        if not went:
            break
    assert (turn == iterations).all(), "joints wait for each other"


def test_a_65th_joint_on_a_dynamic_body_is_refused(tables):
    ends = [(0, 1 + i) for i in range(65)]
    assert tables(ends[:64], [1] * 66)[0] == 64
    assert tables(ends, [1] * 66)[0] == -1
