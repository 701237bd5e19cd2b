// b2g_joints.h -- the joint graph's colours, and each joint's place in the
// update sequences of its bodies. Host code only, without a device header: the
// CPU tests compile it by itself.
#pragma once

#include <algorithm>
#include <vector>

namespace b2g {

constexpr int kMaxJointColours = 64;

// A joint's place: its colour, and how many joints each of its bodies has in
// earlier colours. Joints of one dynamic body differ in colour, so its ranks
// stay below the colour limit; a body that is not dynamic may carry any number
// of joints, is never waited for, and has rank 0 throughout.
struct JointPlace {
  int rank_a, rank_b, colour;
};

struct JointTables {
  std::vector<int> order;          // joints by colour
  std::vector<int> offsets;        // first joint of each colour in `order`, and the end
  std::vector<JointPlace> places;  // in `order`
  std::vector<int> degree;         // per body: joints on it (0 where it is not dynamic)
};

// What the device keeps of a place in two words: both ranks (8 bits each) and
// the colour, in words of their own.
constexpr int pack_joint_ranks(const JointPlace& p) { return p.rank_a | p.rank_b << 8; }

// Greedy colouring in joint order; ends(q) gives joint q's bodies (.body_a,
// .body_b), dynamic(b) says whether body b is. False: more than
// kMaxJointColours colours.
template <class Ends, class Dynamic>
bool joint_tables(int joints, int bodies, Ends ends, Dynamic dynamic, JointTables* out) {
  std::vector<unsigned long long> used(std::max(bodies, 1), 0ull);
  std::vector<int> colour(joints, 0);
  int colours = 0;
  for (int q = 0; q < joints; ++q) {
    const auto& j = ends(q);
    const bool da = dynamic(j.body_a), db = dynamic(j.body_b);
    const unsigned long long m = (da ? used[j.body_a] : 0ull) | (db ? used[j.body_b] : 0ull);
    int c = 0;
    while (c < kMaxJointColours && (m >> c) & 1ull) ++c;
    if (c >= kMaxJointColours) return false;
    colour[q] = c;
    if (da) used[j.body_a] |= 1ull << c;
    if (db) used[j.body_b] |= 1ull << c;
    colours = std::max(colours, c + 1);
  }
  out->offsets.assign(colours + 1, 0);
  for (int q = 0; q < joints; ++q) out->offsets[colour[q] + 1]++;
  for (int c = 0; c < colours; ++c) out->offsets[c + 1] += out->offsets[c];
  out->order.resize(joints);
  std::vector<int> cursor(out->offsets);
  for (int q = 0; q < joints; ++q) out->order[cursor[colour[q]]++] = q;
  out->degree.assign(std::max(bodies, 1), 0);
  out->places.resize(joints);
  for (int k = 0; k < joints; ++k) {
    const auto& j = ends(out->order[k]);
    JointPlace& p = out->places[k];
    p = JointPlace{0, 0, colour[out->order[k]]};
    if (dynamic(j.body_a)) p.rank_a = out->degree[j.body_a];
    if (dynamic(j.body_b)) p.rank_b = out->degree[j.body_b];
    if (dynamic(j.body_a)) ++out->degree[j.body_a];
    if (dynamic(j.body_b) && j.body_b != j.body_a) ++out->degree[j.body_b];
  }
  return true;
}

}  // namespace b2g
