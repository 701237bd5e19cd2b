// b2g_flow_rule.h -- when a step's sweeps are ordered by data (b2g_flow.h).
// Host code only, without a device header: the CPU tests compile it by itself.
#pragma once

#include <algorithm>
#include <climits>

namespace b2g {

constexpr int kFlowLanes = 64;    // lanes of a wavefront
constexpr int kFlowThreads = 256;
constexpr int kFlowWaves = kFlowThreads / kFlowLanes;
constexpr int kFlowSpread = 1024;  // wavefronts that a phase is spread over before its lanes fill up

// Workgroups of a flow launch at most: two per CU (128 registers per lane
// allow four), so that two batches on two streams still fit together.
constexpr int flow_resident_blocks(int compute_units) { return 2 * compute_units; }

// A phase's launch: `per` constraints to a wavefront (few where the waves are
// few: one or two per SIMD; up to one per lane), the joints' workgroups first.
struct FlowPlan {
  int per, joint_blocks, blocks;
};
inline FlowPlan flow_plan(long long contacts, long long joints) {
  const long long even = (contacts + joints + kFlowSpread - 1) / kFlowSpread;
  const int per = (int)std::min<long long>(kFlowLanes, std::max<long long>(1, even));
  const long long share = (long long)per * kFlowWaves;
  const int jb = (int)((joints + share - 1) / share);
  return FlowPlan{per, jb, jb + (int)((contacts + share - 1) / share)};
}

// A launch that found no room for all its workgroups waited a millisecond and
// left its sweeps to one of them (flow_enter). The device then holds other
// work, and is likely to in the next step: steps take a launch per colour for
// a while, then try again.
constexpr int kFlowRestSteps = 256;
struct FlowRest {
  int seen = 0;  // withdrawals counted on the device, as last read
  int left = 0;  // steps yet to take without the flow launches
  // whether the coming step may take them
  bool take(int withdrawn) {
    if (withdrawn != seen) {
      seen = withdrawn;
      left = kFlowRestSteps;
    }
    if (left == 0) return true;
    --left;
    return false;
  }
};

// bytes from one body's flow state to the next: a cache line each (16 bytes,
// eight bodies to a line: 322 us per velocity phase of a settled pile of
// 20,000 against 242)
constexpr int kFlowStride = 128;

// The launches reach the states by 32-bit byte offsets behind one buffer
// descriptor, so a batch with room for more bodies than that takes a launch
// per colour. (16.7 million bodies; with few enough contacts and joints to be
// resident only if nearly all of them are in the air.)
constexpr bool flow_reaches(long long bodies) { return bodies * kFlowStride <= INT_MAX; }

}  // namespace b2g
