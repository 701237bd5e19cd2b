// b2g_flow_rule.h -- when a step's sweeps are ordered by data (b2g_flow.h).
// Host code only, without a device header: the CPU tests compile it by itself.
#pragma once

#include <climits>

namespace b2g {

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
