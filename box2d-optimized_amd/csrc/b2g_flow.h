// b2g_flow.h -- the colour sweeps of a step as two launches, ordered by data.
//
// The colours give every body a fixed sequence of updates: its constraints in
// colour order, once per iteration. One launch per colour orders them by
// kernel boundaries, and on a pile that is a hundred launches of 4 us each.
// Here every lane keeps one constraint in registers for all iterations of the
// phase, and bodies carry their update count beside their state (flow_pack):
// a constraint waits until each of its dynamic bodies has had exactly the
// updates that precede it, solves, and stores the body with the count plus
// one. Each body thus sees the same updates in the same order as with one
// launch per colour, and the results are the same bit for bit.
//
// What bounds it: the longest chain of updates, about (iterations + 1) x (the
// most constraints of a body), times one hop. A hop is a store that another
// CU's poll sees (0.47 us within an XCD, 0.58 us across, measured with a ring
// of 256 workgroups) plus the solve's own dependent arithmetic (0.3-0.4 us).
// A launch per colour costs 4.1 us on the device and 2.4-3 us on the host.
//
// Forward progress. Body states travel through agent-scope atomics only, so
// no cache needs flushing, but every workgroup must be resident. Each counts
// itself in (flow_enter); when all have, the phase goes. If some have not been
// placed within `wait` clock ticks (the GPU is busy with other work), one
// workgroup withdraws the launch: the others leave, and it sweeps the colours
// by itself, with barriers. Go and withdrawal are one compare-and-swap, so
// exactly one happens, before any constraint is touched. Withdrawals are
// counted, and the host lets steps rest from these launches after one
// (FlowRest).
#pragma once

#include "b2g_kernels.h"

namespace b2g {

static_assert(kFlowLanes == kWave);
// words of Dev::flow_ctl: the velocity launch's (arrivals, go), the position
// launch's, then the position launch's barrier counts, one per iteration
constexpr int kFlowVel = 0, kFlowPos = 2, kFlowBar = 4;
constexpr int kFlowMaxPosIters = kFlowCtl - kFlowBar;
enum FlowGo : int { kFlowWait = 0, kFlowRun = 1, kFlowWithdrawn = 2 };
constexpr long long kFlowEnterTicks = 100000;       // 1 ms of the 100 MHz clock
// Polls of a wait in which nothing comes, one memory round trip (0.5 us) each,
// after which a count is taken to be broken: counted from the last progress,
// and in polls rather than by the clock, so that neither a long phase nor a
// preempted queue runs into it.
constexpr int kFlowStallPolls = 1 << 22;          // a constraint: two seconds
constexpr int kFlowMeetPolls = 2 * kFlowStallPolls;  // a meeting: past any constraint's
constexpr int kFlowStalled = 1 << 20;  // added to a meeting's count: a constraint has stalled, all leave

__device__ __forceinline__ int flow_load(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int flow_swap_go(int* go, int to) {  // the value that stands
  int expected = kFlowWait;
  __hip_atomic_compare_exchange_strong(go, &expected, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return expected == kFlowWait ? to : expected;
}
// thread 0 of every workgroup, once, before its own set-up loads
__device__ __forceinline__ void flow_count_in(int* ctl, int blocks) {
  if (__hip_atomic_fetch_add(ctl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == blocks)
    flow_swap_go(ctl + 1, kFlowRun);
}
// All threads, after the set-up loads: whether the phase runs. `sole` is set
// in the workgroup that withdrew the launch and sweeps the colours alone.
__device__ __forceinline__ bool flow_enter(int* ctl, long long wait, bool* sole) {
  __shared__ int s_go;
  if (threadIdx.x == 0) {
    const long long t0 = wall_clock64();
    int go = wait < 0 ? kFlowWait : flow_load(ctl + 1), mine = 0;
    // (the clock is read now and then: hundreds of waves reading it in every
    // turn of a wait cost tens of microseconds)
    for (unsigned turn = 0; go == kFlowWait; ++turn) {
      if ((wait < 0 || (turn & 255u) == 255u) && wall_clock64() - t0 > wait) {
        int expected = kFlowWait;
        mine = __hip_atomic_compare_exchange_strong(ctl + 1, &expected, (int)kFlowWithdrawn, __ATOMIC_RELAXED,
                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                   ? 4
                   : 0;
        go = mine ? kFlowWithdrawn : expected;
      } else {
        go = flow_load(ctl + 1);
      }
    }
    s_go = go | mine;
  }
  __syncthreads();
  const int go = s_go;
  *sole = (go & 4) != 0;
  return (go & 3) == kFlowRun;
}

// The bodies' states (Dev::fvel or Dev::fpos) behind a buffer descriptor: its
// loads take a cache policy, and one that goes past the XCD's own L2. (Sizes
// and offsets are 32-bit: flow_reaches bounds the bodies.)
typedef unsigned flow_u4 __attribute__((ext_vector_type(4)));
struct FlowStates {
  __amdgpu_buffer_rsrc_t rsrc;
};
__device__ __forceinline__ FlowStates flow_states(unsigned long long* words, int bodies) {
  return FlowStates{__builtin_amdgcn_make_buffer_rsrc(words, 0, kFlowStride * bodies, 0x00020000)};
}
constexpr int kFlowPolicy = 16;  // sc1: agent scope
// A body of a lane's constraint and which count to wait for.
struct FlowBody {
  int body;             // < 0: not dynamic, its state is the one loaded
  unsigned want, last;  // count awaited, and the one this lane last stored (16 bits each)
  __device__ __forceinline__ bool waits() const { return body >= 0 && want != last; }
};
// the state words of a body
__device__ __forceinline__ flow_u4 flow_look(const FlowStates& f, int body) {
  return __builtin_amdgcn_raw_buffer_load_b128(f.rsrc, kFlowStride * body, 0, kFlowPolicy);
}
// Lands the state in s when its count is the awaited one (in both words).
__device__ __forceinline__ bool flow_land(flow_u4 w, const FlowBody& b, float* s) {
  if ((w.y >> 16) != b.want || (w.w >> 16) != b.want) return false;
  s[0] = uint_as_float(w.x);
  s[1] = uint_as_float(w.z);
  s[2] = uint_as_float((w.y << 16) | (w.w & 0xffffu));
  return true;
}
__device__ __forceinline__ void flow_post(const FlowStates& f, FlowBody& b, float x, float y, float z) {
  b.last = (b.want + 1) & 0xffffu;
  unsigned long long w[2];
  flow_pack(x, y, z, b.last, w);
  const flow_u4 v = {(unsigned)w[0], (unsigned)(w[0] >> 32), (unsigned)w[1], (unsigned)(w[1] >> 32)};
  __builtin_amdgcn_raw_buffer_store_b128(v, f.rsrc, kFlowStride * b.body, 0, kFlowPolicy);
}

// least key of the wave's active lanes (INT_MAX: none is)
__device__ __forceinline__ int flow_least(bool active, int key) {
  int m = active ? key : INT_MAX;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = min(m, __shfl_xor(m, off, kWave));
  return m;
}

// The lanes of a wave, each with its own constraint, until all are through.
// `key`: the lane's place in the order of the updates (iteration, then
// colour); lanes of the wave's least key go together, once the bodies of all
// of them have landed. (Going lane by lane measured 2.5 times slower on a
// 20,000-body pile: the lanes drift apart, and every pass over the solve, 0.4
// us of one wave's issue slots, then serves one or two of them.) `step`
// solves and posts, moves the lane on to its next wants and key, and says
// whether it has more to do. The update of the least key of all waves never
// waits, so some wave always goes on. False: the wave stalled (a broken count)
// and gave up.
template <class Step>
__device__ __forceinline__ bool flow_run(const Dev& d, const FlowStates& f, bool active, int& key, FlowBody& A,
                                         FlowBody& B, float* sa, float* sb, Step step) {
  bool wa = A.waits(), wb = B.waits();
  int least = flow_least(active, key);
  const bool mixed = __ballot(active && key != least) != 0;  // most waves hold one colour
  for (int idle = 0; least != INT_MAX;) {
    const bool mine = active && (!mixed || key == least);
    if (__ballot(mine && (wa || wb)) != 0) {
      if (mine && (wa || wb)) {
        asm volatile("" ::: "memory");  // (each pass loads afresh)
        // both in flight; where one side is there, its load repeats the other's
        const flow_u4 a = flow_look(f, wa ? A.body : B.body), b = flow_look(f, wb ? B.body : A.body);
        if (wa && flow_land(a, A, sa)) wa = false;
        if (wb && flow_land(b, B, sb)) wb = false;
      }
      if (++idle > kFlowStallPolls) {
        if (active) atomicOr(&d.cnt[C_STATUS], S_FLOW_STALL);
        return false;
      }
    } else {
      idle = 0;
      if (mine) {
        active = step();
        wa = A.waits();
        wb = B.waits();
      }
      if (mixed)
        least = flow_least(active, key);
      else if (__ballot(active) == 0)
        least = INT_MAX;
    }
  }
  return true;
}

// the lane's constraint: `per` to a wave, in its first lanes (-1: none)
__device__ __forceinline__ int flow_slot(int block, int per) {
  return lane_id() < per ? (block * kFlowWaves + wave_id()) * per + lane_id() : -1;
}
// a body's contacts (its colours) and joints
__device__ __forceinline__ int flow_contacts(const Dev& d, int b) { return __popcll(d.bmask[b]); }

// ---------------------------------------------------------------------------
// Velocity phase, as b2Island::Solve orders it (src/dynamics/b2_island.cpp:
// 300-339): the joints' set-up and warm start (the contacts' is k_warm_gather's,
// a third of the time of a sweep), then the iterations, joints before contacts.
// The last update of a body lands in Dev::vel, and the impulses in their
// arrays.
// Measured over steps 361-465 of a pile of 20,000 (34,600 contacts, 15
// colours): 241 us, against 371 us in 64 launches of k_contact_velocity and
// k_sweep_tail plus the gaps between them; its last colours' chain, 14 bodies'
// updates an iteration at 1.7-2.1 us, bounds it.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void flow_velocity_contact(const Dev& d, int s, bool valid, int vi) {
  const FlowStates f = flow_states(d.fvel, d.nb);
  VelocityRegs r{};
  FlowBody A{-1, 0u, 0u}, B{-1, 0u, 0u};
  float sa[3] = {}, sb[3] = {};
  int nA = 0, nB = 0, jA = 0, jB = 0, rA = 0, rB = 0, ia = 0, ib = 0, count = 0;
  int key = 0;
  if (valid) {
    r = load_velocity_regs(d, s);
    ia = as_int(r.v[2].x);
    ib = as_int(r.v[2].y);
    count = as_int(r.v[2].z) & 0xff;
    key = d.ccol[as_int(r.v[2].w)];
    const unsigned long long below = (1ull << key) - 1ull;
    const float4 va = d.vel[ia], vb = d.vel[ib];  // a body that is not dynamic keeps these
    sa[0] = va.x; sa[1] = va.y; sa[2] = va.z;
    sb[0] = vb.x; sb[1] = vb.y; sb[2] = vb.z;
    if (is_dyn(d, ia)) {
      const unsigned long long m = d.bmask[ia];
      nA = __popcll(m);
      rA = __popcll(m & below);
      jA = d.nj ? d.bjdeg[ia] : 0;
      A.body = ia;
    }
    if (is_dyn(d, ib)) {
      const unsigned long long m = d.bmask[ib];
      nB = __popcll(m);
      rB = __popcll(m & below);
      jB = d.nj ? d.bjdeg[ib] : 0;
      B.body = ib;
    }
  }
  A.want = (unsigned)(2 * jA + rA);
  B.want = (unsigned)(2 * jB + rB);
  A.last = B.last = 0xffffffffu;  // no count: the first states are always polled
  int k = 1;
  const bool lastA = rA + 1 == nA, lastB = rB + 1 == nB;  // the body's last update of an iteration
  // a sleeping island's constraints (no points) take no part, all of them
  flow_run(d, f, valid && count > 0 && vi > 0, key, A, B, sa, sb, [&]() {
    VelPair u{mk(sa[0], sa[1]), mk(sb[0], sb[1]), sa[2], sb[2]};
    contact_velocity_core(r, count, u, r.v[4], r.v[6]);
    const bool end = k == vi;
    if (A.body >= 0) {
      sa[0] = u.vA.x; sa[1] = u.vA.y; sa[2] = u.wA;
      if (!end || !lastA) flow_post(f, A, u.vA.x, u.vA.y, u.wA);
      if (end && lastA) d.vel[ia] = make_float4(u.vA.x, u.vA.y, u.wA, 0.0f);
    }
    if (B.body >= 0) {
      sb[0] = u.vB.x; sb[1] = u.vB.y; sb[2] = u.wB;
      if (!end || !lastB) flow_post(f, B, u.vB.x, u.vB.y, u.wB);
      if (end && lastB) d.vel[ib] = make_float4(u.vB.x, u.vB.y, u.wB, 0.0f);
    }
    if (end) {
      put_impulses_global(d, s, r.v[4], r.v[6], count);
      return false;
    }
    ++k;
    key += kMaxColours;
    A.want = (unsigned)(2 * jA + (k - 1) * (nA + jA) + rA) & 0xffffu;
    B.want = (unsigned)(2 * jB + (k - 1) * (nB + jB) + rB) & 0xffffu;
    return true;
  });
}

__device__ __forceinline__ void flow_velocity_joint(const Dev& d, int q, bool valid, int vi) {
  const FlowStates f = flow_states(d.fvel, d.nb);
  Joint j{};
  JointSolve js{};
  FlowBody A{-1, 0u, 0u}, B{-1, 0u, 0u};
  float sa[3] = {}, sb[3] = {};
  float4 pa{}, pb{};
  float aA = 0.0f, aB = 0.0f, h = 0.0f, ratio = 0.0f;
  int nA = 0, nB = 0, jA = 0, jB = 0, ji = 0;
  int2 rank = make_int2(0, 0);
  int key = 0;
  bool warm = false;
  valid = valid && d.jisland[q] >= 0;  // (not of a world or island that sits out the step)
  if (valid) {
    ji = d.jorder[q];
    j = d.joints[ji];
    const int2 place = d.jplace[q];
    key = place.y;
    rank = make_int2(place.x & 0xff, place.x >> 8);
    const float4 wp = d.wpar[j.world];
    h = wp.z;
    ratio = wp.w;
    warm = (d.wflag[j.world] & 1) != 0;
    pa = d.prop[j.a];
    pb = d.prop[j.b];
    aA = d.pos[j.a].z;
    aB = d.pos[j.b].z;
    const float4 va = d.vel[j.a], vb = d.vel[j.b];
    sa[0] = va.x; sa[1] = va.y; sa[2] = va.z;
    sb[0] = vb.x; sb[1] = vb.y; sb[2] = vb.z;
    if (is_dyn(d, j.a)) {
      nA = flow_contacts(d, j.a);
      jA = d.bjdeg[j.a];
      A.body = j.a;
    }
    if (is_dyn(d, j.b)) {
      nB = flow_contacts(d, j.b);
      jB = d.bjdeg[j.b];
      B.body = j.b;
    }
  }
  A.want = (unsigned)rank.x;
  B.want = (unsigned)rank.y;
  A.last = B.last = 0xffffffffu;
  int k = 0;
  flow_run(d, f, valid, key, A, B, sa, sb, [&]() {
    VelPair u{mk(sa[0], sa[1]), mk(sb[0], sb[1]), sa[2], sb[2]};
    if (k > 0)
      joint_velocity_core(j, js, h, u);
    else
      joint_init_core(j, js, pa, pb, aA, aB, warm, ratio, u);
    const bool end = k == vi;
    if (A.body >= 0) {
      sa[0] = u.vA.x; sa[1] = u.vA.y; sa[2] = u.wA;
      flow_post(f, A, u.vA.x, u.vA.y, u.wA);
      // the body's last update, when no contact follows
      if (end && (nA == 0 || vi == 0) && rank.x + 1 == jA) d.vel[j.a] = make_float4(u.vA.x, u.vA.y, u.wA, 0.0f);
    }
    if (B.body >= 0) {
      sb[0] = u.vB.x; sb[1] = u.vB.y; sb[2] = u.wB;
      flow_post(f, B, u.vB.x, u.vB.y, u.wB);
      if (end && (nB == 0 || vi == 0) && rank.y + 1 == jB) d.vel[j.b] = make_float4(u.vB.x, u.vB.y, u.wB, 0.0f);
    }
    if (end) {
      d.joints[ji] = j;
      d.jsol[q] = js;
      return false;
    }
    ++k;
    key += kMaxColours;
    A.want = (unsigned)(jA + (k - 1) * (nA + jA) + rank.x) & 0xffffu;
    B.want = (unsigned)(jB + (k - 1) * (nB + jB) + rank.y) & 0xffffu;
    return true;
  });
}

// one workgroup, the same updates colour by colour
__device__ __forceinline__ void flow_velocity_alone(const Dev& d, int vi) {
  const int tid = (int)threadIdx.x, nt = (int)blockDim.x;
  auto contacts = [&](auto fn) {
    for (int c = 0; c < kMaxColours; ++c) {
      const int lo = d.col_off[c], hi = d.col_off[c + 1];
      if (hi <= lo) continue;
      for (int s = lo + tid; s < hi; s += nt) fn(s);
      __syncthreads();
    }
  };
  auto joints = [&](auto fn) {
    for (int c = 0; c < d.njcol; ++c) {
      for (int q = d.jcol_off[c] + tid; q < d.jcol_off[c + 1]; q += nt) fn(q);
      __syncthreads();
    }
  };
  joints([&](int q) { joint_init(d, q); });
  for (int it = 0; it < vi; ++it) {
    joints([&](int q) { joint_velocity(d, q); });
    contacts([&](int s) { contact_velocity(d, s); });
  }
}

// The first `jblocks` workgroups take the joints, the others the contacts in
// slot (colour) order: the lanes of a wave then wait for about the same
// place in the bodies' sequences.
__global__ void __launch_bounds__(kFlowThreads, 4) k_flow_velocity(Dev d, int cons, int jblocks, int per, int vi,
                                                                   long long wait) {
  int* ctl = d.flow_ctl + kFlowVel;
  if (threadIdx.x == 0) flow_count_in(ctl, (int)gridDim.x + (wait < 0 ? 1 : 0));  // (wait < 0: never complete)
  bool sole;
  if (!flow_enter(ctl, wait, &sole)) {
    if (sole) {
      if (threadIdx.x == 0) ++d.cnt[kCntWithdrawn];
      flow_velocity_alone(d, vi);
    }
    return;
  }
  const bool joints = (int)blockIdx.x < jblocks;
  const int at = flow_slot((int)blockIdx.x - (joints ? 0 : jblocks), per);
  if (joints)
    flow_velocity_joint(d, at, at >= 0 && at < d.nj, vi);
  else
    flow_velocity_contact(d, at, at >= 0 && at < cons, vi);
}

// ---------------------------------------------------------------------------
// Position phase: iterations of contacts, then joints, with the per-island
// early exit (b2_island.cpp:387-409). An iteration reads the island marks of
// the one before, so the workgroups meet between iterations (flow_meet); the
// bodies' update counts run on, so nothing else does.
// Measured on the same pile: 150 us for three iterations, against 214 us in
// 24 launches of k_contact_position and k_sweep_tail plus their gaps.
// ---------------------------------------------------------------------------
// All workgroups of the launch (they are resident): each marks its islands
// with agent-scope stores, waits for them to be done, and counts itself in.
// `ok`: this wave did not stall; false where any of the launch did, in every
// workgroup alike.
__device__ __forceinline__ bool flow_meet(const Dev& d, int* count, int blocks, bool ok) {
  __shared__ int s_met;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);  // this wave's stores have reached the memory side
  const bool stalled = __syncthreads_or(!ok) != 0;
  if (threadIdx.x == 0) {
    __hip_atomic_fetch_add(count, stalled ? kFlowStalled : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int met = flow_load(count);
    for (int polls = 0; met < blocks; met = flow_load(count)) {
      if (++polls > kFlowMeetPolls) {
        atomicOr(&d.cnt[C_STATUS], S_FLOW_STALL);
        met = kFlowStalled;
        break;
      }
    }
    s_met = met;
  }
  __syncthreads();
  return s_met < kFlowStalled;
}

// Whether the island is through before iteration `it` (island_done, from the
// marks as other CUs stored them), and its marks of the next iterations
// cleared where they are used again (island_reset clears the first three).
__device__ __forceinline__ bool flow_island_done(const Dev& d, int isl, int it, int pi) {
  if (it == 0) return false;
  const size_t prev = island_slot(d, isl, it - 1);
  const unsigned bad = __hip_atomic_load(d.sepbad + prev, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int jok = flow_load(d.jok + prev);
  if (bad == 0u && jok != 0) {
    d.solved[isl] = 1;
    return true;
  }
  if (it >= 2 && it + 1 < pi) {
    const size_t nxt = island_slot(d, isl, it + 1);
    if (__hip_atomic_load(d.sepbad + nxt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)
      __hip_atomic_store(d.sepbad + nxt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (flow_load(d.jok + nxt) != 1) __hip_atomic_store(d.jok + nxt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  return false;
}

__device__ __forceinline__ void flow_position_contact(const Dev& d, int s, bool valid, int pi, int* bar) {
  const FlowStates f = flow_states(d.fpos, d.nb);
  PositionRegs r{};
  FlowBody A{-1, 0u, 0u}, B{-1, 0u, 0u};
  float sa[3] = {}, sb[3] = {};
  int nA = 0, nB = 0, jA = 0, jB = 0, rA = 0, rB = 0, ia = 0, ib = 0, key = 0;
  if (valid) {
    r = load_position_regs(d, s);
    ia = as_int(r.v2.x);
    ib = as_int(r.v2.y);
    key = d.ccol[as_int(r.v2.w)];
    const unsigned long long below = (1ull << key) - 1ull;
    const float4 ca = d.pos[ia], cb = d.pos[ib];
    sa[0] = ca.x; sa[1] = ca.y; sa[2] = ca.z;
    sb[0] = cb.x; sb[1] = cb.y; sb[2] = cb.z;
    if (is_dyn(d, ia)) {
      const unsigned long long m = d.bmask[ia];
      nA = __popcll(m);
      rA = __popcll(m & below);
      jA = d.nj ? d.bjdeg[ia] : 0;
      A.body = ia;
    }
    if (is_dyn(d, ib)) {
      const unsigned long long m = d.bmask[ib];
      nB = __popcll(m);
      rB = __popcll(m & below);
      jB = d.nj ? d.bjdeg[ib] : 0;
      B.body = ib;
    }
    valid = as_int(r.p[4].w) != 0;  // else a constraint of a sleeping island
  }
  A.last = B.last = 0xffffffffu;
  for (int it = 0; it < pi; ++it) {
    if (valid && flow_island_done(d, r.isl, it, pi)) valid = false;
    A.want = (unsigned)(it * (nA + jA) + rA) & 0xffffu;
    B.want = (unsigned)(it * (nB + jB) + rB) & 0xffffu;
    bool bad = false;
    const bool through = flow_run(d, f, valid, key, A, B, sa, sb, [&]() {
      PosPair u{mk(sa[0], sa[1]), mk(sb[0], sb[1]), sa[2], sb[2]};
      const float m = contact_position_core(r.p[0], r.p[1], r.p[2], r.p[3], r.p[4], u);
      bad = separation_bad(m);
      if (A.body >= 0) {
        sa[0] = u.cA.x; sa[1] = u.cA.y; sa[2] = u.aA;
        flow_post(f, A, u.cA.x, u.cA.y, u.aA);
        if (rA + 1 == nA && jA == 0) d.pos[ia] = make_float4(u.cA.x, u.cA.y, u.aA, 0.0f);
      }
      if (B.body >= 0) {
        sb[0] = u.cB.x; sb[1] = u.cB.y; sb[2] = u.aB;
        flow_post(f, B, u.cB.x, u.cB.y, u.aB);
        if (rB + 1 == nB && jB == 0) d.pos[ib] = make_float4(u.cB.x, u.cB.y, u.aB, 0.0f);
      }
      return false;
    });
    // (marks of one island by a thousand waves queue at its address for 50 us:
    // a wave that finds it marked stores nothing)
    bad = bad && __hip_atomic_load(d.sepbad + island_slot(d, r.isl, it), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT) == 0u;
    mark_island_sep(d, it, valid ? r.isl : 0, bad, -1.0f);
    if (it + 1 < pi && !flow_meet(d, bar + it, (int)gridDim.x, through)) return;
  }
}

__device__ __forceinline__ void flow_position_joint(const Dev& d, int q, bool valid, int pi, int* bar) {
  const FlowStates f = flow_states(d.fpos, d.nb);
  Joint j{};
  JointSolve js{};
  FlowBody A{-1, 0u, 0u}, B{-1, 0u, 0u};
  float sa[3] = {}, sb[3] = {};
  int nA = 0, nB = 0, jA = 0, jB = 0, isl = -1, key = 0;
  int2 rank = make_int2(0, 0);
  if (valid) {
    isl = d.jisland[q];
    valid = isl >= 0;
  }
  if (valid) {
    j = d.joints[d.jorder[q]];
    js = d.jsol[q];
    const int2 place = d.jplace[q];
    key = place.y;
    rank = make_int2(place.x & 0xff, place.x >> 8);
    const float4 ca = d.pos[j.a], cb = d.pos[j.b];
    sa[0] = ca.x; sa[1] = ca.y; sa[2] = ca.z;
    sb[0] = cb.x; sb[1] = cb.y; sb[2] = cb.z;
    if (is_dyn(d, j.a)) {
      nA = flow_contacts(d, j.a);
      jA = d.bjdeg[j.a];
      A.body = j.a;
    }
    if (is_dyn(d, j.b)) {
      nB = flow_contacts(d, j.b);
      jB = d.bjdeg[j.b];
      B.body = j.b;
    }
  }
  A.last = B.last = 0xffffffffu;
  for (int it = 0; it < pi; ++it) {
    if (valid && flow_island_done(d, isl, it, pi)) valid = false;
    A.want = (unsigned)(it * (nA + jA) + nA + rank.x) & 0xffffu;
    B.want = (unsigned)(it * (nB + jB) + nB + rank.y) & 0xffffu;
    const bool through = flow_run(d, f, valid, key, A, B, sa, sb, [&]() {
      PosPair u{mk(sa[0], sa[1]), mk(sb[0], sb[1]), sa[2], sb[2]};
      const bool ok = joint_position_core(j, js, u);
      if (A.body >= 0) {
        sa[0] = u.cA.x; sa[1] = u.cA.y; sa[2] = u.aA;
        flow_post(f, A, u.cA.x, u.cA.y, u.aA);
        if (rank.x + 1 == jA) d.pos[j.a] = make_float4(u.cA.x, u.cA.y, u.aA, 0.0f);
      }
      if (B.body >= 0) {
        sb[0] = u.cB.x; sb[1] = u.cB.y; sb[2] = u.aB;
        flow_post(f, B, u.cB.x, u.cB.y, u.aB);
        if (rank.y + 1 == jB) d.pos[j.b] = make_float4(u.cB.x, u.cB.y, u.aB, 0.0f);
      }
      if (!ok) __hip_atomic_store(d.jok + island_slot(d, isl, it), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    });
    if (it + 1 < pi && !flow_meet(d, bar + it, (int)gridDim.x, through)) return;
  }
}

__device__ __forceinline__ void flow_position_alone(const Dev& d, int pi) {
  const int tid = (int)threadIdx.x, nt = (int)blockDim.x;
  for (int it = 0; it < pi; ++it) {
    for (int c = 0; c < kMaxColours; ++c) {
      const int lo = d.col_off[c], hi = d.col_off[c + 1];
      if (hi <= lo) continue;
      for (int base = lo; base < hi; base += nt) {
        const int s = base + tid;
        const bool valid = s < hi;
        const int isl = valid ? d.cisland[s] : 0;
        const float m = valid ? contact_position(d, s, isl, it) : 0.0f;
        mark_island_sep(d, it, isl, valid, m);
      }
      __syncthreads();
    }
    for (int c = 0; c < d.njcol; ++c) {
      for (int q = d.jcol_off[c] + tid; q < d.jcol_off[c + 1]; q += nt) joint_position(d, q, it);
      __syncthreads();
    }
    __threadfence();  // the next iteration reads the marks
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kFlowThreads, 4) k_flow_position(Dev d, int cons, int jblocks, int per, int pi,
                                                                   long long wait) {
  int* ctl = d.flow_ctl + kFlowPos;
  if (threadIdx.x == 0) flow_count_in(ctl, (int)gridDim.x + (wait < 0 ? 1 : 0));
  bool sole;
  if (!flow_enter(ctl, wait, &sole)) {
    if (sole) {
      if (threadIdx.x == 0) ++d.cnt[kCntWithdrawn];
      flow_position_alone(d, pi);
    }
    return;
  }
  int* bar = d.flow_ctl + kFlowBar;
  const bool joints = (int)blockIdx.x < jblocks;
  const int at = flow_slot((int)blockIdx.x - (joints ? 0 : jblocks), per);
  if (joints)
    flow_position_joint(d, at, at >= 0 && at < d.nj, pi, bar);
  else
    flow_position_contact(d, at, at >= 0 && at < cons, pi, bar);
}

}  // namespace b2g
