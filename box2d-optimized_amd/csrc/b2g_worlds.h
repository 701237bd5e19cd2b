// b2g_worlds.h -- a world's whole solve in one workgroup, from the coloured
// contacts to the written-back bodies (b2Island::Solve, src/dynamics/
// b2_island.cpp:253-438, with islands, constraint set-up and write-back).
//
// Each lane keeps its constraints in registers for all iterations of a phase,
// the bodies live in LDS, and a barrier separates the colours: the same
// updates in the same order as a launch per colour, so the results are the
// same bit for bit. Constraint records, colour-sorted slots, island labels and
// marks never reach global memory.
//
// What bounds it: the chain of a workgroup's colours, 0.55-0.65 us each (the
// solve's own dependent arithmetic is 0.35 us, the rest LDS and the barrier),
// a set-up of 25 us (49 with every CU at it), and, in large batches, the
// registers that hold the constraints: 1024 to a CU, one to each of 1024 lanes
// of 128 registers. 256 workgroups of 930 contacts take 108 us, eight
// velocity and three position iterations. With the constraints re-read from
// global memory in every sweep (k_solve_worlds) a colour took 2.1 us: 154 us
// for the largest of 64 small worlds.
//
// Worlds are listed by class on the device (k_colour_init): a class is how many
// worlds of that size fit a workgroup. The workgroup sorts the contacts of all
// its worlds by colour together, so that its waves hold one or two colours
// each, and steps the colours of all its worlds at once. (A launch per class
// left the small classes waiting for each other, 60 us each whatever their
// size.) Worlds of 1025 to 2048 contacts take a workgroup of 512 lanes with
// four constraints to a lane, which spills: 122 us for the largest of 64 worlds
// that still fall, 230 us settled, against 159 and about 270 for the set-up
// launches and k_solve_worlds; all worlds that way cost the smaller ones 25%.
// Worlds past 2048 contacts or 4096 bodies take k_solve_worlds, and those of
// 1025 to 2048 with them where the last step had any (Dev::classes_on).
#pragma once

#include "b2g_kernels.h"

namespace b2g {

// the walk to a body's island root in the finished forest
__device__ __forceinline__ int lds_root(const int* par, int x) {
  for (int p = par[x]; p != x; p = par[x]) x = p;
  return x;
}

constexpr int kGroupMax = class_worlds(0);  // worlds of a workgroup at most
constexpr int kPairThreads = 512;  // lanes of the workgroups that hold 2048 contacts
// Workgroups for n worlds of class c; one of fewer lanes than a full one (a
// launch for one world) holds one.
__device__ __host__ __forceinline__ int class_blocks(int n, int c, bool full) {
  const int per = full ? class_worlds(c) : 1;
  return (n + per - 1) / per;
}
// The fields of a constraint that its updates read, without the repeats of the
// symmetric matrices (K and its inverse: equal off-diagonals, bit for bit).
struct HeldFields {
  float4 v0, v1, v3, v5, q0, q1, bk, nk;  // bk: biases, K.ex.x, K.ey.y; nk: inverse ex.x, ex.y, ey.y, K.ex.y
  __device__ __forceinline__ float4 vc(int k) const {
    switch (k) {
      case 0: return v0;
      case 1: return v1;
      case 3: return v3;
      case 4: return q0;
      case 5: return v5;
      case 6: return q1;
      case 7: return make_float4(bk.x, bk.y, nk.w, nk.w);
      case 8: return make_float4(nk.x, nk.y, nk.y, nk.z);
      default: return make_float4(bk.z, nk.w, nk.w, bk.w);
    }
  }
};
// What a lane holds of a constraint beside them, in two words: places in LDS
// (12 bits each: la, lb, the island's root), whether the solve writes the
// bodies, warm starting, point count, colour (-1 none).
struct HeldIndex {
  unsigned a, b;
  __device__ __forceinline__ int la() const { return (int)(a & 0xfffu); }
  __device__ __forceinline__ int lb() const { return (int)((a >> 12) & 0xfffu); }
  __device__ __forceinline__ bool wa() const { return (a >> 24) & 1u; }
  __device__ __forceinline__ bool wb() const { return (a >> 25) & 1u; }
  __device__ __forceinline__ bool warm() const { return (a >> 26) & 1u; }
  __device__ __forceinline__ int points() const { return (int)((a >> 27) & 3u); }
  __device__ __forceinline__ int root() const { return (int)(b & 0xfffu); }
  __device__ __forceinline__ int turn() const { return (int)((b >> 12) & 0xfffu); }  // of a serial contact
  __device__ __forceinline__ int col() const { return (int)(b >> 24) - 1; }
};
static_assert(kGroupBodies <= 4096 && kGroupSlots <= 4096, "12-bit places");

// Classes [first, last], largest worlds first; NT lanes of K constraints each.
template <int NT, int K>
__global__ void __launch_bounds__(NT, NT / kWave / 4) k_step_worlds(Dev d, int vi, int pi, int rounds_run, int first_cls,
                                                                    int last_cls) {
  constexpr int kBodies = NT * K > kGroupThreads ? kGroupBodies : kGroupBodies / 2;
  __shared__ float4 s_body[kBodies];        // velocities, then positions
  __shared__ int s_par[kBodies];            // union-find forests of the islands
  __shared__ int s_bad[kBodies];            // per island root: 1 + the last iteration that marked it
  __shared__ unsigned s_slot[NT * K];        // by colour: colour << 16 | source slot
  __shared__ int s_hist[kColourSlots], s_off[kColourSlots + 1];
  // the worlds: index, first body, bodies, first solved contact, contacts, colours, serial contacts
  __shared__ int s_w[kGroupMax], s_b0[kGroupMax], s_nb[kGroupMax], s_t0[kGroupMax], s_T[kGroupMax];
  __shared__ unsigned long long s_mask[kGroupMax];
  __shared__ int s_ser[kGroupMax];
  const int tid = (int)threadIdx.x, nt = (int)blockDim.x;
  if (rounds_run && blockIdx.x == 0 && tid == 0) d.cnt[C_ROUND] += rounds_run;
  int total = 0;  // workgroups of all classes, the largest worlds first
  const bool full = nt == NT;
  for (int c = last_cls; c >= first_cls; --c) total += class_blocks(d.cnt[kCntClass + c], c, full);
  for (int i = (int)blockIdx.x; i < total; i += (int)gridDim.x) {
    __syncthreads();  // the last worlds' LDS is done with
    int cls = last_cls, at = i;
    for (; cls > first_cls; --cls) {
      const int n = class_blocks(d.cnt[kCntClass + cls], cls, full);
      if (at < n) break;
      at -= n;
    }
    const int groups = full ? class_worlds(cls) : 1;
    // source slot u of world u / share is its (u % share)-th solved contact
    const int share = nt * K / groups, room = full ? class_bodies(cls) : kBodies;
    const int listed = d.cnt[kCntClass + cls];
    if (tid < groups) {
      const int pick = at * groups + tid;
      const int w = pick < listed ? d.wclass[(size_t)cls * d.nw + pick] : -1;
      const int2 wb = w >= 0 ? d.wbody[w] : make_int2(0, 0);
      const int2 r = w >= 0 ? world_solved(d, w) : make_int2(0, 0);
      s_w[tid] = w;
      s_b0[tid] = wb.x;
      s_nb[tid] = wb.y - wb.x;
      s_t0[tid] = r.x;
      s_T[tid] = r.y - r.x;
      s_mask[tid] = 0ull;
      s_ser[tid] = 0;
    }
    for (int c = tid; c < kColourSlots; c += nt) s_hist[c] = 0;
    __syncthreads();
    // fn(place in LDS, body) for the bodies of the workgroup's worlds
    auto bodies = [&](auto fn) {
      for (int at_b = tid; at_b < groups * room; at_b += nt) {
        const int g = at_b / room, b = at_b - g * room;
        if (b < s_nb[g]) fn(at_b, s_b0[g] + b, g);
      }
    };
    bodies([&](int at_b, int b, int g) {
      s_body[at_b] = d.vel[b];
      s_par[at_b] = at_b - g * room;
      s_bad[at_b] = 0;
    });
    __syncthreads();
    // slots by colour, and the islands
    int col[K], rank[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int u = tid + j * nt, g = min(u / share, groups - 1), t = u - g * share;
      col[j] = -1;
      rank[j] = 0;
      if (t < share && t < s_T[g]) {
        const int k = s_t0[g] + t;
        col[j] = d.ccolour[k];
        if (col[j] < 0) col[j] = kSerialColour;  // unreachable once colouring has finished
        rank[j] = atomicAdd(&s_hist[col[j]], 1);
        if (col[j] < kMaxColours)
          atomicOr(&s_mask[g], 1ull << col[j]);
        else
          atomicAdd(&s_ser[g], 1);
        d.ccol[d.clist[k]] = col[j];
        const int2 bp = d.cbody[k];
        if ((bp.x | bp.y) >= 0) lds_union(s_par + g * room, bp.x - s_b0[g], bp.y - s_b0[g]);
      }
    }
    __syncthreads();
    static_assert(kMaxColours == kWave, "one lane per normal colour");
    if (tid < kWave) {
      const int h = s_hist[tid];
      const int inc = wave_inclusive_scan(h);
      s_off[tid] = inc - h;
      if (tid == kWave - 1) {
        s_off[kSerialColour] = inc;
        s_off[kSerialColour + 1] = inc + s_hist[kSerialColour];
      }
    }
    if (tid < groups && s_w[tid] >= 0) {
      const unsigned long long used = s_mask[tid];
      const int topn = used ? 64 - __clzll((long long)used) : 0;
      const int top = s_ser[tid] ? kColourSlots : topn;
      if (top) atomicMax(&d.cnt[C_NCOLOURS], top);
      if (s_ser[tid]) atomicAdd(&d.cnt[C_SERIAL], s_ser[tid]);
      world_colour_stats(d, s_w[tid], topn);
    }
    unsigned long long mask = 0;  // the colours and the serial contacts of any world here
    int serial = 0;
    for (int g = 0; g < groups; ++g) {
      mask |= s_mask[g];
      serial = max(serial, s_ser[g]);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (col[j] >= 0) s_slot[s_off[col[j]] + rank[j]] = (unsigned)(col[j] << 16 | (tid + j * nt));
    __syncthreads();
    // this lane's constraints
    HeldFields f[K];
    HeldIndex x[K];
    int con[K];
    const int slots = s_off[kSerialColour + 1];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int s = tid + j * nt;
      con[j] = 0;
      x[j] = HeldIndex{0u, 0u};
      if (s < slots) {
        const unsigned e = s_slot[s];
        const int u = (int)(e & 0xffffu), g = min(u / share, groups - 1), t = u - g * share;
        const int c = (int)(e >> 16);
        const int k = s_t0[g] + t, gb = g * room, first = s_b0[g];
        int turn = 0;
        if (c == kSerialColour)  // in contact order, one after the other
          for (int q = 0; q < t; ++q) {
            const int cq = d.ccolour[s_t0[g] + q];
            turn += cq < 0 || cq == kSerialColour ? 1 : 0;
          }
        con[j] = d.clist[k];
        const int2 bp = d.cbody[k];
        const int ia = bp.x >= 0 ? bp.x : ~bp.x, ib = bp.y >= 0 ? bp.y : ~bp.y;
        const int la = gb + ia - first, lb = gb + ib - first;
        const int root = gb + lds_root(s_par + gb, bp.x >= 0 ? ia - first : ib - first);
        const ConFields v = contact_fields(d, con[j], d.cpair[con[j]], ia, ib, s_w[g], d.pos[ia], d.pos[ib],
                                           s_body[la], s_body[lb]);
        f[j] = HeldFields{v.v[0], v.v[1], v.v[3], v.v[5], v.v[4], v.v[6],
                          make_float4(v.v[7].x, v.v[7].y, v.v[9].x, v.v[9].w),
                          make_float4(v.v[8].x, v.v[8].y, v.v[8].w, v.v[9].y)};
        const int flags = as_int(v.v[2].z);
        x[j].a = (unsigned)la | (unsigned)lb << 12 | (writes_body(d, ia) ? 1u << 24 : 0u) |
                 (writes_body(d, ib) ? 1u << 25 : 0u) | (flags & 256 ? 1u << 26 : 0u) | (unsigned)(flags & 3) << 27;
        x[j].b = (unsigned)root | (unsigned)turn << 12 | (unsigned)(c + 1) << 24;
      }
    }
    __syncthreads();  // the set-up read velocities that the sweeps change
    // one colour at a time, then the serial contacts one by one
    auto sweep = [&](auto fn) {
      for (unsigned long long m = mask; m; m &= m - 1) {
        const int c = __ffsll((long long)m) - 1;
#pragma unroll
        for (int j = 0; j < K; ++j)
          if (x[j].col() == c) fn(j);
        __syncthreads();
      }
      for (int q = 0; q < serial; ++q) {
#pragma unroll
        for (int j = 0; j < K; ++j)
          if (x[j].col() == kSerialColour && x[j].turn() == q) fn(j);
        __syncthreads();
      }
    };
    auto bodies_of = [&](int j) { return vel_pair(s_body[x[j].la()], s_body[x[j].lb()]); };
    auto put = [&](int j, const VelPair& u) {
      if (x[j].wa()) s_body[x[j].la()] = make_float4(u.vA.x, u.vA.y, u.wA, 0.0f);
      if (x[j].wb()) s_body[x[j].lb()] = make_float4(u.vB.x, u.vB.y, u.wB, 0.0f);
    };
    sweep([&](int j) {
      if (!x[j].warm()) return;
      VelPair u = bodies_of(j);
      warm_start_core(f[j], x[j].points(), u);
      put(j, u);
    });
    for (int it = 0; it < vi; ++it) {
      sweep([&](int j) {
        VelPair u = bodies_of(j);
        contact_velocity_core(f[j], x[j].points(), u, f[j].q0, f[j].q1);
        put(j, u);
      });
    }
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (x[j].col() >= 0) store_contact_impulses(d, con[j], x[j].points(), f[j].q0, f[j].q1);
    bodies([&](int at_b, int b, int g) {
      float4 p = d.pos[b];
      if (d.btype[b] != kStaticBody) {
        float4 v = s_body[at_b];
        p = integrated_position(d.wpar[s_w[g]].z, p, v);
        d.vel[b] = v;
      }
      s_body[at_b] = p;
    });
    // the position phase's fields (the manifold and the masses stand)
    float4 q[K][5];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (x[j].col() < 0) continue;
      const float4* mp = d.cman + 4 * (size_t)con[j];
      const float4 m0 = mp[0], m1 = mp[1], m2 = mp[2], m3 = mp[3];
      const int2 pr = d.cpair[con[j]];
      const float4 pa = d.prop[d.shdr[pr.x].y], pb = d.prop[d.shdr[pr.y].y];
      q[j][0] = make_float4(m2.z, m2.w, m2.x, m2.y);
      q[j][1] = make_float4(m0.x, m0.y, m1.x, m1.y);
      q[j][2] = make_float4(pa.z, pa.w, pb.z, pb.w);
      q[j][3] = make_float4(pa.x, pb.x, pa.y, pb.y);
      q[j][4] = make_float4(d.geo[9 * (size_t)pr.x].x, d.geo[9 * (size_t)pr.y].x, as_float(as_int(m3.z) & 0xff),
                            as_float((as_int(m3.z) >> 8) & 0xff));
    }
    __syncthreads();
    bool through[K];  // the island is: no contact separated too far in the iteration before (island_done)
#pragma unroll
    for (int j = 0; j < K; ++j) through[j] = false;
    for (int it = 0; it < pi; ++it) {
      if (it > 0) {
        int left = 0;
#pragma unroll
        for (int j = 0; j < K; ++j) {
          through[j] = through[j] || s_bad[x[j].root()] != it;
          left |= x[j].col() >= 0 && !through[j] ? 1 : 0;
        }
        // (read before this iteration marks); no island left: the rest would change nothing
        if (__syncthreads_or(left) == 0) break;
      }
      sweep([&](int j) {
        if (through[j]) return;
        PosPair u = pos_pair(s_body[x[j].la()], s_body[x[j].lb()]);
        const float m = contact_position_core(q[j][0], q[j][1], q[j][2], q[j][3], q[j][4], u);
        if (x[j].wa()) s_body[x[j].la()] = make_float4(u.cA.x, u.cA.y, u.aA, 0.0f);
        if (x[j].wb()) s_body[x[j].lb()] = make_float4(u.cB.x, u.cB.y, u.aB, 0.0f);
        if (separation_bad(m)) s_bad[x[j].root()] = it + 1;
      });
    }
    __syncthreads();
    // write back: SynchronizeTransform and ClearForces
    bodies([&](int at_b, int b, int) {
      if (d.btype[b] != kStaticBody) {
        const float4 p = s_body[at_b], pr = d.prop[b];
        const rot2 r = rot_of(p.z);
        const vec2 c = mk(p.x, p.y) - mul(r, mk(pr.z, pr.w));
        d.pos[b] = p;
        d.xf[b] = make_float4(c.x, c.y, r.s, r.c);
      }
      d.force[b] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    });
  }
}

// Constraint records and island states of the worlds of `list` (slots and
// labels are ready): blockIdx.y shares a world's slots out.
__global__ void __launch_bounds__(kBlock) k_worlds_init(Dev d, const int* list) {
  const int* off = d.wcol + list[blockIdx.x] * (kColourSlots + 1);
  const int n = d.cnt[C_CONS];
  for (int s = off[0] + (int)(blockIdx.y * blockDim.x + threadIdx.x); s < off[kColourSlots];
       s += (int)(gridDim.y * blockDim.x)) {
    contact_init(d, s);
    island_assign(d, n, s);
  }
}

}  // namespace b2g
