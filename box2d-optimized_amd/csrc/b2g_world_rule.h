// b2g_world_rule.h -- the workgroup size of the captured per-world solve. Host
// code only, without a device header: the CPU tests compile it by itself.
#pragma once

namespace b2g {

// Lanes of the workgroups that solve a captured step's worlds (k_solve_worlds,
// bodies staged in LDS; worlds past 1024 bodies have 1024 lanes in a launch of
// their own wherever this is less). A wide workgroup shortens each colour of a
// world, a narrow one lets more worlds run at once: a CU holds 20 wavefronts
// of the solve. So the widest that leaves every world resident: one workgroup
// a CU at 1024 lanes, two and a half at 512, and at 256 twice the five that
// are resident, because many worlds are through early; 128 past that.
// ms of a replayed step at 64 / 128 / 256 / 512 / 1024 lanes on 256 CUs,
// worlds of 100 bodies in the median, settled:
//     50 worlds  0.75 / 0.57 / 0.47 / 0.44 / 0.44
//    200 worlds  1.04 / 0.77 / 0.63 / 0.55 / 0.49
//    300 worlds  0.98 / 0.73 / 0.59 / 0.52 / 0.51  (falling 0.71 / 0.55 / 0.49 / 0.48 / 0.53)
//    500 worlds  1.14 / 0.87 / 0.71 / 0.63 / 0.66  (falling 0.79 / 0.63 / 0.56 / 0.57 / 0.63)
//   1000 worlds  1.28 / 1.00 / 0.91 / 0.91 / 1.12  (falling 0.91 / 0.74 / 0.68 / 0.79 / 1.01)
//   2500 worlds  1.98 / 1.65 / 1.55 / 1.92 / 2.57  (falling 1.33 / 1.17 / 1.21 / 1.64 / 2.31)
//   4096 worlds  2.56 / 2.21 / 2.25 / 2.96 / 4.09  (falling 1.72 / 1.62 / 1.86 / 2.57 / 3.68)
constexpr int captured_world_lanes(int worlds, int compute_units) {
  return worlds <= compute_units ? 1024 : 2 * worlds <= 5 * compute_units ? 512 : worlds <= 10 * compute_units ? 256 : 128;
}

}  // namespace b2g
