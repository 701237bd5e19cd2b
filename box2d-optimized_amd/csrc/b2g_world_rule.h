// b2g_world_rule.h -- rules of the per-world solves' launches. Host code only,
// without a device header: the CPU tests compile it by itself.
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
  return worlds <= compute_units            ? 1024
         : 2LL * worlds <= 5LL * compute_units ? 512
         : worlds <= 10LL * compute_units      ? 256
                                               : 128;
}

// Whether the worlds of the last but one class (1025 to 2048 contacts) join
// the launch of the worlds past the classes in an eager step, going by the
// last step's counts: `worlds` of both, `past` of them past the classes. A
// world past them takes k_solve_worlds for longer than a smaller one does, so
// beside one, and with a CU for each, the class costs nothing there, where its
// own launch (k_step_worlds, 512 lanes) would queue behind it. With more
// worlds than CUs the launch is bound by their sum, and the class's own is the
// faster per world; so it is where no world is past the classes. ms a settled
// step with a launch of its own / joined:
//     50 worlds of up to  2900 contacts          0.72 / 0.49
//     50 worlds of up to  1400 contacts          0.37 / 0.46
//   1000 worlds, 150 in the two classes          1.49 / 1.21 (both with the classes' launch submitted late)
//   2500 worlds, 360 in them                     2.14 / 2.23
//   4096 worlds, 590 in them                     3.09 / 3.39
constexpr bool pair_class_joins(int worlds, int past, int compute_units) {
  return past > 0 && worlds <= compute_units;
}

}  // namespace b2g
