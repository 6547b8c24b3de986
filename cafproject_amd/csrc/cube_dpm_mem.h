/*
 * cube_dpm_mem.h -- when a box of the differentiable model keeps the force
 * meshes of its steps (include/cube_dpm.h).  Plain C: the tests build it too.
 */
#ifndef CUBE_DPM_MEM_H
#define CUBE_DPM_MEM_H
#include <stdint.h>

/*
 * The force meshes of all steps save the adjoint a force evaluation per step,
 * but take more than the rest of a box (128^3 particles on 256^3 points, 10
 * steps: 1.8 GB beside 1.3), and boxes made later need room too.  They are
 * kept while, behind them,
 *  - three quarters of the device stay free, and
 *  - what stays free is at least the part of a device that a set of boxes like
 *    this one needs without them, if with 30 bytes per mesh point and 36 per
 *    particle more in each the set would just fill it.  That is what a box
 *    took when it scattered its deposits into 64-bit meshes: however many
 *    boxes fitted then still fit, the first ones with their force meshes (156
 *    of the size above on 288 GB then, 195 now, 23 of them with).  The bound
 *    binds where positions are most of a box (above 28 steps of that size).
 * free_b, total_b: the device's memory, the box's other arrays in place;
 * base_b: what these take; extra_b: the force meshes beyond the first.
 */
static inline int dpm_keep_force(uint64_t free_b, uint64_t total_b, uint64_t base_b, uint64_t extra_b, int64_t nf3,
                                 int64_t np) {
  const double b = (double)base_b, full = b + 30.0 * (double)nf3 + 36.0 * (double)np, tot = (double)total_b;
  const double part = b / full > 0.75 ? b / full : 0.75;
  return free_b >= extra_b && (double)(free_b - extra_b) >= part * tot;
}

#endif
