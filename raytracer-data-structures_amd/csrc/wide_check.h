// Host check of a 4-wide node's record, one axis at a time: the planes on its grid
// against the exact planes of its slots (rq_bvh_export_wide). No HIP types.
#pragma once
#include <cmath>
#include <cstdint>

namespace rq {

// What is wrong with an axis of a record, or null: lo / hi are the exact planes of
// the four slots (slots with used 0 are not looked at), base, step, qlo, qhi the
// record's. Each plane has to lie outside the exact one, by 2^-10 of a step (the walk
// relies on that) and by no more than two steps; the step has to be the least that
// covers the slots; a NaN step, which reads as a box everywhere, is for extents or
// coordinates of 2^100 or more only. Planes that are NaN, or lo above hi (spheres of
// negative radius), bound nothing that could be hit: only the outside is checked.
inline const char* wide_axis_fault(const float lo[4], const float hi[4], const int32_t used[4],
                                   float base, float step, uint32_t qlo, uint32_t qhi) {
  double l = INFINITY, h = -INFINITY;
  bool plain = true;
  for (int k = 0; k < 4; ++k) {
    if (!used[k]) continue;
    plain = plain && lo[k] <= hi[k];
    l = std::fmin(l, (double)lo[k]), h = std::fmax(h, (double)hi[k]);
  }
  const double ext = h - l, mag = std::fmax(std::fabs(l), std::fabs(h)), big = std::ldexp(1.0, 100);
  if (std::isnan(step))
    return plain && ext < big * (1.0 - 1e-6) && mag < big ? "no grid where one is possible" : nullptr;
  if (!(step > 0.0f) || !std::isfinite(base)) return "no grid";
  const double least = std::fmax(std::fmax(ext / 252.0, std::ldexp(mag, -21)), std::ldexp(1.0, -60));
  if (plain && step > least * (1.0 + 1e-6)) return "its grid is too coarse";
  for (int k = 0; k < 4; ++k) {
    if (!used[k]) continue;
    const double a = base + (1024.0 + (qlo >> (8 * k) & 255u)) * (double)step;
    const double b = base + (1024.0 + (qhi >> (8 * k) & 255u)) * (double)step;
    const double margin = std::ldexp((double)step, -10);
    if (a > lo[k] - margin || b < hi[k] + margin) return "its box does not hold the exact one";
    if (plain && (a < lo[k] - 2.0 * step || b > hi[k] + 2.0 * step)) return "its box is too large";
  }
  return nullptr;
}

}  // namespace rq
