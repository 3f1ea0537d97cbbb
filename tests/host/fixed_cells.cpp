// Compares the cloud weight's fixed-point cells with the reference's
// (floor((float)(s + o) / res), Grid3d.cpp:174-187) on the host, one axis at a
// time, with the library's own grid metadata: points aimed at cell faces and
// uniform ones, under offsets of many poses.  Reads lines of
//   nx ny nz  res  minx miny minz  cut  draws  seed
// (max lies `cut` cells below the last face) and prints for each
//   fixed  near-fraction-bound  compared  wrong  outside-near
// (compared: evaluations away from the faces; outside-near: lanes that would be
// redone for the point that stands for padding and non-finite points)
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "../../amcl3d_amd/csrc/a3d_internal.h"

namespace {

struct Cell {
  bool in;
  uint32_t i;
};

// The reference's cell of a point at s of a pose at offset o.
Cell reference(const a3d::GridDev& g, int a, float s, double o) {
  const float q = (float)((double)s + o);
  if (!(q >= 0.0f) || !((double)q < g.ext[a])) return {false, 0};
  const double c = std::floor((double)q / g.res);
  if (!(c < (double)g.size[a])) return {false, 0};
  return {true, (uint32_t)c};
}

// The fixed-point form; false where the kernel redoes the lane.
bool fixed(const a3d::GridDev& g, int a, float s, double o, Cell& out) {
  const double x = std::fma((double)s, g.fx_scale, a3d::fixed_offset(g, o));
  uint64_t b;
  std::memcpy(&b, &x, 8);
  if ((uint32_t)b < g.fx_near) return false;
  const uint32_t i = (uint32_t)(b >> 32);
  out = {i < g.fx_size[a], i};
  return true;
}

}  // namespace

int main() {
  unsigned nx, ny, nz;
  double res, m[3], cut;
  long draws;
  unsigned long seed;
  while (std::scanf("%u %u %u %lf %lf %lf %lf %lf %ld %lu", &nx, &ny, &nz, &res, &m[0], &m[1], &m[2], &cut, &draws,
                    &seed) == 10) {
    const unsigned size[3] = {nx, ny, nz};
    double mx[3];
    for (int a = 0; a < 3; ++a) mx[a] = m[a] + ((double)size[a] - cut) * res;
    a3d::GridDev g{};
    a3d::grid_meta(m, mx, res, g);
    long compared = 0, wrong = 0;
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> u01(0.0, 1.0);
    for (long d = 0; g.fixed && d < draws; ++d) {
      const int a = (int)(d % 3);
      // offsets of poses in and around the map, and now and then far from it
      double t = m[a] + g.ext[a] * (1.4 * u01(rng) - 0.2);
      if (d % 64 == 0) t = m[a] + g.ext[a] * std::ldexp(u01(rng) - 0.5, (int)(rng() % 40));
      const float tx = (float)t;
      const double o = (double)tx - m[a];
      float s;
      if (u01(rng) < 0.7) {  // at a face, the ends of the axis more often than the others
        double k = std::floor(u01(rng) * (g.size[a] + 3)) - 1.0;
        if (u01(rng) < 0.2) k = (rng() & 1) ? 0.0 : (double)g.size[a];
        s = (float)(k * res - o);
        const int steps = (int)(rng() % 9) - 4;
        for (int j = 0; j < std::abs(steps); ++j) s = std::nextafter(s, steps < 0 ? -INFINITY : INFINITY);
      } else {
        s = (float)(g.ext[a] * u01(rng) - o);
      }
      Cell f{}, r = reference(g, a, s, o);
      if (!fixed(g, a, s, o, f)) continue;
      ++compared;
      wrong += f.in != r.in || (r.in && f.i != r.i);
    }
    long outside = 0;
    for (int d = 0; g.fixed && d < 20000; ++d) {  // rotated by any yaw, as the kernel does
      const float yaw = (float)(6.4 * u01(rng) - 3.2), c = std::cos(yaw), n = std::sin(yaw), p = a3d::kOutside;
      const float s[3] = {p * c + p * -n, p * n + p * c, p};
      for (int a = 0; a < 3; ++a) {
        Cell f{};
        const double o = (double)(float)(m[a] + g.ext[a] * u01(rng)) - m[a];
        outside += !fixed(g, a, s[a], o, f) || f.in;
      }
    }
    std::printf("%u %.9g %ld %ld %ld\n", g.fixed, std::ldexp((double)g.fx_near, -32), compared, wrong, outside);
  }
  return 0;
}
