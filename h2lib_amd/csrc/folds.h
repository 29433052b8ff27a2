// Surfaces that fold back on themselves (host).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace h2hip {

// Whether two triangles with a common vertex have opposite normals (to 18
// degrees): the surface folds back on itself there, as the finer cylinder
// meshes do.  Where the folded sheets overlap, <x - y, n> is zero up to the
// rounding of the points, which 1/r^3 magnifies: forming it from anything
// but the difference x - y moves such entries by up to 1e-9 of the largest
// (cylinder, 46240 triangles; 8e-13 in the norm of all entries).
//
// v2t[v2t_ptr[v] ..]: the triangles of vertex v; n: their normals, of any
// length.  The work per triangle is bounded: at a vertex of more than 32
// triangles (poles, apexes of fans) the normals are binned into cells of
// edge 1/3, a little more than the chord of 18.4 degrees, and each is
// compared with those in the 27 cells around its opposite.  A vertex where
// that finds more than 64 candidates per triangle counts as folded (a sharp
// cone of many triangles): such surfaces only lose the faster kernels.  A
// fan of 100000 triangles took 5e9 comparisons without the cells.
inline bool folds(uint32_t nv, const uint32_t *v2t_ptr, const uint32_t *v2t,
                  const double *n) {
  constexpr uint32_t DIRECT = 32, BUDGET = 64;
  constexpr int E = 6;  // cells per edge of [-1, 1]^3
  auto opposite = [&](const double *a, const double *b) {
    const double ab = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
    return ab < 0.0 &&
           ab * ab > 0.9 * (a[0] * a[0] + a[1] * a[1] + a[2] * a[2]) *
                         (b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
  };
  std::vector<uint32_t> head, next;  // lists per cell, 1 + position
  for (uint32_t v = 0; v < nv; v++) {
    const uint32_t *t = v2t + v2t_ptr[v];
    const uint32_t cnt = v2t_ptr[v + 1] - v2t_ptr[v];
    if (cnt <= DIRECT) {
      for (uint32_t p = 0; p < cnt; p++)
        for (uint32_t q = p + 1; q < cnt; q++)
          if (opposite(n + 3 * (size_t)t[p], n + 3 * (size_t)t[q]))
            return true;
      continue;
    }
    head.assign(E * E * E, 0);
    next.assign(cnt, 0);
    uint64_t left = (uint64_t)BUDGET * cnt;
    for (uint32_t p = 0; p < cnt; p++) {
      const double *a = n + 3 * (size_t)t[p];
      const double len =
          std::sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
      if (!(len > 0.0) || !std::isfinite(len)) continue;  // opposite to none
      int c[3], o[3];  // cells of the normal and of its opposite
      for (int d = 0; d < 3; d++) {
        const double u = a[d] / len;
        c[d] = std::min(E - 1, std::max(0, (int)((1.0 + u) * (E / 2))));
        o[d] = std::min(E - 1, std::max(0, (int)((1.0 - u) * (E / 2))));
      }
      for (int i = std::max(0, o[0] - 1); i <= std::min(E - 1, o[0] + 1); i++)
        for (int j = std::max(0, o[1] - 1); j <= std::min(E - 1, o[1] + 1);
             j++)
          for (int k = std::max(0, o[2] - 1);
               k <= std::min(E - 1, o[2] + 1); k++)
            for (uint32_t q = head[(i * E + j) * E + k]; q; q = next[q - 1]) {
              if (opposite(a, n + 3 * (size_t)t[q - 1]) || left-- == 0)
                return true;
            }
      uint32_t &h = head[(c[0] * E + c[1]) * E + c[2]];
      next[p] = h;
      h = p + 1;
    }
  }
  return false;
}

}  // namespace h2hip
