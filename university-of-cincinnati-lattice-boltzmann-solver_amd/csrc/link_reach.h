// How far the coordinates of a link-table build reach from the origin
// (LinkGeom::reach).  Host code, without any dependence on HIP.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace uclbs {

// Sum over the axes of the largest |coordinate| of a node or a triangle.  A
// level of one box: extent nodes from the origin on.  A level of nbox boxes
// (valid regions blo..bhi, [nbox][3]): their corners with the one-node shell;
// extent, the flat count of the stored nodes there, is no length and is not
// read.  gbb: the triangles' box (max, min per axis), null without triangles.
inline double link_reach(const double origin[3], double dx, const int extent[3], size_t nbox,
                         const int32_t* blo, const int32_t* bhi, const double* gbb) {
  double reach = 0.0;
  for (int d = 0; d < 3; ++d) {
    double far = nbox ? 0.0
                      : std::max(std::fabs(origin[d]),
                                 std::fabs(origin[d] + (double)(extent[d] - 1) * dx));
    for (size_t b = 0; b < nbox; ++b)
      far = std::max(far, std::max(std::fabs(origin[d] + (double)(blo[3 * b + d] - 1) * dx),
                                   std::fabs(origin[d] + (double)(bhi[3 * b + d] + 1) * dx)));
    if (gbb) far = std::max(far, std::max(std::fabs(gbb[2 * d]), std::fabs(gbb[2 * d + 1])));
    reach += far;
  }
  return reach;
}

}  // namespace uclbs
