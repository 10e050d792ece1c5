// sdg_launch_planar.hip -- kernel sets of lines and triangles
#include "launchers.hpp"

namespace sdg {

// 1-D: vector kernels (P+1 modes, P+1 Gauss points, two end-point faces)
bool selectLine(int order, bool mixed, Launchers& l) {
  switch (order) {
    case 1: return pickLine<2>(mixed, l);
    case 2: return pickLine<3>(mixed, l);
    case 3: return pickLine<4>(mixed, l);
    case 4: return pickLine<5>(mixed, l);
    case 5: return pickLine<6>(mixed, l);
    default: return false;
  }
}

// bases of 3..15 functions
bool selectTriangle(int order, bool force_valu, bool mixed, Launchers& l) {
  switch (order) {
    case 1: return pickSimplex<2, 3, 3, 3, 2>(force_valu, mixed, l);
    case 2: return pickSimplex<2, 6, 6, 3, 3>(force_valu, mixed, l);
    case 3: return pickSimplex<2, 10, 12, 3, 4>(force_valu, mixed, l);
    case 4: return pickSimplex<2, 15, 16, 3, 5>(force_valu, mixed, l);
    default: return false;
  }
}

}  // namespace sdg
