// sdg_launch_pyramid.hip -- kernel sets of pyramids
#include "launchers.hpp"

namespace sdg {

// (P+1)^3 collapsed points, five faces of (P+1)^2 slots: vector kernels
bool selectPyramid(int order, bool mixed, Launchers& l) {
  switch (order) {
    case 1: return pickValu<3, 5, 8, 5, 4>(mixed, l);
    case 2: return pickValu<3, 14, 27, 5, 9>(mixed, l);
    case 3: return pickValu<3, 30, 64, 5, 16>(mixed, l);
    case 4: return pickValu<3, 55, 125, 5, 25>(mixed, l);
    default: return false;
  }
}

}  // namespace sdg
