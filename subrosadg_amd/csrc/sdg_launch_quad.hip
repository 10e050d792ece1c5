// sdg_launch_quad.hip -- kernel sets of quadrangles
#include "launchers.hpp"

namespace sdg {

bool selectQuadrangle(int order, bool force_valu, bool mixed, Launchers& l) {
  switch (order) {
    case 1: return pickValu<2, 4, 4, 4, 2>(mixed, l);
    case 2: return pickValu<2, 9, 9, 4, 3>(mixed, l);
    case 3: return pickMfma<2, 16, 16, 4, 4>(force_valu, mixed, l);
    case 4: return pickMfma<2, 25, 25, 4, 5>(force_valu, mixed, l);
    case 5: return pickMfma<2, 36, 36, 4, 6>(force_valu, mixed, l);
    default: return false;
  }
}

}  // namespace sdg
