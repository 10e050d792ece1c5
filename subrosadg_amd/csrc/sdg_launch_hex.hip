// sdg_launch_hex.hip -- kernel sets of hexahedra (dense operators)
#include "launchers.hpp"

namespace sdg {

bool selectHexahedron(int order, bool force_valu, bool mixed, Launchers& l) {
  switch (order) {
    case 1: return pickValu<3, 8, 8, 6, 4>(mixed, l);
    case 2: return pickMfma<3, 27, 27, 6, 9>(force_valu, mixed, l);
    case 3: return pickMfma<3, 64, 64, 6, 16>(force_valu, mixed, l);
    case 4: return pickMfma<3, 125, 125, 6, 25>(force_valu, mixed, l);
    default: return false;
  }
}

}  // namespace sdg
