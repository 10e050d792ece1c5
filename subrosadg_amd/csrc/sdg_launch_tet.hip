// sdg_launch_tet.hip -- kernel sets of tetrahedra
#include "launchers.hpp"

namespace sdg {

// bases of 4..35 functions, Grundmann-Moeller volume rules
bool selectTetrahedron(int order, bool force_valu, bool mixed, Launchers& l) {
  switch (order) {
    case 1: return pickSimplex<3, 4, 5, 4, 4>(force_valu, mixed, l);
    case 2: return pickSimplex<3, 10, 15, 4, 7>(force_valu, mixed, l);
    case 3: return pickSimplex<3, 20, 35, 4, 13>(force_valu, mixed, l);
    case 4: return pickSimplex<3, 35, 70, 4, 19>(force_valu, mixed, l);
    default: return false;
  }
}

}  // namespace sdg
