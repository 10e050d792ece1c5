// sdg_launch_tensor.hip -- sum-factorised kernel sets of hexahedra and quadrangles
#include "launchers.hpp"

namespace sdg {

bool selectTensor(int order, bool mixed, Launchers& l) {
  switch (order) {
    case 2: return pickTensor<3>(mixed, l);
    case 3: return pickTensor<4>(mixed, l);
    case 4: return pickTensor<5>(mixed, l);
    default: return false;
  }
}

bool selectTensorAv(int order, bool mixed, Launchers& l) {
  return mixed ? selectTensorAvT<float>(order, l) : selectTensorAvT<double>(order, l);
}

bool selectQuadTensor(int order, Launchers& l) {
  switch (order) {
    case 1: return pickQuad<2>(l);
    case 2: return pickQuad<3>(l);
    case 3: return pickQuad<4>(l);
    case 4: return pickQuad<5>(l);
    case 5: return pickQuad<6>(l);
    default: return false;
  }
}

}  // namespace sdg
