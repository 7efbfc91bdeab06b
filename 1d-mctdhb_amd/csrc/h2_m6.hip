// h2_m6.hip - two-stage H.C and one-workgroup SIL kernels instantiated for M = 6 orbitals.
#include "sil_small.hpp"

namespace mctdhb {
template struct HcTwo<6>;
template struct HcTwoRows<6>;
}  // namespace mctdhb
