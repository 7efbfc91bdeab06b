// h2_m7.hip - two-stage H.C and one-workgroup SIL kernels instantiated for M = 7 orbitals.
#include "sil_small.hpp"

namespace mctdhb {
template struct HcTwo<7>;
template struct HcTwoRows<7>;
}  // namespace mctdhb
