// h2_m2.hip - pair form of the last Lanczos iteration and one-workgroup SIL kernels instantiated for M = 2 orbitals.
#include "sil_small.hpp"

namespace mctdhb {
template struct HcTwo<2>;
}  // namespace mctdhb
