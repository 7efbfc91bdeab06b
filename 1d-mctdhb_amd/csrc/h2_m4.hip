// h2_m4.hip - pair form of the last Lanczos iteration and one-workgroup SIL kernels instantiated for M = 4 orbitals.
#include "sil_small.hpp"

namespace mctdhb {
template struct HcTwo<4>;
}  // namespace mctdhb
