// h2_m3.hip - pair form of the last Lanczos iteration and one-workgroup SIL kernels instantiated for M = 3 orbitals.
#include "sil_small.hpp"

namespace mctdhb {
template struct HcTwo<3>;
}  // namespace mctdhb
