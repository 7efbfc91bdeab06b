// h2_m5.hip - pair form of the last Lanczos iteration and one-workgroup SIL kernels instantiated for M = 5 orbitals.
#include "sil_small.hpp"

namespace mctdhb {
template struct HcTwo<5>;
}  // namespace mctdhb
