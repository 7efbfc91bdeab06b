// h2_m4.hip - two-stage H.C kernels instantiated for M = 4 orbitals.
#include "hamiltonian_two.hpp"

namespace mctdhb {
template struct HcTwo<4>;
}  // namespace mctdhb
