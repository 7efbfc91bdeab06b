// h2_m7.hip - two-stage H.C kernels instantiated for M = 7 orbitals.
#include "hamiltonian_two.hpp"

namespace mctdhb {
template struct HcTwo<7>;
}  // namespace mctdhb
