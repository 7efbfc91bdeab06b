// h2_m6.hip - two-stage H.C kernels instantiated for M = 6 orbitals.
#include "hamiltonian_two.hpp"

namespace mctdhb {
template struct HcTwo<6>;
}  // namespace mctdhb
