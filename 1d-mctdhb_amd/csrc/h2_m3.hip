// h2_m3.hip - two-stage H.C kernels instantiated for M = 3 orbitals.
#include "hamiltonian_two.hpp"

namespace mctdhb {
template struct HcTwo<3>;
}  // namespace mctdhb
