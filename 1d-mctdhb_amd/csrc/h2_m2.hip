// h2_m2.hip - two-stage H.C kernels instantiated for M = 2 orbitals.
#include "hamiltonian_two.hpp"

namespace mctdhb {
template struct HcTwo<2>;
}  // namespace mctdhb
