// h2_m5.hip - two-stage H.C kernels instantiated for M = 5 orbitals.
#include "hamiltonian_two.hpp"

namespace mctdhb {
template struct HcTwo<5>;
}  // namespace mctdhb
