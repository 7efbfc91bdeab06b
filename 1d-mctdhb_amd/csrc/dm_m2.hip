// dm_m2.hip - pair-sum density kernel instantiated for M = 2 orbitals.
#include "density_impl.hpp"

namespace mctdhb {
template struct DmPairs<2>;
}  // namespace mctdhb
