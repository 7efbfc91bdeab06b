// dm_m6.hip - pair-sum density kernel instantiated for M = 6 orbitals.
#include "density_impl.hpp"

namespace mctdhb {
template struct DmPairs<6>;
}  // namespace mctdhb
