// dm_m7.hip - pair-sum density kernel instantiated for M = 7 orbitals.
#include "density_impl.hpp"

namespace mctdhb {
template struct DmPairs<7>;
}  // namespace mctdhb
