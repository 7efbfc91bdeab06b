// dm_m3.hip - pair-sum density kernel instantiated for M = 3 orbitals.
#include "density_impl.hpp"

namespace mctdhb {
template struct DmPairs<3>;
}  // namespace mctdhb
