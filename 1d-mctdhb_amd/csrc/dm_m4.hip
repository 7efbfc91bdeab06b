// dm_m4.hip - pair-sum density kernel instantiated for M = 4 orbitals.
#include "density_impl.hpp"

namespace mctdhb {
template struct DmPairs<4>;
}  // namespace mctdhb
