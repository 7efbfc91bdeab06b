// dm_m5.hip - pair-sum density kernel instantiated for M = 5 orbitals.
#include "density_impl.hpp"

namespace mctdhb {
template struct DmPairs<5>;
}  // namespace mctdhb
