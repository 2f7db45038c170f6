// Instances of the one-launch sweep (mg_instances.hpp).
#include "mg_instances.hpp"

namespace stzmg {
STZ_HALO_SYM(, float)
}  // namespace stzmg
