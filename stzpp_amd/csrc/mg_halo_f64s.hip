// Instances of the small levels' one-launch kernels (mg_instances.hpp).
#include "mg_instances.hpp"

namespace stzmg {
STZ_HALO_SYM(, double)
}  // namespace stzmg
