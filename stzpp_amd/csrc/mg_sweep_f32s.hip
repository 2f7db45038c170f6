// Instances of the marching sweep kernel (mg_instances.hpp).
#include "mg_instances.hpp"

namespace stzmg {
STZ_SWEEP_SYM(, float)
}  // namespace stzmg
