// Instances of the marching residual kernel (mg_instances.hpp).
#include "mg_instances.hpp"

namespace stzmg {
STZ_RESID_ALL(, float)
}  // namespace stzmg
