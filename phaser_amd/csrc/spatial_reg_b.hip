// Register-engine passes of the translation stage for the lengths of one group.
#include "spatial_reg.hpp"

namespace phz {
PHZ_SPATIAL_REG_GROUP(spatial_reg_b, PHZ_REG_LENGTHS_B)
}  // namespace phz
